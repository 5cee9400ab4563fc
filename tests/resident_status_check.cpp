// The host's reading of the one-launch solves' record (resident_status.h), on
// records as the kernels leave them.
#include <math.h>
#include <stdio.h>

#include "resident_status.h"

using namespace mono;

static int failed = 0;
static void expect(const char *what, long long got, long long want) {
    if(got == want) return;
    printf("%s: %lld, expected %lld\n", what, got, want);
    failed = 1;
}

// What block 0 writes at the end of a solve of `its` iterations and `outer` sweeps.
static void note(ResidentStatus &s, uint32_t exchanges, int its, int outer, double err) {
    s.epoch += exchanges;
    s.solves += 1;
    s.cg_total += its;
    s.inner_total += its - 1;
    s.outer_total += outer;
    s.last_its = its;
    s.last_outer = outer;
    s.last_err = err;
    if(err != err) s.stop = kResidentNan;
}

static void check(const char *what, const ResidentStatus &r, int stop, long long solves, long long cg, long long inner, long long outer) {
    printf("%s\n", what);
    expect("stop", r.stop, stop);
    expect("solves", r.solves, solves);
    expect("iterations", r.cg_total, cg);
    expect("inner iterations", r.inner_total, inner);
    expect("sweeps", r.outer_total, outer);
}

int main() {
    ResidentStatus seen{}, s{};
    for(int k = 0; k < 5; k++) note(s, 9 + k, 10 + k, 2, 1e-17);
    check("all done", resident_since(s, seen), kResidentGoing, 5, 60, 55, 10);
    seen = s;

    // three more; in the fourth every waiting block gives up before its end
    for(int k = 0; k < 3; k++) note(s, 8, 9, 1, 1e-17);
    s.left = s.epoch + 4;
    s.stop = kResidentTimeout;
    check("a solve left in its middle", resident_since(s, seen), kResidentTimeout, 3, 27, 24, 3);

    // the fourth is counted by block 0, another block gave up in its last exchange
    ResidentStatus half = s;
    half.left = s.epoch + 8;
    note(half, 8, 9, 1, 1e-17);
    check("a solve left in its last exchange", resident_since(half, seen), kResidentTimeout, 3, 27, 24, 3);

    // the same as the last solve of those enqueued: count - 1 are done
    ResidentStatus only = seen;
    only.left = only.epoch + 1;
    only.stop = kResidentTimeout;
    note(only, 1, 1, 1, 1e-17);
    check("the only solve, converged at its start, left in its one exchange", resident_since(only, seen), kResidentTimeout, 0, 0, 0, 0);

    // block 0 notes a NaN over another block's time-out
    ResidentStatus nan = seen;
    nan.left = nan.epoch + 3;
    nan.stop = kResidentTimeout;
    note(nan, 3, 4, 1, NAN);
    check("a NaN noted over a time-out", resident_since(nan, seen), kResidentTimeout, 0, 0, 0, 0);

    // a NaN by itself counts
    ResidentStatus bad = seen;
    note(bad, 3, 4, 1, NAN);
    check("a NaN", resident_since(bad, seen), kResidentNan, 1, 4, 3, 1);

    // after the record was cleared (resident_reset) the totals go on
    seen = half;
    ResidentStatus next = half;
    next.epoch = next.left = 0;
    next.stop = kResidentGoing;
    note(next, 8, 9, 1, 1e-17);
    check("after a time-out", resident_since(next, seen), kResidentGoing, 1, 9, 8, 1);
    printf(failed ? "FAILED\n" : "ok\n");
    return failed;
}
