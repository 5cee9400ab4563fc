// How long the one-launch solves stay away after time-outs (ResidentPause).
#include <stdio.h>

#include <initializer_list>

#include "resident_status.h"

using mono::ResidentPause;

// Solves done by the other kernels until the next one may run in one launch.
static int away(ResidentPause &p) {
    int n = 0;
    while(p.left > 0) {
        p.spent();
        n++;
    }
    return n;
}

int main() {
    int failed = 0;
    auto expect = [&](const char *what, int got, int want) {
        if(got != want) {
            printf("%s: %d, expected %d\n", what, got, want);
            failed = 1;
        }
    };
    ResidentPause p;
    expect("no time-out", away(p), 0);
    for(int want : {16, 80, 336, 1360, 1360}) {
        p.timed_out();
        expect("one time-out after another", away(p), want);
    }
    p.solved(1359);
    p.timed_out();
    expect("fewer solves without a time-out than the pause was long", away(p), 1360);
    p.solved(1000);
    p.solved(360);
    p.timed_out();
    expect("as many: as after the first", away(p), 16);
    for(int k = 0; k < 5; k++) p.spent();
    p.solved(0);
    expect("solves elsewhere without a pause", p.left, 0);
    printf(failed ? "FAILED\n" : "ok\n");
    return failed;
}
