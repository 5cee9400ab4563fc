// Record of the one-launch diffusion solves and what the host makes of it.
#pragma once

#include <stdint.h>

namespace mono {

// Device record of the one-launch solves on one workspace.  The kernels of a
// step do nothing while `stop` is set, so solves can be enqueued ahead of the
// host's look at it.
enum ResidentStop : int32_t {
    kResidentGoing = 0,
    kResidentNan = 1,      // the last solve ended with r.r = NaN (it is counted)
    kResidentTimeout = 2,  // a block waited too long for another: the solve is not done
};
struct ResidentStatus {
    int32_t stop;
    uint32_t epoch;        // number of the last completed solve's last exchange
    uint32_t left;         // number of the last exchange that a block gave up in, 0: none did
    int64_t solves;        // solves completed
    int64_t cg_total;      // sum of the reference's iteration counts
    int64_t inner_total;   // CG iterations run
    int64_t outer_total;   // outer sweeps
    int32_t last_its;
    int32_t last_outer;
    double last_err;
};

// What happened since the record `seen`, given the record `now`: its totals are
// differences, its `stop` is what the host acts on.
//
// Block 0 counts a solve when it has the words of the last exchange.  Another
// block may give up in that very exchange, and then its part of x is as it was
// before the solve: the solve is taken out of the count again, to be done anew
// from the x that is there (the right-hand side is untouched, since nothing that
// was enqueued behind the solve has run).  `left` says so whatever `stop` holds: a
// NaN noted by block 0 may have replaced the time-out there.
inline ResidentStatus resident_since(const ResidentStatus &now, const ResidentStatus &seen) {
    ResidentStatus r = now;
    r.solves -= seen.solves;
    r.cg_total -= seen.cg_total;
    r.inner_total -= seen.inner_total;
    r.outer_total -= seen.outer_total;
    if(now.left != 0) {
        r.stop = kResidentTimeout;
        if(now.epoch >= now.left && r.solves > 0) {
            r.solves--;
            r.cg_total -= now.last_its;
            r.inner_total -= now.last_its - 1;
            r.outer_total -= now.last_outer;
        }
    }
    return r;
}

// After a time-out the chip is shared with launches of the same kind: the next
// solves are left to the kernels of cg.hip, more of them after each further
// time-out (16, 80, 336, then 1360).  As many solves in one launch without a
// time-out as the last pause was long end the lengthening.
struct ResidentPause {
    int left = 0;      // solves still to be left to the other kernels
    int length = 0;    // of the last pause
    int64_t good = 0;  // solves in one launch since the last time-out

    void timed_out() {
        length = length < 1024 ? 4 * length + 16 : length;
        left = length;
        good = 0;
    }
    void solved(int64_t n) {
        good += n;
        if(good >= length) length = 0;
    }
    // a solve was done by the other kernels
    void spent() {
        if(left > 0) left--;
    }
};

}  // namespace mono
