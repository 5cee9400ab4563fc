// Whole diffusion solve in one launch (host interface of cg_resident.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mono_common.h"
#include "operator.h"
#include "resident_status.h"

namespace mono {

struct CgConfig;

// One block's share of the box and how many blocks there are.
struct ResidentGeom {
    int bx, by, bz;     // cells of a tile
    int tx, ty, tz;     // tiles
    int rpt;            // cells per thread
    int threads;
    int halo;           // most halo cells of a tile
    size_t lds;
    bool cooperative;
};

// Buffers of the resident solves of one workspace.
struct ResidentPlan {
    int state = 0;               // 0 not planned, 1 usable, -1 not for this operator
    // what the plan was made for
    int nx = 0, ny = 0, nz = 0, pat = 0, mode = 0, mixed = -1;
    ResidentGeom g{};
    unsigned long long *words = nullptr;  // exchanged values of both parities
    unsigned long long *sums = nullptr;   // partial sums of both parities
    void *cells = nullptr;                // halo cells of every tile
    int *ncells = nullptr;                // how many each tile has
    bool cleared = false;        // words and sums hold no word of another run (resident_reset)
    uint64_t wait_ticks = 2000000;  // longest wait of a block for another: 20 ms of the 100 MHz clock
    size_t words_bytes = 0;
    size_t sums_bytes = 0;
};

// Decide the tiles for an operator and make the buffers (p->state).  New ones
// must be cleared before the first solve: memory that an earlier workspace gave
// back holds words with the first epochs' numbers, which a reader would take.
int resident_plan(ResidentPlan *p, const OpView<double> &op64, const OpView<float> *op32, const CgConfig &cfg);
int resident_release(ResidentPlan *p);
// Enqueues the solve; op32 null: FP64 CG.
int resident_launch(const ResidentPlan &p, const OpView<double> &op64, const OpView<float> *op32, const double *b, double *x,
                    const CgConfig &cfg, ResidentStatus *st, hipStream_t s);
// Clears the exchange buffers, the epoch, `stop` and `left` on the stream.
int resident_reset(ResidentPlan *plans, int nplans, ResidentStatus *st, hipStream_t s);

}  // namespace mono
