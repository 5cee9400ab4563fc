// The diffusion solve of a small or middle-sized domain as one launch.
//
// cg.hip runs a solve as two launches per CG iteration.  On a domain whose
// vectors fit on the chip each of them takes 4-9 us whatever its size, nearly
// all of it launch, drain and the re-reading of partial sums: a 64 x 64 x 16
// box needs 28 of them (170 us) for 8 us of memory traffic.  Here every block
// owns one tile of the domain, keeps its cells' vectors in registers and the
// residual (with a one-cell halo) in LDS for the whole solve, and exchanges
// with the other blocks only what CG needs: halo values and dot products.
//
// The recurrence is CG with w = A r kept beside s = A p, so that s needs no
// product of its own and all sums of an iteration come from one exchange (the
// idea of A. T. Chronopoulos and C. W. Gear, s-step iterative methods for
// symmetric linear systems, J. Comput. Appl. Math. 25, 1989):
//     beta  = r.r / (r.r)_old
//     p.s   = r.w + beta (r.s_old + p_old.w) + beta^2 (p.s)_old
//     alpha = r.r / p.s
//     p = r + beta p, s = w + beta s, x += alpha p, r -= alpha s, w = A r
// The expansion of p.s = p.Ap holds for any A (the anisotropic rows are not
// symmetric), so in exact arithmetic the iterates are those of the
// two-reduction form, after any number of iterations; the stopping rule and the
// iteration count are the same (linear_system_solver.c:47-183).  A block
// updates r and s also on its halo, from the halo values of w: so one exchange
// per iteration carries them and the sums.
//
// Measured (one MI355X, whole steps, launches of cg.hip -> here): 300-cell cable
// TT2006 FP64 129 -> 25 us; 64 x 64 x 16 TT2006 FP64 210 -> 66; 256 x 256
// Mitchell-Schaeffer FP32+refine, per-cell rows, 177 -> 53; 490k-cell TT2006
// FP32+refine with holes 323 -> 145; 492k-cell ORd FP32+refine, 27-point rows
// per cell, 585 -> 343; 4M-cell batch TT2006 FP32+refine 942 -> 680.  What
// bounds an iteration: 1.1 us of block sums, divisions and barriers on one
// block, 3.1 us on 128 blocks (two trips of a word through the memory-side
// cache), 6-14 us where a block holds 2,000-16,000 cells (LDS reads, and the
// wait for the slowest of the blocks).
//
// Exchanges need no grid barrier and no fences.  Every 64-bit word that goes
// from one block to another carries 32 bits of value and the 32-bit number of
// the exchange (epoch) that it belongs to, is written and read with relaxed
// agent-scope atomics (which go past the XCDs' L2 caches), and a reader polls
// until the epoch is the one it waits for.  A double is two such words, a
// float one.  Two buffers alternate by the parity of the epoch: a block writes
// epoch e + 2 only after it has all sums of epoch e + 1, which every block
// wrote after it had read everything of epoch e.  One exchange between 128
// blocks takes 2.3 us; a pair of kernel boundaries took 12.
//
// Waits are bounded (ResidentPlan::wait_ticks): if a block of the launch does not get a
// place on the chip because others' blocks wait there for theirs, the waiting
// blocks give up, mark the status record and end; x still is a valid start,
// and the host solves that step with the kernels of cg.hip.  Launches whose
// blocks could not share the chip with those of a second such launch are made
// cooperative, which the runtime runs one at a time; it costs 19 us more per
// launch than a plain one.
#include "cg_resident.h"

#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "cg.h"
#include "wave_sum.h"

namespace mono {

namespace {

typedef unsigned long long u64;

__device__ __forceinline__ u64 word_load(const u64 *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void word_store(u64 *p, u64 v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ u64 tagged(uint32_t epoch, uint32_t half) { return ((u64)epoch << 32) | half; }

// values of type T in an exchange: one word (float) or two (double)
template <typename T> constexpr int kWords = sizeof(T) / 4;
__device__ __forceinline__ void put_value(u64 *w, uint32_t epoch, float v) { word_store(w, tagged(epoch, __float_as_uint(v))); }
__device__ __forceinline__ void put_value(u64 *w, uint32_t epoch, double v) {
    const u64 bits = (u64)__double_as_longlong(v);
    word_store(w, tagged(epoch, (uint32_t)bits));
    word_store(w + 1, tagged(epoch, (uint32_t)(bits >> 32)));
}

constexpr int kSums = 3;       // sums of an exchange
constexpr int kSumWords = 8;   // words of a block's sums: two each, to a line of 64 bytes that only it writes
constexpr int kSumBlocks = 8;  // blocks whose sums one load of a wave covers
constexpr int kSumLoads = 16;  // such loads in flight together
constexpr int kMaxSumWaves = 2;
constexpr int kXcds = 8;

// One halo cell of a tile.  Listed once per plan: found by every block in every
// launch (a scan of its tile with divisions, an LDS counter) they took 8 of the
// 11 us before the first exchange of 490k cells.
struct HaloCell {
    uint32_t word;  // index of its value in the word buffer
    uint32_t cell;  // cell of the box
    uint32_t ext;   // index in the tile with halo
    uint32_t pad;
};

struct ResidentArgs {
    OpView<double> op64;
    OpView<float> op32;
    int bx, by, bz, tx, ty, tz;
    uint32_t div_bx, div_by;  // floor(2^32 / b) + 1: a quotient of numbers below 2^16 is one high product
    int nblocks, halo;
    const double *b;
    double *x;
    double tol, rel_tol, inner_rel;
    const double *tol_dev;
    int max_its, max_outer;
    u64 *words, *sums;
    const HaloCell *cells;  // [block][halo]
    const int *ncells;
    u64 wait_ticks;
    ResidentStatus *st;
};

// Threads per block and cells per thread that kernels are built for.  Small
// tiles take one wave per SIMD (cheaper block sums), large ones as many waves
// as their registers allow.
struct Shape {
    int threads, rpt;
};
constexpr Shape kShapes[] = {{256, 1}, {256, 2}, {512, 2}, {512, 4}, {512, 8}, {512, 32}};

// Whether the rows of own cells are kept for the whole solve (rows stored per
// cell): read again in every iteration they would come from the memory-side
// cache at a latency that these few waves cannot hide (27-point rows of 492k
// cells: 40 us an iteration, 8 us kept).  The bound is on the coefficients
// alone: up to 64 or 112 registers a thread.  In the largest such shapes the
// compiler then spills other values, or some of the rows, to scratch: 77
// registers of FP64 7-point rows at 512 x 8, 36 of mixed 27-point rows at
// 512 x 4, 24 of mixed 7-point rows at 512 x 8, 7 of mixed 19-point rows at 512 x 4,
// 2 of FP64 27-point rows at 512 x 2.
constexpr bool keeps_rows(bool mixed, int P, int T, int rpt, bool table) {
    return !table && rpt * P * (mixed ? 1 : 2) <= (T == 512 ? 112 : 64);
}
// Whether own x and b stay in registers through the solve (else read again).
constexpr bool holds_xb(bool mixed, int P, int rpt, bool table) {
    return rpt <= 8 && (table ? 0 : rpt * P * (mixed ? 1 : 2)) + 4 * rpt <= 124;
}

// A domain is solved here whenever its vectors fit (resident_plan) and its rows
// are a table or stored per cell: from the smallest to the largest that fits,
// no size was found where the launches of cg.hip take less time (1.1-6x over
// domains of 300 to 4M cells).  Rows formed from neighbourhood masks, Jacobi
// and CSR solves stay there, and so do rows that reach across an axis of one
// cell: a tile has no halo along such an axis (its neighbour strides are 0), so
// their coefficients would multiply the cell itself.  Assembled rows are 0 there.
//
// Which shapes are built: a table in LDS with few cells per block or many;
// rows per cell only where they are kept.
constexpr bool built(bool mixed, int P, int T, int rpt, bool table) {
    if(rpt == 32) return mixed && table && P == 7;
    if(T == 512 && rpt == 2) return !table && P != 7;
    return table || keeps_rows(mixed, P, T, rpt, table);
}

// table rows of a tile: 9 position classes of each of its layers, or the code rows
constexpr int kTableLayers = 16;  // most layers of a tile in class mode

template <bool MIXED, int P, int T, int RPT, bool TABLE> struct Resident {
    using TV = typename std::conditional<MIXED, float, double>::type;
    static constexpr int NW = T / 64;
    static constexpr bool kKeepRows = keeps_rows(MIXED, P, T, RPT, TABLE);

    const ResidentArgs &a;
    // LDS
    double *ext64;   // x with halo (shares its space with ext)
    TV *ext;         // the residual with halo
    TV *hs, *hw;     // halo: s and the received values
    TV *hp, *hd;     // mixed, halo: p and the correction d
    double *hx;      // mixed, halo: x
    uint32_t *hword; // halo: index of the value in the word buffer
    uint16_t *hext;  // halo: index in ext
    double *tab64;
    TV *tab;
    double *part;    // [3][NW] wave sums, then [4 kMaxSumWaves][3] sums of blocks'
    int *flags;      // [0] a wait ended without its word, [1] halo count

    int tid, lane, wave;
    int block;       // its tile and the place of its words
    int x0, y0, z0, ex, ey, ez, hx_, hy_, hz_;
    int dy, dz;      // neighbour strides in ext (0 along an axis of one cell)
    int nh;
    uint32_t meta[RPT];  // ext index | table row << 16
    uint32_t cells[TABLE ? 1 : RPT];  // own cells in the box (rows stored per cell)
    uint32_t mask;       // bit q: own cell q is in the box
    uint32_t edge;       // bit q: a neighbour tile needs it
    uint32_t epoch;
    TV w[RPT];

    __device__ Resident(const ResidentArgs &args) : a(args) {}

    __device__ __forceinline__ bool own(int q) const { return (mask >> q) & 1u; }
    __device__ __forceinline__ int local(int q) const { return tid + q * T; }
    __device__ __forceinline__ int64_t cell(int q) const {
        int lx, ly, lz, l = local(q);
        asm volatile("" : "+v"(l));
        split(l, lx, ly, lz);
        return (x0 + lx) + (int64_t)a.op64.nx * ((y0 + ly) + (int64_t)a.op64.ny * (z0 + lz));
    }
    __device__ __forceinline__ void split(int l, int &lx, int &ly, int &lz) const {
        const int r = a.bx == 1 ? l : (int)__umulhi((uint32_t)l, a.div_bx);
        lx = l - r * a.bx;
        lz = a.by == 1 ? r : (int)__umulhi((uint32_t)r, a.div_by);
        ly = r - lz * a.by;
    }
    // this thread's place: own cells and their masks
    __device__ __forceinline__ void place() {
        tid = threadIdx.x;
        lane = tid & 63;
        wave = tid >> 6;
        const int nx = a.op64.nx, ny = a.op64.ny, nz = a.op64.nz;
        // Blocks go to the eight XCDs in turn; an XCD's blocks take consecutive
        // tiles, so that most neighbours are on one XCD and the lines that their
        // rows, x and b share are in its L2 (490k-cell wedges, a step: 27-point
        // rows per cell 415 -> 349 us, a table of rows 179 -> 149).
        {
            const int full = a.nblocks / kXcds, rest = a.nblocks % kXcds, x = blockIdx.x % kXcds;
            block = x * full + (x < rest ? x : rest) + blockIdx.x / kXcds;
        }
        const int bt = block, btx = bt % a.tx, bty = (bt / a.tx) % a.ty, btz = bt / (a.tx * a.ty);
        x0 = btx * a.bx;
        y0 = bty * a.by;
        z0 = btz * a.bz;
        mask = edge = 0;
        const int tile = a.bx * a.by * a.bz;
#pragma unroll
        for(int q = 0; q < RPT; q++) {
            const int l = local(q);
            int lx, ly, lz;
            split(l, lx, ly, lz);
            const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
            if(l < tile && gx < nx && gy < ny && gz < nz) {
                mask |= 1u << q;
                if((lx == 0 && gx > 0) || (lx == a.bx - 1 && gx < nx - 1) || (ly == 0 && gy > 0) || (ly == a.by - 1 && gy < ny - 1) ||
                   (lz == 0 && gz > 0) || (lz == a.bz - 1 && gz < nz - 1))
                    edge |= 1u << q;
            }
        }
    }

    __device__ __forceinline__ void setup(char *lds) {
        const int nx = a.op64.nx, ny = a.op64.ny, nz = a.op64.nz;
        hx_ = nx > 1;
        hy_ = ny > 1;
        hz_ = nz > 1;
        ex = a.bx + 2 * hx_;
        ey = a.by + 2 * hy_;
        ez = a.bz + 2 * hz_;
        dy = hy_ ? ex : 0;
        dz = hz_ ? ex * ey : 0;
        const int ne = ex * ey * ez;
        char *at = lds;
        auto take = [&](size_t bytes) {
            char *p = at;
            at += (bytes + 15) / 16 * 16;
            return p;
        };
        ext64 = (double *)take(sizeof(double) * ne);
        ext = (TV *)ext64;
        hs = (TV *)take(sizeof(TV) * a.halo);
        hw = (TV *)take(sizeof(TV) * a.halo);
        if constexpr(MIXED) {
            hp = (TV *)take(sizeof(TV) * a.halo);
            hd = (TV *)take(sizeof(TV) * a.halo);
            hx = (double *)take(sizeof(double) * a.halo);
        }
        hword = (uint32_t *)take(sizeof(uint32_t) * a.halo);
        hext = (uint16_t *)take(sizeof(uint16_t) * a.halo);
        part = (double *)take(sizeof(double) * kSums * (NW + 4 * kMaxSumWaves));
        flags = (int *)take(2 * sizeof(int));
        if constexpr(TABLE) {
            const int rows = a.op64.codes ? kCodes : 9 * a.bz;
            tab = (TV *)take(sizeof(TV) * rows * P);
            if constexpr(MIXED) tab64 = (double *)take(sizeof(double) * rows * P);
            fill_table(a.op64, rows, MIXED ? tab64 : (double *)tab);
            if constexpr(MIXED) fill_table(a.op32, rows, (float *)tab);
        }
        if(tid == 0) flags[0] = __hip_atomic_load(&a.st->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != kResidentGoing;
        nh = a.nblocks > 1 ? a.ncells[block] : 0;
        for(int i = tid; i < nh; i += T) {
            const HaloCell h = a.cells[(size_t)block * a.halo + i];
            hword[i] = h.word;
            hext[i] = (uint16_t)h.ext;
        }
#pragma unroll
        for(int q = 0; q < RPT; q++) {
            int lx, ly, lz;
            split(local(q), lx, ly, lz);
            const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
            meta[q] = 0;
            if constexpr(!TABLE) cells[q] = 0;
            if(own(q)) {
                const uint32_t c = (uint32_t)(gx + (int64_t)nx * (gy + (int64_t)ny * gz));
                uint32_t row = 0;
                if constexpr(TABLE) row = a.op64.codes ? a.op64.codes[c] : (lz * 3 + pos(gy, ny)) * 3 + pos(gx, nx);
                if constexpr(!TABLE) cells[q] = c;
                meta[q] = (uint32_t)((lx + hx_) + ex * ((ly + hy_) + ey * (lz + hz_))) | (row << 16);
            }
        }
        __syncthreads();
    }

    static __device__ __forceinline__ int pos(int i, int len) { return i == 0 ? 0 : (i == len - 1 ? 2 : 1); }

    // rows [row][P] of the tile: the classes of its layers, or the codes
    template <typename TC> __device__ __forceinline__ void fill_table(const OpView<TC> &op, int rows, TC *t) {
        for(int j = tid; j < rows * P; j += T) {
            const int i = j / P, k = j - i * P;
            if(op.codes) t[j] = op.ctab[j];
            else {
                const bool in = z0 + i / 9 < op.nz;
                t[j] = op.table[(in ? ((int64_t)z0 * 9 + i) * 27 : 0) + slot_of(RowPattern<P>::o[k][0], RowPattern<P>::o[k][1], RowPattern<P>::o[k][2])];
            }
        }
    }

    // Neighbour strides in ext.  The empty asm hides them from the compiler:
    // where both a float and a double array were indexed with the same strides
    // it derived the address 4 d from 8 d with the wrong sign for d = -1.
    struct Strides {
        int x, y, z;
        __device__ __forceinline__ int of(int k) const {
            return RowPattern<P>::o[k][0] * x + RowPattern<P>::o[k][1] * y + RowPattern<P>::o[k][2] * z;
        }
    };
    __device__ __forceinline__ Strides strides() const {
        Strides d{__builtin_amdgcn_readfirstlane(hx_), __builtin_amdgcn_readfirstlane(dy), __builtin_amdgcn_readfirstlane(dz)};
        asm volatile("" : "+s"(d.x), "+s"(d.y), "+s"(d.z));
        return d;
    }

    // meta of own cell q.  (The empty asm keeps the compiler from forming the
    // addresses of all own cells ahead of the loops and holding them in
    // registers.)
    __device__ __forceinline__ uint32_t about(int q) const {
        uint32_t m = meta[q];
        asm volatile("" : "+v"(m));
        return m;
    }
    __device__ __forceinline__ int at(int q) const { return (int)(about(q) & 0xffff); }

    // keeps the operands of at most nine terms (or four cells) in registers
    // where registers are few
    template <bool ON, int EVERY = 9> static __device__ __forceinline__ void breathe(int k) {
        if constexpr(ON)
            if(k % EVERY == EVERY - 1) __builtin_amdgcn_sched_barrier(0);
    }

    // row of own cell q times the values v around it
    template <typename TC> __device__ __forceinline__ TC row_times(const OpView<TC> &op, const TC *table, int q, const TC *v) const {
        const uint32_t m = about(q);
        const int e = m & 0xffff;
        const Strides d = strides();
        TC acc = TC(0);
        if constexpr(TABLE) {
            const TC *row = table + (m >> 16) * P;
#pragma unroll
            for(int k = 0; k < P; k++) acc += row[k] * v[e + d.of(k)];
        } else {
            uint32_t c = cells[q];
            asm volatile("" : "+v"(c));
            const TC *row = op.percell + c;
            int64_t n = op.n;
            asm volatile("" : "+s"(n));  // (else 27 row addresses are kept in scalar registers, and spilled)
#pragma unroll
            for(int k = 0; k < P; k++) {
                acc += *row * v[e + d.of(k)];
                row += n;
            }
        }
        // one row's operands in registers at a time, two rows' with a table
        if(RPT > 1 && (!TABLE || q % 2 == 1)) __builtin_amdgcn_sched_barrier(0);
        return acc;
    }

    // Load the words p[0..N) again and again until all of them carry this
    // exchange's epoch; their values.  All N loads are in flight together, so a
    // wait ends one load's latency after the last word has arrived.
    template <int N> __device__ __forceinline__ void await(const u64 *const (&p)[N], uint32_t (&h)[N], bool &bad) {
        u64 v[N];
        u64 began = 0;
        bool last = bad;  // an earlier wait of this exchange has ended without its words
        for(int n = 1;; n++) {
            bool all = true;
#pragma unroll
            for(int k = 0; k < N; k++) v[k] = word_load(p[k]);
#pragma unroll
            for(int k = 0; k < N; k++) all &= (uint32_t)(v[k] >> 32) == epoch;
            if(all) break;
            if(last) {
                bad = true;
                break;
            }
            if((n & 63) == 0 || a.wait_ticks == 0) {
                const u64 now = wall_clock64();
                if(began == 0) began = now;
                // (one more look at the words follows, and counts: a wave that was
                // held up itself finds them there)
                if(now - began >= a.wait_ticks || __hip_atomic_load(&a.st->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == kResidentTimeout)
                    last = true;
            }
        }
#pragma unroll
        for(int k = 0; k < N; k++) h[k] = (uint32_t)v[k];
    }

    // waves that add up the blocks' sums; the others receive the halo
    __device__ __forceinline__ int sum_waves() const { return a.nblocks > kSumBlocks * kSumLoads ? kMaxSumWaves : 1; }

    // the neighbour eight lanes on, round each row of 16
    static __device__ __forceinline__ double row_ror8(double v) {
        struct Halves {
            int lo, hi;
        } h = __builtin_bit_cast(Halves, v);
        h.lo = __builtin_amdgcn_update_dpp(0, h.lo, 0x128, 0xf, 0xf, false);
        h.hi = __builtin_amdgcn_update_dpp(0, h.hi, 0x128, 0xf, 0xf, false);
        return __builtin_bit_cast(double, h);
    }

    // Adds a value of blocks i + sub, i + sub + 8, ... (N of them) to sum; valid
    // in the lanes of low words.
    template <int N>
    __device__ __forceinline__ void add_sums(const u64 *S, int i, int sub, int word, double &sum, bool &bad) {
        const u64 *p[N];
#pragma unroll
        for(int j = 0; j < N; j++) {
            const int b = i + sub + j * kSumBlocks;
            p[j] = S + (size_t)kSumWords * (b < a.nblocks ? b : a.nblocks - 1) + word;
        }
        uint32_t h[N];
        await<N>(p, h, bad);
#pragma unroll
        for(int j = 0; j < N; j++) {
            const uint32_t high = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h[j], 0xB1, 0xf, 0xf, false);  // the other lane of the pair
            if(i + sub + j * kSumBlocks < a.nblocks) sum += join(h[j], high);
        }
    }

    // Halo values i0, i0 + step, ... (M of them; past the end: the first again).
    template <typename T2, int M, class Store>
    __device__ __forceinline__ void receive(const u64 *W, int i0, int step, bool &bad, Store &&store) {
        constexpr int K = kWords<T2>;
        const u64 *p[M * K];
        int i[M];
#pragma unroll
        for(int j = 0; j < M; j++) {
            i[j] = i0 + j * step < nh ? i0 + j * step : i0;
            const u64 *w = W + (size_t)K * hword[i[j]];
#pragma unroll
            for(int k = 0; k < K; k++) p[j * K + k] = w + k;
        }
        uint32_t h[M * K];
        await<M * K>(p, h, bad);
#pragma unroll
        for(int j = 0; j < M; j++) {
            if constexpr(K == 1) store(i[j], __uint_as_float(h[j]));
            else store(i[j], join(h[2 * j], h[2 * j + 1]));
        }
    }

    // Wait for all blocks' sums (wave 0) and the halo values (the other waves)
    // of this exchange; both totals to every thread.  False when a wait ended
    // without its words.
    template <typename T2, class Store> __device__ __forceinline__ bool finish_exchange(double (&t)[kSums], Store &&store) {
        const u64 *W = a.words + (size_t)(epoch & 1) * ((size_t)a.nblocks * RPT * T * 2);
        const u64 *S = a.sums + (size_t)(epoch & 1) * ((size_t)a.nblocks * kSumWords);
        bool bad = false;
        const int nsum = sum_waves();
        if(wave < nsum) {
            // lane 8 i + k takes word k of block i of eight: a load touches
            // eight lines once, where a lane to a block touched 64 lines in
            // each of six loads (168 blocks: an exchange 5.9 -> 4.9 us).  Each
            // line stays one block's: with the sums laid out by word, eight
            // blocks to a line, 128 blocks took 2.8 us where now it is 2.3.
            const int word = (lane & 7) < 2 * kSums ? lane & 7 : 0, sub = lane >> 3;
            double sum = 0.0;
            for(int i = wave * kSumBlocks * kSumLoads; i < a.nblocks; i += nsum * kSumBlocks * kSumLoads) {
                const int left = (a.nblocks - i + kSumBlocks - 1) / kSumBlocks;
                if(left <= kSumLoads / 4) add_sums<kSumLoads / 4>(S, i, sub, word, sum, bad);
                else if(left <= kSumLoads / 2) add_sums<kSumLoads / 2>(S, i, sub, word, sum, bad);
                else add_sums<kSumLoads>(S, i, sub, word, sum, bad);
            }
            sum += row_ror8(sum);
            // four rows of 16 lanes: their sums are added after the barrier
            if((lane & 15) < 2 * kSums && (lane & 1) == 0) part[kSums * NW + (wave * 4 + (lane >> 4)) * kSums + ((lane & 15) >> 1)] = sum;
        } else {
            // (the edge cells' words keep their places in the tile, each cell
            // written by its own thread as soon as it is known: packed face by
            // face, in fewer lines but several waves to a line, the exchange of
            // 128 blocks took 0.5 us longer.)
            // The values of up to four words a lane are waited for together,
            // no more than this wave has left
            const int step = T - 64 * nsum;
            for(int i0 = tid - 64 * nsum; i0 < nh; ) {
                const int left = __builtin_amdgcn_readfirstlane((nh - (i0 - lane) + step - 1) / step);
                if(left == 1) receive<T2, 1>(W, i0, step, bad, store), i0 += step;
                else if(left == 2 || sizeof(T2) == 8) receive<T2, 2>(W, i0, step, bad, store), i0 += 2 * step;
                else receive<T2, sizeof(T2) == 8 ? 2 : 4>(W, i0, step, bad, store), i0 += 4 * step;
            }
        }
        if(bad) flags[0] = 1;
        __syncthreads();
#pragma unroll
        for(int k = 0; k < kSums; k++) {
            const double *v = part + kSums * NW + k;
            t[k] = (v[0] + v[kSums]) + (v[2 * kSums] + v[3 * kSums]);
            if(nsum == 2) t[k] += (v[4 * kSums] + v[5 * kSums]) + (v[6 * kSums] + v[7 * kSums]);
        }
        return flags[0] == 0;
    }

    static __device__ __forceinline__ double join(uint32_t lo, uint32_t hi) { return __longlong_as_double((long long)(((u64)hi << 32) | lo)); }

    // One exchange: own boundary values and this thread's sums out, halo values
    // (through `store`) and the totals in.
    template <typename T2, class Get, class Store>
    __device__ __forceinline__ bool exchange(Get &&value, double (&t)[kSums], Store &&store) {
        epoch++;
        u64 *W = a.words + (size_t)(epoch & 1) * ((size_t)a.nblocks * RPT * T * 2);
        u64 *S = a.sums + (size_t)(epoch & 1) * ((size_t)a.nblocks * kSumWords);
#pragma unroll
        for(int q = 0; q < RPT; q++) {
            if((edge >> q) & 1u) put_value(W + (size_t)kWords<T2> * ((size_t)block * (RPT * T) + local(q)), epoch, value(q));
            breathe<RPT == 32, 8>(q);
        }
        wave_sums(t);
        if(lane == kSumLane) {
#pragma unroll
            for(int k = 0; k < kSums; k++) part[k * NW + wave] = t[k];
        }
        __syncthreads();
        if(a.nblocks == 1) {
#pragma unroll
            for(int k = 0; k < kSums; k++) {
                t[k] = 0.0;
#pragma unroll
                for(int i = 0; i < NW; i++) t[k] += part[k * NW + i];
            }
            return true;
        }
        if(tid < 2 * kSums) {
            double total = 0.0;
#pragma unroll
            for(int i = 0; i < NW; i++) total += part[(tid >> 1) * NW + i];
            const u64 bits = (u64)__double_as_longlong(total);
            word_store(&S[(size_t)block * kSumWords + tid], tagged(epoch, (tid & 1) ? (uint32_t)(bits >> 32) : (uint32_t)bits));
        }
        return finish_exchange<T2>(t, store);
    }

    // CG in TV on A d = r, added to d: on entry ext holds r (with halo, padding
    // zero), rr = r.r.  Returns the status through its arguments; false after a
    // wait that did not end.
    __device__ __forceinline__ bool cg(TV (&d)[RPT], double rr, double tol, int &iters, double &rr_end) {
        // With many cells a thread p lies in LDS, where x was: in registers the
        // 32 cells of a thread spilled (4M-cell batch: 950 -> 720 us a step).
        constexpr bool kLdsP = MIXED && RPT == 32;
        TV preg[kLdsP ? 1 : RPT], s[RPT];
        TV *const pl = ext + ex * ey * ez;
        auto p = [&](int q) -> TV & {
            if constexpr(kLdsP) return pl[at(q)];
            else return preg[q];
        };
#pragma unroll
        for(int q = 0; q < RPT; q++) {
            s[q] = TV(0);
            if(!kLdsP || own(q)) p(q) = TV(0);
        }
        TV keep[kKeepRows ? RPT : 1][kKeepRows ? P : 1];
        if constexpr(kKeepRows) {
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                uint32_t c = cells[q];
                asm volatile("" : "+v"(c));  // (read in every sweep, not kept through the residual's product)
#pragma unroll
                for(int k = 0; k < P; k++) keep[q][k] = (view()->percell + (int64_t)k * view()->n)[c];
            }
        }
        for(int i = tid; i < nh; i += T) {
            hs[i] = TV(0);
            if constexpr(MIXED) hp[i] = hd[i] = TV(0);
        }
        __syncthreads();
        double beta = 0.0, pq = 0.0;
        for(int k = 0;; k++) {
            // w = A r; r.r, r.w, r.s + p.w
            double t[kSums] = {0.0, 0.0, 0.0};
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                w[q] = TV(0);
                if(!own(q)) continue;
                if constexpr(kKeepRows) {
                    const int e = at(q);
                    const Strides sd = strides();
#pragma unroll
                    for(int j = 0; j < P; j++) {
                        w[q] += keep[q][j] * ext[e + sd.of(j)];
                    }
                } else {
                    w[q] = row_times<TV>(*view(), tab, q, ext);
                }
                const TV r = ext[at(q)];
                t[0] += (double)r * (double)r;
                t[1] += (double)r * (double)w[q];
                t[2] += (double)r * (double)s[q] + (double)p(q) * (double)w[q];
            }
            if(!exchange<TV>([&](int q) { return w[q]; }, t, [&](int i, TV v) { hw[i] = v; })) return false;
            if(k > 0) {
                iters = 1 + k;
                rr_end = t[0];
                if((t[0] <= tol) || (iters >= a.max_its) || (t[0] != t[0])) return true;
                beta = t[0] / rr;
                rr = t[0];
            }
            pq = t[1] + beta * (t[2] + beta * pq);
            const TV al = (TV)(rr / pq), be = (TV)beta;
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                if(!own(q)) continue;
                TV &r = ext[at(q)];
                const TV ro = r;
                s[q] = fused(be, s[q], w[q]);
                const TV pv = fused(be, p(q), ro);
                p(q) = pv;
                d[q] = fused(al, pv, d[q]);
                r = fused(-al, s[q], ro);
                breathe<RPT == 32, 8>(q);
            }
            for(int i = tid; i < nh; i += T) {
                TV &r = ext[hext[i]];
                const TV ro = r, sv = fused(be, hs[i], hw[i]);
                hs[i] = sv;
                if constexpr(MIXED) {
                    const TV pv = fused(be, hp[i], ro);
                    hp[i] = pv;
                    hd[i] = fused(al, pv, hd[i]);
                }
                r = fused(-al, sv, ro);
            }
            __syncthreads();
        }
    }

    // The halo repeats its owners' operations, so that its r, p, d and x are
    // theirs bit for bit: fused on both sides by name, not as the compiler likes.
    static __device__ __forceinline__ float fused(float x, float y, float z) { return __builtin_fmaf(x, y, z); }
    static __device__ __forceinline__ double fused(double x, double y, double z) { return __builtin_fma(x, y, z); }

    __device__ __forceinline__ const OpView<TV> *view() const {
        if constexpr(MIXED) return &a.op32;
        else return &a.op64;
    }

    __device__ __forceinline__ void zero_ext(int ne_words) {
        uint32_t *p = (uint32_t *)ext64;
        for(int i = tid; i < ne_words; i += T) p[i] = 0u;
        __syncthreads();
    }

    __device__ __forceinline__ void note(int its, int outer, int inner, double err) {
        if(block == 0 && tid == 0) {
            ResidentStatus *st = a.st;
            st->epoch = epoch;
            st->solves += 1;
            st->cg_total += its;
            st->inner_total += inner;
            st->outer_total += outer;
            st->last_its = its;
            st->last_outer = outer;
            st->last_err = err;
            if(err != err) st->stop = kResidentNan;
        }
    }
    __device__ __forceinline__ void timed_out() {
        if(tid == 0) {
            __hip_atomic_fetch_max(&a.st->left, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.st->stop, (int32_t)kResidentTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }

    __device__ __forceinline__ void run(char *lds) {
        place();
        constexpr bool kHold = holds_xb(MIXED, P, RPT, TABLE);
        double xh[kHold ? RPT : 1], bh[kHold ? RPT : 1];
        if constexpr(kHold) {
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                const int64_t c = own(q) ? cell(q) : 0;
                xh[q] = a.x[c];
                bh[q] = a.b[c];
            }
        }
        setup(lds);
        if(flags[0]) return;  // an earlier solve, or another block of this one, has stopped the run
        epoch = a.st->epoch;
        const int ne = ex * ey * ez;
        TV d[RPT];
        double tol_abs = 0.0, rr = 0.0;
        int inner_total = 0, corrections = 0;
        for(int sweep = 0;; sweep++) {
            // x with its halo into LDS, corrected by the last sweep's d
            zero_ext(2 * ne);
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                if(!own(q)) continue;
                double xn;
                if constexpr(kHold) {
                    if(sweep > 0) xh[q] += (double)d[q];
                    xn = xh[q];
                } else {
                    const int64_t c = cell(q);
                    xn = a.x[c];
                    if(sweep > 0) {
                        xn += (double)d[q];
                        a.x[c] = xn;
                    }
                }
                ext64[at(q)] = xn;
                breathe<RPT == 32, 8>(q);
            }
            for(int i = tid; i < nh; i += T) {
                double xn;
                if constexpr(MIXED) {
                    if(sweep == 0) xn = a.x[a.cells[(size_t)block * a.halo + i].cell];
                    else xn = hx[i] + (double)hd[i];
                    hx[i] = xn;
                } else {
                    xn = a.x[a.cells[(size_t)block * a.halo + i].cell];
                }
                ext64[hext[i]] = xn;
            }
            __syncthreads();
            // r = b - A x in FP64, r.r, b.b
            double t[kSums] = {0.0, 0.0, 0.0};
            TV r[RPT];
#pragma unroll
            for(int q = 0; q < RPT; q++) {
                r[q] = TV(0);
                if(!own(q)) continue;
                double bc;
                if constexpr(kHold) bc = bh[q];
                else bc = a.b[cell(q)];
                const double rc = bc - row_times<double>(a.op64, MIXED ? tab64 : (const double *)tab, q, ext64);
                r[q] = (TV)rc;
                t[0] += rc * rc;
                t[1] += bc * bc;
                breathe<RPT == 32, 4>(q);
            }
            __syncthreads();
            zero_ext(MIXED ? ne : 2 * ne);
#pragma unroll
            for(int q = 0; q < RPT; q++)
                if(own(q)) ext[at(q)] = r[q];
            if(!exchange<TV>([&](int q) { return ext[at(q)]; }, t, [&](int i, TV v) { ext[hext[i]] = v; })) {
                timed_out();
                return;
            }
            const double bb = t[1];
            rr = t[0];
            if(sweep == 0) tol_abs = a.tol_dev ? *a.tol_dev : (a.rel_tol > 0.0 ? a.rel_tol * a.rel_tol * bb : a.tol);
            int iters = 1;
            double rr_end = rr;
            if constexpr(!MIXED) {
                if(!(rr >= tol_abs) || a.max_its <= 1) {
                    note(1, 1, 0, rr);
                    return;
                }
#pragma unroll
                for(int q = 0; q < RPT; q++) {
                    if constexpr(kHold) d[q] = xh[q];
                    else d[q] = own(q) ? a.x[cell(q)] : 0.0;
                }
                if(!cg(d, rr, tol_abs, iters, rr_end)) {
                    timed_out();
                    return;
                }
#pragma unroll
                for(int q = 0; q < RPT; q++)
                    if(own(q)) a.x[cell(q)] = d[q];
                note(iters, 1, iters - 1, rr_end);
                return;
            } else {
                if(!(rr > tol_abs) || sweep >= a.max_outer || rr != rr) {
                    if constexpr(kHold) {
                        if(sweep > 0) {
#pragma unroll
                            for(int q = 0; q < RPT; q++)
                                if(own(q)) a.x[cell(q)] = xh[q];
                        }
                    }
                    note(inner_total + 1, corrections + 1, inner_total, rr);
                    return;
                }
                const double t_rel = a.inner_rel * a.inner_rel * rr;
#pragma unroll
                for(int q = 0; q < RPT; q++) d[q] = TV(0);
                if(!cg(d, rr, t_rel > 0.5 * tol_abs ? t_rel : 0.5 * tol_abs, iters, rr_end)) {
                    timed_out();
                    return;
                }
                inner_total += iters - 1;
                corrections++;
                __syncthreads();  // every wave is past its last use of ext, hs and hw
            }
        }
    }
};

template <bool MIXED, int P, int T, int RPT, bool TABLE>
__global__ __launch_bounds__(T) void k_resident(ResidentArgs a) {
    extern __shared__ __align__(16) char resident_lds[];
    Resident<MIXED, P, T, RPT, TABLE> solve(a);
    solve.run(resident_lds);
}

__global__ void k_resident_reset(u64 *words, size_t nwords, u64 *sums, size_t nsums, ResidentStatus *st) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    for(size_t k = i; k < nwords; k += step) words[k] = 0;
    for(size_t k = i; k < nsums; k += step) sums[k] = 0;
    if(i == 0) {
        st->epoch = 0;
        st->left = 0;
        st->stop = kResidentGoing;
    }
}

template <int A> using IC = std::integral_constant<int, A>;

// f(kernel) for a plan
template <bool MIXED, class F> void with_kernel(int P, int threads, int rpt, bool table, F &&f) {
    auto by_shape = [&](auto P_, auto T_) {
        constexpr int PP = decltype(P_)::value;
        constexpr bool TT = decltype(T_)::value != 0;
        auto one = [&](auto N_, auto R_) {
            constexpr int NN = decltype(N_)::value, RR = decltype(R_)::value;
            if constexpr(built(MIXED, PP, NN, RR, TT))
                if(threads == NN && rpt == RR) f(&k_resident<MIXED, PP, NN, RR, TT>);
        };
        one(IC<256>{}, IC<1>{});
        one(IC<256>{}, IC<2>{});
        one(IC<512>{}, IC<2>{});
        one(IC<512>{}, IC<4>{});
        one(IC<512>{}, IC<8>{});
        one(IC<512>{}, IC<32>{});
    };
    auto by_table = [&](auto P_) {
        if(table) by_shape(P_, IC<1>{});
        else by_shape(P_, IC<0>{});
    };
    if(P == 7) by_table(IC<7>{});
    else if(P == 19) by_table(IC<19>{});
    else by_table(IC<27>{});
}

// operator storage that the kernels read: 1 class table, 2 code table, 0 per-cell rows, -1 none
template <typename TC> int storage(const OpView<TC> &op) {
    if(op.thin) return -1;
    if(op.table) return 1;
    if(op.codes) return 2;
    return op.percell ? 0 : -1;
}

size_t lds_bytes(bool mixed, int P, const ResidentGeom &g, int mode, const int (&h)[3]) {
    auto up = [](size_t b) { return (b + 15) / 16 * 16; };
    const size_t ne = (size_t)(g.bx + 2 * h[0]) * (g.by + 2 * h[1]) * (g.bz + 2 * h[2]), w = mixed ? 4 : 8, nh = (size_t)g.halo;
    size_t b = up(8 * ne) + 2 * up(w * nh) + (mixed ? 2 * up(w * nh) + up(8 * nh) : 0) + up(4 * nh) + up(2 * nh) + up(8 * kSums * (g.threads / 64 + 4 * kMaxSumWaves)) + up(8);
    if(mode > 0) {
        const size_t rows = mode == 2 ? kCodes : 9 * (size_t)g.bz;
        b += up(w * rows * P) + (mixed ? up(8 * rows * P) : 0);
    }
    return b;
}

// The tiles of a shape for which an exchange and the work of
// an iteration cost least by the model below (false: none fits).
bool best_tiles(const int (&L)[3], int P, bool mixed, int mode, Shape shape, int max_blocks, ResidentGeom *best, double *cost) {
    const int T = shape.threads, rpt = shape.rpt;
    bool found = false;
    for(int tz = 1; tz <= L[2] && tz <= max_blocks; tz++) {
        const int bz = (L[2] + tz - 1) / tz;
        if((int64_t)(tz - 1) * bz >= L[2] || (mode == 1 && bz > kTableLayers)) continue;
        for(int ty = 1; ty <= L[1] && tz * ty <= max_blocks; ty++) {
            const int by = (L[1] + ty - 1) / ty;
            if((int64_t)(ty - 1) * by >= L[1]) continue;
            for(int tx = 1; tx <= L[0] && tz * ty * tx <= max_blocks; tx++) {
                const int bx = (L[0] + tx - 1) / tx;
                if((int64_t)(tx - 1) * bx >= L[0]) continue;
                const int64_t cells = (int64_t)bx * by * bz;
                if(cells > (int64_t)rpt * T) continue;
                const int h[3] = {L[0] > 1, L[1] > 1, L[2] > 1};
                const int64_t ne = (int64_t)(bx + 2 * h[0]) * (by + 2 * h[1]) * (bz + 2 * h[2]);
                if(ne >= 65536) continue;
                ResidentGeom g{};
                g.bx = bx;
                g.by = by;
                g.bz = bz;
                g.tx = tx;
                g.ty = ty;
                g.tz = tz;
                g.rpt = rpt;
                g.threads = T;
                const int64_t faces = (tx > 1 ? 2 : 0) * (int64_t)by * bz + (ty > 1 ? 2 : 0) * (int64_t)bx * bz + (tz > 1 ? 2 : 0) * (int64_t)bx * by;
                g.halo = (int)(P == 7 ? faces : (tx * ty * tz > 1 ? ne - cells : 0));
                g.lds = lds_bytes(mixed, P, g, mode, h);
                if(g.lds > 160 * 1024) continue;
                const int blocks = tx * ty * tz;
                // us: block sums, the sums of all blocks, halo words and rows per
                // thread (128 -> 256 blocks with half the rows: 64 x 64 x 16 FP64
                // 69 -> 75 us a step, 256 x 256 FP32 53 -> 59; 168 blocks of 2,900
                // cells -> 252 of 1,900: 200 -> 179)
                const double c = 1.0 + (T > 256 ? 0.3 : 0.0) + (blocks > 1 ? 0.8 + 0.006 * blocks : 0.0) +
                                 0.08 * ((g.halo + T - 65) / (T - 64)) * (mixed ? 1.0 : 1.5) +
                                 ((cells + T - 1) / T) * (T / 256) * (0.05 + 0.03 * P);
                if(!found || c < *cost) {
                    found = true;
                    *best = g;
                    *cost = c;
                }
            }
        }
    }
    return found;
}

// Halo cells of every tile: those of the box that lie next to it and that the
// row pattern reaches, [block][g.halo], and their counts.  Direction by
// direction, so that consecutive cells are consecutive words of one owner.
std::vector<HaloCell> halo_cells(const int (&L)[3], int P, const ResidentGeom &g, std::vector<int> *count) {
    const int blocks = g.tx * g.ty * g.tz, b[3] = {g.bx, g.by, g.bz}, t[3] = {g.tx, g.ty, g.tz};
    const int h[3] = {L[0] > 1, L[1] > 1, L[2] > 1};
    std::vector<HaloCell> list((size_t)blocks * g.halo);
    count->assign(blocks, 0);
    for(int blk = 0; blk < blocks; blk++) {
        const int tile[3] = {blk % t[0], (blk / t[0]) % t[1], blk / (t[0] * t[1])};
        int n = 0;
        for(int dir = 0; dir < 27; dir++) {
            const int o[3] = {dir % 3 - 1, dir / 3 % 3 - 1, dir / 9 - 1};
            const int out = abs(o[0]) + abs(o[1]) + abs(o[2]);
            if(out == 0 || (P == 7 && out > 1)) continue;
            int lo[3], hi[3], owner[3];
            bool in = true;
            for(int k = 0; k < 3; k++) {
                owner[k] = tile[k] + o[k];
                in = in && owner[k] >= 0 && owner[k] < t[k];
                const int len = std::min(b[k], L[k] - tile[k] * b[k]);  // the tile's cells in the box
                lo[k] = o[k] < 0 ? -1 : (o[k] > 0 ? b[k] : 0);
                hi[k] = o[k] == 0 ? len - 1 : lo[k];
            }
            if(!in) continue;
            const uint32_t first = (uint32_t)((owner[0] + t[0] * (owner[1] + t[1] * owner[2])) * (g.rpt * g.threads));
            for(int z = lo[2]; z <= hi[2]; z++)
                for(int y = lo[1]; y <= hi[1]; y++)
                    for(int x = lo[0]; x <= hi[0]; x++) {
                        const int l[3] = {x - o[0] * b[0], y - o[1] * b[1], z - o[2] * b[2]};  // its place in the owner
                        HaloCell &c = list[(size_t)blk * g.halo + n++];
                        c.word = first + (uint32_t)(l[0] + b[0] * (l[1] + b[1] * l[2]));
                        c.cell = (uint32_t)((tile[0] * b[0] + x) +
                                            (int64_t)L[0] * ((tile[1] * b[1] + y) + (int64_t)L[1] * (tile[2] * b[2] + z)));
                        c.ext = (uint32_t)((x + h[0]) + (b[0] + 2 * h[0]) * ((y + h[1]) + (b[1] + 2 * h[1]) * (z + h[2])));
                        c.pad = 0;
                    }
        }
        (*count)[blk] = n;
    }
    return list;
}

}  // namespace

int resident_plan(ResidentPlan *p, const OpView<double> &op64, const OpView<float> *op32, const CgConfig &cfg) {
    const int mode = storage(op64), mixed = op32 != nullptr;
    const int P = mode == 1 ? op64.full_pat : op64.pat;
    if(p->state != 0 && p->nx == op64.nx && p->ny == op64.ny && p->nz == op64.nz && p->pat == P && p->mode == mode && p->mixed == mixed)
        return 0;
    const uint64_t ticks = p->wait_ticks;
    if(resident_release(p)) return -1;
    p->wait_ticks = ticks;
    p->nx = op64.nx;
    p->ny = op64.ny;
    p->nz = op64.nz;
    p->pat = P;
    p->mode = mode;
    p->mixed = mixed;
    p->state = -1;
    if(mode < 0 || (op32 && storage(*op32) != mode)) return 0;
    int dev = 0, cus = 0;
    MONO_CHECK(hipGetDevice(&dev));
    MONO_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int L[3] = {op64.nx, op64.ny, op64.nz};
    const int max_blocks = std::min(cus, 256);
    bool found = false;
    double cost = 0.0;
    for(const Shape shape : kShapes) {
        if(!built(mixed, P, shape.threads, shape.rpt, mode > 0)) continue;
        ResidentGeom g;
        double c = 0.0;
        if(!best_tiles(L, P, mixed, mode, shape, max_blocks, &g, &c)) continue;
        if(!found || c < cost) {
            p->g = g;
            cost = c;
        }
        found = true;
    }
    if(!found) return 0;
    ResidentGeom &g = p->g;
    const int blocks = g.tx * g.ty * g.tz;
    int per_cu = 0;
    hipError_t err = hipSuccess;
    auto query = [&](auto kernel) {
        const void *k = reinterpret_cast<const void *>(kernel);
        err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(160 * 1024));
        if(err == hipSuccess) err = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, g.threads, g.lds);
    };
    if(mixed) with_kernel<true>(P, g.threads, g.rpt, mode > 0, query);
    else with_kernel<false>(P, g.threads, g.rpt, mode > 0, query);
    MONO_CHECK(err);
    if((int64_t)per_cu * cus < blocks) return 0;
    g.cooperative = (int64_t)per_cu * cus < 2 * (int64_t)blocks;
    if(blocks > 1) {
        p->words_bytes = sizeof(u64) * 2 * (size_t)blocks * g.rpt * g.threads * 2;
        p->sums_bytes = sizeof(u64) * 2 * (size_t)blocks * kSumWords;
        MONO_CHECK(hipMalloc(&p->words, p->words_bytes));
        MONO_CHECK(hipMalloc(&p->sums, p->sums_bytes));
        std::vector<int> count;
        const std::vector<HaloCell> list = halo_cells(L, P, g, &count);
        MONO_CHECK(hipMalloc(&p->cells, sizeof(HaloCell) * list.size()));
        MONO_CHECK(hipMalloc(&p->ncells, sizeof(int) * count.size()));
        MONO_CHECK(hipMemcpy(p->cells, list.data(), sizeof(HaloCell) * list.size(), hipMemcpyHostToDevice));
        MONO_CHECK(hipMemcpy(p->ncells, count.data(), sizeof(int) * count.size(), hipMemcpyHostToDevice));
    }
    if(getenv("MONO_TRACE_SLOTS"))
        fprintf(stderr, "[mono] resident solve %s, mode %d, %d-point rows, %dx%dx%d: %dx%dx%d tiles of %dx%dx%d, %d threads, %d cells per thread, %zu bytes of LDS, %d per CU%s\n",
                mixed ? "FP32+refine" : "FP64", mode, P, p->nx, p->ny, p->nz, g.tx, g.ty, g.tz, g.bx, g.by, g.bz, g.threads, g.rpt, g.lds,
                per_cu, g.cooperative ? ", cooperative" : "");
    p->state = 1;
    return 0;
}

int resident_release(ResidentPlan *p) {
    if(p->words) MONO_CHECK(hipFree(p->words));
    if(p->sums) MONO_CHECK(hipFree(p->sums));
    if(p->cells) MONO_CHECK(hipFree(p->cells));
    if(p->ncells) MONO_CHECK(hipFree(p->ncells));
    *p = ResidentPlan();
    return 0;
}

int resident_reset(ResidentPlan *plans, int nplans, ResidentStatus *st, hipStream_t s) {
    for(int i = 0; i < nplans; i++) {
        if(i > 0 && plans[i].state != 1) continue;
        k_resident_reset<<<256, 256, 0, s>>>(plans[i].words, plans[i].words_bytes / sizeof(u64), plans[i].sums,
                                             plans[i].sums_bytes / sizeof(u64), st);
        plans[i].cleared = true;
    }
    MONO_CHECK(hipGetLastError());
    return 0;
}

int resident_launch(const ResidentPlan &p, const OpView<double> &op64, const OpView<float> *op32, const double *b, double *x,
                    const CgConfig &cfg, ResidentStatus *st, hipStream_t s) {
    const ResidentGeom &g = p.g;
    ResidentArgs a{};
    a.op64 = op64;
    if(op32) a.op32 = *op32;
    a.bx = g.bx;
    a.by = g.by;
    a.bz = g.bz;
    a.tx = g.tx;
    a.ty = g.ty;
    a.tz = g.tz;
    a.div_bx = (uint32_t)((1ull << 32) / (unsigned)g.bx) + 1u;
    a.div_by = (uint32_t)((1ull << 32) / (unsigned)g.by) + 1u;
    a.nblocks = g.tx * g.ty * g.tz;
    a.halo = g.halo;
    a.b = b;
    a.x = x;
    a.tol = cfg.tol;
    a.rel_tol = cfg.rel_tol;
    a.inner_rel = cfg.inner_rel;
    a.tol_dev = cfg.tol_dev;
    a.max_its = cfg.max_its;
    a.max_outer = cfg.max_outer;
    a.words = p.words;
    a.sums = p.sums;
    a.cells = (const HaloCell *)p.cells;
    a.ncells = p.ncells;
    a.wait_ticks = p.wait_ticks;
    a.st = st;
    hipError_t err = hipSuccess;
    auto launch = [&](auto kernel) {
        if(g.cooperative) {
            void *args[] = {&a};
            err = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(kernel), dim3(a.nblocks), dim3(g.threads), args, (unsigned)g.lds, s);
        } else {
            kernel<<<a.nblocks, g.threads, g.lds, s>>>(a);
            err = hipGetLastError();
        }
    };
    if(op32) with_kernel<true>(p.pat, g.threads, g.rpt, p.mode > 0, launch);
    else with_kernel<false>(p.pat, g.threads, g.rpt, p.mode > 0, launch);
    MONO_CHECK(err);
    return 0;
}

}  // namespace mono
