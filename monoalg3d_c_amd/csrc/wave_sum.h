// Sums over the 64 lanes of a wave.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mono {

// One step of wave_sums: every sum plus its value from the lane that the DPP
// control CTRL names (0 where that lane or row is masked off).
template <int CTRL, int ROWS, int NR> __device__ __forceinline__ void wave_sum_step(double (&v)[NR]) {
    double u[NR];
#pragma unroll
    for(int k = 0; k < NR; k++) {
        const uint64_t bits = (uint64_t)__double_as_longlong(v[k]);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)bits, CTRL, ROWS, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(bits >> 32), CTRL, ROWS, 0xf, false);
        u[k] = __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
    }
#pragma unroll
    for(int k = 0; k < NR; k++) v[k] += u[k];
    __builtin_amdgcn_sched_barrier(0);
}

// Sums over the wave, valid in its last lane; all lanes take part; fixed order.
// DPP row shifts and broadcasts instead of __shfl: an instruction of the vector
// ALU against a trip through LDS for each half of a double and step.  All sums
// take each step together, so they hide one another's latency.
template <int NR> __device__ __forceinline__ void wave_sums(double (&v)[NR]) {
    wave_sum_step<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    wave_sum_step<0x112, 0xf>(v);
    wave_sum_step<0x114, 0xf>(v);
    wave_sum_step<0x118, 0xf>(v);
    wave_sum_step<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    wave_sum_step<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}
constexpr int kSumLane = 63;  // the lane that holds them

}  // namespace mono
