// Device code shared by the kernels that sum element forces into nodes.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace hoefem {
namespace dev {

// s + component c of the forces that blocks inc_blk, local nodes inc_loc, entries it .. end - 1, hold for a node,
// added in the entries' order (the colors'). The places and then the values of FORCE_BATCH terms are
// read before the first is used: a node of the Tet10 cube has up to 24 terms, each two dependent reads from
// memory, and one after the other they took 13.9 us where the traffic needs 1.
constexpr int FORCE_BATCH = 8;
__device__ inline double force_sum(double s, int it, int end, const int32_t* __restrict__ inc_blk,
                                   const int32_t* __restrict__ inc_loc, int n, const double* __restrict__ fe, int c) {
    for (; it < end; it += FORCE_BATCH) {
        int64_t at[FORCE_BATCH];
        double x[FORCE_BATCH];
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) {
            const int q = min(it + k, end - 1);
            at[k] = ((int64_t)inc_blk[q] * n + inc_loc[q]) * 3 + c;
        }
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) x[k] = fe[at[k]];
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k)
            if (it + k < end) s += x[k];
    }
    return s;
}

}  // namespace dev
}  // namespace hoefem
