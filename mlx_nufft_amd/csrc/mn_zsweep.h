// Helpers shared by the z-sweep spread (mn_zsweep.hip) and the z-gather
// interpolation (mn_zgather.hip): the workgroup -> (column block, z-segment)
// order, the ES weight and a wave-wide maximum.
#pragma once

#include "mn_common.h"

namespace mn {

// Workgroup index -> (column block bx, by; z-segment seg). The segment
// varies slowest; within a segment the blocks go in bands of ZS_BAND
// consecutive bx rows, bx fastest inside a band. The -x, -y and -xy
// neighbours of a block, which read the same reaching points, are then
// dispatched at most ZS_BAND + 1 workgroups earlier (except across a band
// edge) and run on the same XCD at about the same z. Measured on MI355X with
// 2e7 uniform points on a 512^3 grid: 18 % less HBM fetch than the
// segment-fastest order.
constexpr int ZS_BAND = 16;
__device__ __forceinline__ void zs_block(int64_t wid, int nbx, int nby, int &bx, int &by,
                                         int &seg) {
    const int64_t plane = (int64_t)nbx * nby;
    seg = (int)(wid / plane);
    const int64_t r = wid % plane, bandc = (int64_t)ZS_BAND * nby;
    const int b0 = (int)(r / bandc) * ZS_BAND;
    const int tx = min(ZS_BAND, nbx - b0);
    const int local = (int)(r % bandc);
    by = local / tx;
    bx = b0 + local % tx;
}

// ES weight exp(beta (sqrt(1 - z^2) - 1)) at the scaled distance z, as
// exp2(bl2e sqrt|1 - z^2| - bl2e): |z| <= 1 for every tap up to rounding,
// and the absolute value (a free source modifier) stands in for a clamp.
// STABLE: the same exponent as -bl2e z^2 / (1 + sqrt(1 - z^2)), without its
// cancellation near z = 0 (one reciprocal and two products more, 2-3 % of a
// sweep). The grids stored with extents, whose other route sums in fp64, take
// it: with it their transforms are nearer to 64 bits than that route's (eps
// 1e-6: 1.39e-6 against 1.52e-6 on 64 x 48 x 56 modes, 1.46e-6 against 1.58e-6
// on 32 x 40 x 36; 1.57e-6 and 1.69e-6 without it).
template <bool STABLE = false>
__device__ __forceinline__ float zs_es(float z, float bl2e) {
    if constexpr (STABLE) {
        const float z2 = z * z;
        return __builtin_amdgcn_exp2f(
            -bl2e * z2 *
            __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(__builtin_fabsf(1.0f - z2))));
    }
    const float t = __builtin_fmaf(-z, z, 1.0f);
    return __builtin_amdgcn_exp2f(
        __builtin_fmaf(bl2e, __builtin_amdgcn_sqrtf(__builtin_fabsf(t)), -bl2e));
}

// Wave-wide maximum of a small non-negative integer (< 512), by ballots.
__device__ __forceinline__ int wave_max9(int v) {
    int m = 0;
#pragma unroll
    for (int b = 8; b >= 0; --b) {
        const int cand = m | (1 << b);
        if (__ballot(v >= cand)) m = cand;
    }
    return m;
}

}  // namespace mn
