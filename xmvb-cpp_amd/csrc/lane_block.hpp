// One overlap block per lane: gather and inversion in registers (the pair kernels of pairs_lane.hip, the
// conditioning of the string pairs in strings.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace xmvb_amd {

template <int M>
struct LaneBlock {
    static constexpr int K = M > 0 ? M : 1;
    int R[K], L[K];  // occupied orbitals of the right (ket) and left (bra) strings
    double a[K][K];  // X on entry; X^{-1} after inversion, so D[r][l] = a[l][r]
    double det;
    double inverse, cond;  // max|X^{-1}|; max|X| max|X^{-1}|, infinite for a vanishing pivot
};

template <int M>
__device__ __forceinline__ void occupied(uint32_t mask, int* out) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
        out[k] = __builtin_ctz(mask);
        mask &= mask - 1;
    }
}

// In-place Gauss-Jordan inversion with row pivoting. A row interchange of X is an interchange of
// two ket orbitals, so it is applied to R as well and never undone: the result is the inverse of
// the row-permuted block, paired with the permuted R, which every consumer sums over in any order
// (same-spin terms are symmetric under r <-> r2; the compound W index sorts the pair itself).
// det keeps the sign of the unpermuted block. Returns whether the block stays on the lane path.
template <int M>
__device__ __forceinline__ bool lane_invert(const double* __restrict__ sact, int n, double cond_limit, LaneBlock<M>& b) {
    if constexpr (M == 0) {
        b.det = b.cond = b.inverse = 1.0;
        return true;
    } else {
        auto& a = b.a;
        double amax = 0.0;
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int j = 0; j < M; ++j) {
                a[i][j] = sact[b.R[i] + n * b.L[j]];
                amax = fmax(amax, fabs(a[i][j]));
            }
        double det = 1.0;
        bool ok = true;
#pragma unroll
        for (int k = 0; k < M; ++k) {
            int p = k;
            double best = fabs(a[k][k]);
#pragma unroll
            for (int i = k + 1; i < M; ++i) {
                const double v = fabs(a[i][k]);
                const bool g = v > best;
                best = g ? v : best;
                p = g ? i : p;
            }
#pragma unroll
            for (int i = k + 1; i < M; ++i) {
                const bool s = p == i;
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    const double t = a[k][j];
                    a[k][j] = s ? a[i][j] : t;
                    a[i][j] = s ? t : a[i][j];
                }
                const int tr = b.R[k];
                b.R[k] = s ? b.R[i] : tr;
                b.R[i] = s ? tr : b.R[i];
            }
            const double pv = a[k][k];
            ok = ok && best > 0.0;
            det = (p != k) ? -det * pv : det * pv;
            const double inv = best > 0.0 ? 1.0 / pv : 0.0;
            a[k][k] = 1.0;
#pragma unroll
            for (int j = 0; j < M; ++j) a[k][j] *= inv;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (i == k) continue;
                const double f = a[i][k];
                a[i][k] = 0.0;
#pragma unroll
                for (int j = 0; j < M; ++j) a[i][j] -= f * a[k][j];
            }
        }
        double ymax = 0.0;
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int j = 0; j < M; ++j) ymax = fmax(ymax, fabs(a[i][j]));
        b.det = det;
        b.inverse = ymax;
        b.cond = ok ? amax * ymax : HUGE_VAL;
        return b.cond < cond_limit;
    }
}

}  // namespace xmvb_amd
