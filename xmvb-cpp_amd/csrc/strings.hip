// Evaluation over the strings of the active space ("string form").
//
// Writing the column h|l> of a determinant overlap in the active orbitals, h_rl = sum_q S_rq ht_ql
// with ht = S_act^-1 h, every operator acts on a determinant as in an orthonormal basis, with the
// transformed integrals ht and gt[ql, q2l2] = sum S^-1_qr S^-1_q2r2 (r l | r2 l2):
//   <d|H|e> = sum_x S_dx Ht_xe,  Ht_xe the Slater-Condon coefficient between the strings of e and of x,
// and S_dx = M_a[d_a, x_a] M_b[d_b, x_b] are minors of S_act. With the determinant coefficients c,
//   f[x_a, x_b] = sum_d M_a[x_a, d_a] c_d M_b[d_b, x_b],   sigma = Ht c,
// the derivative of c^T H c - lambda c^T S c needs no pair of determinants at all:
//   dgt[ql, q2l2] = sum_e c_e <f|E_ql E_q2l2|e> (opposite spin; likewise same spin and dht),
//   dS_act = S^-1 (Z - W), Z_ql = <f|E_ql|sigma - lambda c>, W_qp = sum dgt[ql, Y] gt[pl, Y] + dht_ql ht_pl.
// For the 252 determinants of 10 covalent orbitals that is one product of 252 x 252 matrices and
// sums over single replacements, where the pair kernels invert two blocks and gather 1,100 kernel
// elements for each of 16,002 pairs.
//
// No overlap block is inverted; what matters is the conditioning of S_act itself, and a slot whose S_act^-1
// has an element above kStringInverseLimit keeps the pair kernels (FLAG_STRINGS stays clear). Pairs whose
// regular inverse form loses digits, and those it does not cover, stay with the list kernels
// (k_pairs, k_pairs_singular) in the energy and the gradient, as they do behind the lane kernels: the
// results are those of the pair kernels to their own rounding (kStringListError), whichever form a launch takes.
// Every sum here has a fixed order that does not depend on the launch; the list kernels' rows follow the
// batch unless the launch is pinned.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "lane_block.hpp"
#include "wave.hpp"

namespace xmvb_amd {

namespace {

constexpr int kMaxN = MAX_ACT;

__device__ __forceinline__ double signed_value(double v, uint32_t odd) { return odd >> 31 ? -v : v; }

// ---- S_act^-1 and the route -----------------------------------------------------------------------

// One wavefront per problem: Gauss-Jordan inversion of the symmetric positive definite S_act in LDS (no
// pivoting is needed), ht = S_act^-1 h_act, and the route: the slot takes the string form when no
// element of the inverse exceeds kStringInverseLimit.
__global__ void __launch_bounds__(64) k_string_frame(const SlotDesc* __restrict__ slots, int n) {
    const SlotDesc& sd = slots[blockIdx.z];
    __shared__ double a[kMaxN * kMaxN], hl[kMaxN * kMaxN];
    const int lane = threadIdx.x;
    for (int t = lane; t < n * n; t += 64) {
        a[t] = to_global(sd.sact)[t];
        hl[t] = to_global(sd.hact)[t];
    }
    __syncthreads();
    bool ok = true;
    for (int k = 0; k < n; ++k) {
        const double pivot = a[k * n + k];
        ok = ok && pivot > 0.0;
        const double inv = 1.0 / pivot;
        double next[4];  // n^2 <= 196 elements
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = lane + 64 * u, i = t / n, j = t - i * n;
            if (t >= n * n) continue;
            const double r = a[i * n + k], c = a[k * n + j];
            next[u] = i == k ? (j == k ? inv : c * inv) : (j == k ? -r * inv : a[t] - r * c * inv);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (lane + 64 * u < n * n) a[lane + 64 * u] = next[u];
        __syncthreads();
    }
    double big = 0.0;
    const auto Sinv = to_global(sd.sw.Sinv);
    const auto ht = to_global(sd.sw.ht);
    for (int t = lane; t < n * n; t += 64) {
        const int i = t / n, j = t - i * n;
        const double v = 0.5 * (a[t] + a[j * n + i]);
        big = fmax(big, fabs(v));
        Sinv[t] = v;
        double acc = 0.0;
        for (int r = 0; r < n; ++r) acc += 0.5 * (a[i * n + r] + a[r * n + i]) * hl[r * n + j];
        ht[t] = acc;
    }
    ok = ok && big <= kStringInverseLimit;  // false for NaN
    if (__all(ok) && lane == 0) to_global(sd.flags)[FLAG_STRINGS] = 1;
}

// ---- minors -----------------------------------------------------------------------------------------

constexpr int kMinorRows = 8;

// M[x][y] = det S_act[x, y] over all strings, by expansion along the rows: the minors of the first k
// rows over every k of the M columns, k = 1..M (M 2^(M-1) multiplications, no division), all in
// registers. A thread owns a column string and kMinorRows row strings; the row orbitals are
// uniform, so the M reads of a row are conflict-free LDS reads. FP64 VALU bound.
template <int M>
__global__ void __launch_bounds__(256) k_string_minors(const SlotDesc* __restrict__ slots, int n, StringSpace sp,
                                                       bool beta) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    __shared__ double s[kMaxN * kMaxN];
    for (int t = threadIdx.x; t < n * n; t += blockDim.x) s[t] = to_global(sd.sact)[t];
    __syncthreads();
    const int y = blockIdx.x * blockDim.x + threadIdx.x;
    if (y >= sp.N) return;
    int L[M];
    {
        uint32_t m = sp.mask[y];
#pragma unroll
        for (int k = 0; k < M; ++k) {
            L[k] = __builtin_ctz(m);
            m &= m - 1;
        }
    }
    const auto out = to_global(beta ? sd.sw.Mb : sd.sw.Ma);
    for (int u = 0; u < kMinorRows; ++u) {
        const int x = blockIdx.y * kMinorRows + u;
        if (x >= sp.N) break;
        uint32_t rows = sp.mask[x];
        double D[1 << M];
        D[0] = 1.0;
#pragma unroll
        for (int k = 1; k <= M; ++k) {
            const double* row = s + __builtin_ctz(rows) * n;
            rows &= rows - 1;
            double v[M];
#pragma unroll
            for (int j = 0; j < M; ++j) v[j] = row[L[j]];
#pragma unroll
            for (int c = 1; c < (1 << M); ++c) {
                if (__builtin_popcount(c) != k) continue;
                double acc = 0.0;
                int at = 0;
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    if (!(c >> j & 1)) continue;
                    const double term = v[j] * D[c ^ (1 << j)];
                    acc += ((k - 1 + at) & 1) ? -term : term;
                    ++at;
                }
                D[c] = acc;
            }
        }
        out[(size_t)x * sp.N + y] = D[(1 << M) - 1];
    }
}

// Conditioning of the overlap block of every string pair: 0 where the lane kernels keep it, else the power of
// two above max|X^-1|, or kMaybeSingular where the complete-pivoting rank rule may call it deficient. Every minor of
// S_act is at most 1 (Hadamard's bound, orbitals of unit norm), so max|X| max|X^-1| <= 1 / |det X| and only blocks
// of a small minor are inverted, as the lane kernels do it: a workgroup collects those of its 2,048 unordered
// pairs, then takes one per lane. 192 problems of 10 orbitals 50 us, 32 of 12 122, one of 14 152 (every block inverted and
// both triangles written: 129, 500 and 303). Bound by the reads of M and, beyond 12 orbitals, the inversions.
constexpr int kMaybeSingular = 255, kConditionSteps = 8;
template <int M>
__global__ void __launch_bounds__(256) k_string_condition(const SlotDesc* __restrict__ slots, int n, StringSpace sp,
                                                          bool beta) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!to_global(sd.flags)[FLAG_STRINGS]) return;
    __shared__ double s[kMaxN * kMaxN];
    __shared__ int small[256 * kConditionSteps], smalls;
    for (int t = threadIdx.x; t < n * n; t += blockDim.x) s[t] = to_global(sd.sact)[t];
    if (threadIdx.x == 0) smalls = 0;
    __syncthreads();
    const auto minors = to_global(static_cast<const double*>(beta ? sd.sw.Mb : sd.sw.Ma));
    const auto near = to_global(beta ? sd.sw.nearb : sd.sw.neara);
    const int pairs = sp.N * (sp.N + 1) / 2;  // at most 5.9 million
#pragma unroll
    for (int u = 0; u < kConditionSteps; ++u) {
        const int t = (blockIdx.x * kConditionSteps + u) * 256 + threadIdx.x;
        int x, y;
        unpack_pair(min(t, pairs - 1), x, y);
        const size_t at = (size_t)y * sp.N + x;  // x <= y, lanes along x
        const double det = minors[at];
        if (t >= pairs) continue;
        if (fabs(det) > 1.01 / kLaneConditionDefault) near[at] = 0;
        else small[atomicAdd(&smalls, 1)] = t;  // in any order: each is its own element
    }
    __syncthreads();
    for (int i = threadIdx.x; i < smalls; i += 256) {
        int x, y;
        unpack_pair(small[i], x, y);
        LaneBlock<M> b;
        occupied<M>(sp.mask[x], b.R);
        occupied<M>(sp.mask[y], b.L);
        int code = 0;
        if (!lane_invert<M>(s, n, kLaneConditionDefault, b))  // a NaN counts as singular
            code = b.cond < kLaneConditionMax ? ilogb(b.inverse) + 1 : kMaybeSingular;
        near[(size_t)y * sp.N + x] = (unsigned char)code;
    }
}

// Pairs left to the list kernels (kStringListError), flagged per work item of the lane kernels, so that
// they are listed as the lane kernels' own deferred pairs are, and counted in FLAG_NEAR.
__global__ void __launch_bounds__(256) k_string_list(const SlotDesc* __restrict__ slots, TopoDesc topo) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!to_global(sd.flags)[FLAG_STRINGS]) return;
    const StringTopo& t = topo.str;
    const int na = t.a.N, nb = t.b.N;
    const auto pa = to_global(sd.sw.neara), pb = to_global(sd.sw.nearb);
    const double limit = kStringListError * topo.n_det;
    int count = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < topo.n_lane_pairs;
         i += (long long)gridDim.x * blockDim.x) {
        int d, e;
        unpack_pair(topo.lane_pairs ? (long long)topo.lane_pairs[i] : i, d, e);
        auto at = [](int x, int y, int N) { return x <= y ? (size_t)y * N + x : (size_t)x * N + y; };
        const size_t a = at(t.arank[d], t.arank[e], na), b = at(t.brank[d], t.brank[e], nb);
        const int p = max((int)pa[a], (int)pb[b]);
        const bool listed =
            p == kMaybeSingular || (p > 0 && ldexp(fabs(to_global(sd.sw.Ma)[a] * to_global(sd.sw.Mb)[b]), 3 * p) >= limit);
        to_global(sd.defer_flag)[i] = listed;
        count += listed ? (topo.flip ? 2 : 1) : 0;
    }
#pragma unroll
    for (int off = 32; off; off >>= 1) count += __shfl_xor(count, off, 64);
    if ((threadIdx.x & 63) == 0 && count) atomicAdd(sd.flags + FLAG_NEAR, count);
}

// ---- transformed integrals --------------------------------------------------------------------------

// U[ql][P] = sum_r S^-1_qr (r l | P)
__global__ void __launch_bounds__(256) k_string_half(const SlotDesc* __restrict__ slots, int n, int np) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * n * np) return;
    const int P = t % np, X = t / np, q = X / n, l = X - q * n;
    double acc = 0.0;
    for (int r = 0; r < n; ++r)
        acc += to_global(sd.sw.Sinv)[q * n + r] * to_global(sd.G)[pair_index(pair_index(r, l), P)];
    to_global(sd.sw.U)[t] = acc;
}

// gt[ql][q2 l2] = sum_r2 S^-1_q2r2 U[ql][(r2 l2)]
__global__ void __launch_bounds__(256) k_string_full(const SlotDesc* __restrict__ slots, int n, int np) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x, n2 = n * n;
    if (t >= n2 * n2) return;
    const int X = t / n2, Y = t - X * n2, q2 = Y / n, l2 = Y - q2 * n;
    double acc = 0.0;
    for (int r = 0; r < n; ++r)
        acc += to_global(sd.sw.Sinv)[q2 * n + r] * to_global(sd.sw.U)[X * np + pair_index(r, l2)];
    to_global(sd.sw.gt)[t] = acc;
}

// J[x][ql] = sum of gt[l2 l2][ql] over the occupied l2 of x; F[x][ql] = ht_ql + J - the exchange sum of
// gt[q l2][l2 l]: the string's own field
__global__ void __launch_bounds__(256) k_string_coulomb(const SlotDesc* __restrict__ slots, int n, StringSpace sp,
                                                        bool beta) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    const int n2 = n * n, t = bx * blockDim.x + threadIdx.x;
    if (t >= sp.N * n2) return;
    const int x = t / n2, X = t - x * n2, q = X / n, l = X - q * n;
    const auto gt = to_global(static_cast<const double*>(sd.sw.gt));
    double j = 0.0, k = 0.0;
    for (uint32_t m = sp.mask[x]; m; m &= m - 1) {
        const int l2 = __builtin_ctz(m);
        j += gt[l2 * (n + 1) * n2 + X];
        k += gt[(q * n + l2) * n2 + l2 * n + l];
    }
    to_global(beta ? sd.sw.Jb : sd.sw.Ja)[t] = j;
    to_global(beta ? sd.sw.Fb : sd.sw.Fa)[t] = to_global(sd.sw.ht)[X] + (j - k);
}

__device__ __forceinline__ int below(uint32_t mask, int k) { return __popc(mask & ((1u << k) - 1)); }

// Ht[x][a]: one- and two-electron part of the transformed Hamiltonian between strings of one spin
// (zero beyond double replacements). One thread per element, lanes over a.
__global__ void __launch_bounds__(256) k_string_hamiltonian(const SlotDesc* __restrict__ slots, int n, StringSpace sp,
                                                            bool beta) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const int y = blockIdx.x * blockDim.x + threadIdx.x, x = blockIdx.y, n2 = n * n;
    if (y >= sp.N) return;
    const uint32_t ket = sp.mask[y], bra = sp.mask[x];
    const uint32_t add = bra & ~ket, drop = ket & ~bra;
    const auto gt = to_global(sd.sw.gt);
    const auto ht = to_global(sd.sw.ht);
    const auto F = to_global(beta ? sd.sw.Fb : sd.sw.Fa) + (size_t)y * n2;
    double v = 0.0;
    const int degree = __popc(add);
    if (degree == 0) {
        for (uint32_t m = ket; m; m &= m - 1) {
            const int l = __builtin_ctz(m) * (n + 1);
            v += 0.5 * (ht[l] + F[l]);
        }
    } else if (degree == 1) {
        const int l = __builtin_ctz(drop), q = __builtin_ctz(add);
        v = F[q * n + l];
        if ((below(ket, l) + below(ket ^ (1u << l), q)) & 1) v = -v;
    } else if (degree == 2) {
        const int l = __builtin_ctz(drop), l2 = 31 - __builtin_clz(drop);
        const int q = __builtin_ctz(add), q2 = 31 - __builtin_clz(add);
        v = gt[(q * n + l) * n2 + q2 * n + l2] - gt[(q * n + l2) * n2 + q2 * n + l];
        const uint32_t one = ket ^ (1u << l), mid = one ^ (1u << q);
        const int odd = below(ket, l) + below(one, q) + below(mid, l2) + below(mid ^ (1u << l2), q2);
        if (odd & 1) v = -v;
    }
    to_global(beta ? sd.sw.Hb : sd.sw.Ha)[(size_t)x * sp.N + y] = v;
}

// ---- products of string matrices ---------------------------------------------------------------------

typedef double string_double4 __attribute__((ext_vector_type(4)));

constexpr int kProductTile = 64;   // rows and columns per workgroup, 32 x 32 per wavefront
constexpr int kProductTilesFew = 128;  // launches of fewer 64 x 64 tiles take the 16 x 16 form
constexpr int kProductDepth = 16;  // summation indices staged at a time
constexpr int kProductLd = kProductTile + 16;  // row of a staged block: the four k of a fragment fall on distinct banks

// Tile of a workgroup: all ti x tj of them, or with sym != 0 (C^T = sym C) the ones on and above the diagonal.
__device__ __forceinline__ void product_tile(int at, int tiles_j, int sym, int& ti, int& tj) {
    if (sym) {
        unpack_pair(at, ti, tj);  // ti <= tj
    } else {
        ti = at / tiles_j;
        tj = at - ti * tiles_j;
    }
}

// C[i][j] = sum_k A[k][i] B[k][j] (A symmetric or its transpose stored), one 64 x 64 tile of C per
// workgroup of four wavefronts, v_mfma_f64_16x16x4. The depth-16 blocks of A and B are staged in
// LDS twice over, so the loads of the next block are in flight during the products of this one.
// With sym != 0 only the elements on and above the diagonal are kept and also written below it, times sym.
// Every element is summed in ascending k by one accumulator, so its bits do not depend on the tile or the form.
template <typename PA, typename PB, typename PC>
__device__ __forceinline__ void string_product(PA A, int lda, PB B, int ldb, PC C, int ldc, int ni, int nj, int nk, int ti,
                                               int tj, int sym) {
    __shared__ double As[2][kProductDepth][kProductLd], Bs[2][kProductDepth][kProductLd];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    const int i0 = ti * kProductTile, j0 = tj * kProductTile;
    // thread t stages column t % 64 of rows t / 64 + 4 u
    const int sc = threadIdx.x & 63, sr = threadIdx.x >> 6;
    const int ia = min(i0 + sc, ni - 1), jb = min(j0 + sc, nj - 1);
    double ra[4], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + sr + 4 * u, kc = min(k, nk - 1);
            const double va = A[(size_t)kc * lda + ia], vb = B[(size_t)kc * ldb + jb];
            ra[u] = k < nk ? va : 0.0;
            rb[u] = k < nk ? vb : 0.0;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            As[buf][sr + 4 * u][sc] = ra[u];
            Bs[buf][sr + 4 * u][sc] = rb[u];
        }
    };
    string_double4 acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = string_double4{0.0, 0.0, 0.0, 0.0};
    fetch(0);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < nk; k0 += kProductDepth) {
        const bool more = k0 + kProductDepth < nk;
        if (more) fetch(k0 + kProductDepth);
#pragma unroll
        for (int kk = 0; kk < kProductDepth; kk += 4) {
            double a[2], b[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                a[p] = As[buf][kk + k4][wi + 16 * p + i16];
                b[p] = Bs[buf][kk + k4][wj + 16 * p + i16];
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[p], b[q], acc[p][q], 0, 0, 0);
        }
        if (more) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wi + 16 * p + 4 * v + k4, j = j0 + wj + 16 * q + i16;
                if (i >= ni || j >= nj || (sym && i > j)) continue;
                C[(size_t)i * ldc + j] = acc[p][q][v];
                if (sym && i < j) C[(size_t)j * ldc + i] = sym > 0 ? acc[p][q][v] : -acc[p][q][v];
            }
}

// The same for launches whose 64 x 64 tiles would leave most of the device idle: one 16 x 16 tile per
// wavefront, operands straight from memory, twelve summation steps in flight (one problem of 10 orbitals:
// 23 us staged, 16 workgroups; bounded by load latency either way).
template <typename PA, typename PB, typename PC>
__device__ __forceinline__ void string_product_few(PA A, int lda, PB B, int ldb, PC C, int ldc, int ni, int nj, int nk, int ti,
                                                   int tj, int sym) {
    const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
    const int ia = min(16 * ti + i16, ni - 1), jb = min(16 * tj + i16, nj - 1);
    string_double4 acc = string_double4{0.0, 0.0, 0.0, 0.0};
    constexpr int kAhead = 12;
    for (int k0 = 0; k0 < nk; k0 += 4 * kAhead) {
        double a[kAhead], b[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(k0 + 4 * u + k4, nk - 1);
            a[u] = A[(size_t)k * lda + ia];
            b[u] = B[(size_t)k * ldb + jb];
        }
        __builtin_amdgcn_sched_barrier(0);  // all loads issued before the first product waits for one
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const bool live = k0 + 4 * u + k4 < nk;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(live ? a[u] : 0.0, live ? b[u] : 0.0, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = 16 * ti + 4 * v + k4, j = 16 * tj + i16;
        if (i >= ni || j >= nj || (sym && i > j)) continue;
        C[(size_t)i * ldc + j] = acc[v];
        if (sym && i < j) C[(size_t)j * ldc + i] = sym > 0 ? acc[v] : -acc[v];
    }
}

// K = M Ht: the same-spin Hamiltonian between strings of one spin (symmetric)
template <bool Few>
__global__ void __launch_bounds__(256) k_string_same_spin(const SlotDesc* __restrict__ slots, int N, int tiles, bool beta) {
    int x, z, ti, tj;
    problem_block(x, z);
    const SlotDesc& sd = slots[z];
    if (!string_slot(sd)) return;
    const auto M = to_global(static_cast<const double*>(beta ? sd.sw.Mb : sd.sw.Ma));
    const auto H = to_global(static_cast<const double*>(beta ? sd.sw.Hb : sd.sw.Ha));
    const auto K = to_global(beta ? sd.sw.Kb : sd.sw.Ka);
    const int at = Few ? x * 4 + (int)(threadIdx.x >> 6) : x;
    if (at >= tiles * (tiles + 1) / 2) return;
    product_tile(at, tiles, 1, ti, tj);
    if (Few) string_product_few(M, N, H, N, K, N, N, N, N, ti, tj, 1);
    else string_product(M, N, H, N, K, N, N, N, N, ti, tj, 1);
}

// ---- determinant pairs --------------------------------------------------------------------------------

// H and S between one determinant e (one of its spin-flip couple) and a range of determinants d
// (StringPairItem), one item per wavefront:
//   H_de = K_a M_b + M_a K_b + sum_ij M_a[d_a, x_i] g_e[i][j] M_b[d_b, y_j],
// x_i, y_j the single replacements of e's strings (and the strings themselves, last), g_e the signed
// transformed integrals. g_e stays in registers as matrix-core operands; for 16 determinants at
// a time v_mfma_f64_16x16x4 forms g_e M_b^T (KK steps over j, TI tiles over i), each lane multiplies
// its rows with M_a and the four lane groups are added. The columns of M are read along the
// determinants' strings; the lane groups write the four equal elements (d, e), (e, d) and their partners.
// KK = ceil((replacements + 1) / 4) of the spin with more of them. 192 problems of 10 orbitals: 418 us, of
// which the matrix cores need 75; neither more wavefronts per SIMD (454 us), nor collecting
// the elements in LDS for runs of writes (439 us) helps: about 25 loads of 64 lanes per 16 determinants
// keep the address and cache path busy.
template <int KK>
__global__ void __launch_bounds__(256) k_string_pairs(const SlotDesc* __restrict__ slots, TopoDesc topo) {
    constexpr int TI = (KK + 3) / 4;
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    const StringTopo& t = topo.str;
    const int item = bx * 4 + (threadIdx.x >> 6);
    if (item >= t.npitem) return;
    const int e = t.pitem[item].det, begin = t.pitem[item].begin, end = t.pitem[item].end,
              couple = t.pitem[item].couple;
    const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
    const int a = t.arank[e], b = t.brank[e], n_det = topo.n_det;
    const int n = topo.n, n2 = n * n, na = t.a.N, nb = t.b.N, ia = t.a.noff, ib = t.b.noff;
    const uint32_t* ea = t.a.e1 + (size_t)a * t.a.J;
    const uint32_t* eb = t.b.e1 + (size_t)b * t.b.J;
    const auto gt = to_global(static_cast<const double*>(sd.sw.gt));
    const auto Ja = to_global(static_cast<const double*>(sd.sw.Ja)) + (size_t)a * n2;
    const auto Jb = to_global(static_cast<const double*>(sd.sw.Jb)) + (size_t)b * n2;
    const double both = wave_sum(lane < n && (t.a.mask[a] >> lane & 1) ? Jb[lane * (n + 1)] : 0.0);
    // one unconditional load per element through a selected address: loads under branches would each
    // wait for the ones before (447 us instead of the present time for 192 problems of 10 orbitals)
    uint32_t xe[TI], ye[KK];
#pragma unroll
    for (int ti = 0; ti < TI; ++ti) xe[ti] = ea[min(16 * ti + i16, ia)];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) ye[kk] = eb[min(4 * kk + k4, ib)];
    double g[TI][KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) {
            const int X = (int)(xe[ti] >> 16 & 0xff), Y = (int)(ye[kk] >> 16 & 0xff);
            const bool x = 16 * ti + i16 < ia, y = 4 * kk + k4 < ib;
            const auto at = x ? (y ? gt + X * n2 + Y : Jb + X) : Ja + Y;
            g[ti][kk] = *at;
        }
    int yo[KK], xo[TI][4];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        const int j = 4 * kk + k4;
        yo[kk] = (j < ib ? (int)(ye[kk] & 0xffff) : b) * nb;
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) {
            const int i = 16 * ti + i16;
            // entry ia (ib) is an unreplaced string: even parity
            const double v = i == ia && j == ib ? both : signed_value(g[ti][kk], xe[ti] ^ ye[kk]);
            g[ti][kk] = i <= ia && j <= ib ? v : 0.0;
        }
    }
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * ti + 4 * v + k4;
            const int rank = (int)(ea[min(i, ia)] & 0xffff);
            xo[ti][v] = (i < ia ? rank : a) * na;
        }
    const auto Ma = to_global(static_cast<const double*>(sd.sw.Ma)), Mb = to_global(static_cast<const double*>(sd.sw.Mb));
    const auto Ka = to_global(static_cast<const double*>(sd.sw.Ka)) + (size_t)a * na;
    const auto Kb = to_global(static_cast<const double*>(sd.sw.Kb)) + (size_t)b * nb;
    const auto Hd = to_global(sd.Hdet), Sd = to_global(sd.Sdet);
    const int fe = topo.flip ? topo.flip[e] : e;
    // the next 16 determinants' elements are read during the products of these where the registers allow
    constexpr bool Ahead = KK <= 10;
    double mv[KK], av[TI][4], ma, mb, ka, kb;
    auto fetch = [&](const StringDet& d, double (&mvx)[KK], double (&avx)[TI][4], double& max, double& mbx, double& kax,
                     double& kbx) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) mvx[kk] = Mb[yo[kk] + d.b];
#pragma unroll
        for (int ti = 0; ti < TI; ++ti)
#pragma unroll
            for (int v = 0; v < 4; ++v) avx[ti][v] = Ma[xo[ti][v] + d.a];
        max = Ma[(size_t)a * na + d.a];
        mbx = Mb[(size_t)b * nb + d.b];
        kax = Ka[d.a];
        kbx = Kb[d.b];
    };
    StringDet d = t.order[begin + i16];
    StringDet next = t.order[min(begin + 16, end - 16) + i16];
    if (Ahead) fetch(d, mv, av, ma, mb, ka, kb);
    for (int base = begin; base < end; base += 16) {
        double mn[KK], an[TI][4], man, mbn, kan, kbn;
        StringDet after{};
        if (Ahead) {
            fetch(next, mn, an, man, mbn, kan, kbn);
            after = t.order[min(base + 32, end - 16) + i16];
        } else {
            fetch(d, mv, av, ma, mb, ka, kb);
        }
        string_double4 acc[TI];
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) acc[ti] = string_double4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int ti = 0; ti < TI; ++ti)
                acc[ti] = __builtin_amdgcn_mfma_f64_16x16x4f64(g[ti][kk], mv[kk], acc[ti], 0, 0, 0);
        double h = 0.0;
#pragma unroll
        for (int ti = 0; ti < TI; ++ti)
#pragma unroll
            for (int v = 0; v < 4; ++v) h += av[ti][v] * acc[ti][v];
        h += __shfl_xor(h, 16, 64);
        h += __shfl_xor(h, 32, 64);
        h += ka * mb + ma * kb;
        // Where e is its own partner, d and its partner (i16 and i16 + 8) have the same four elements, equal but for
        // rounding: the first writes them, else the order of the lanes' stores would choose.
        const bool writes = fe != e || d.flip == d.det || i16 < 8;
        if (d.det >= 0 && writes && order_couple(base + i16, topo.flip != nullptr) <= couple && (k4 < 2 || topo.flip)) {
            const int p = k4 < 2 ? d.det : d.flip, q = k4 < 2 ? e : fe;
            const size_t at = k4 & 1 ? (size_t)q + (size_t)n_det * p : (size_t)p + (size_t)n_det * q;
            Hd[at] = h;
            Sd[at] = ma * mb;
        }
        d = next;
        if (Ahead) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) mv[kk] = mn[kk];
#pragma unroll
            for (int ti = 0; ti < TI; ++ti)
#pragma unroll
                for (int v = 0; v < 4; ++v) av[ti][v] = an[ti][v];
            ma = man;
            mb = mbn;
            ka = kan;
            kb = kbn;
            next = after;
        } else {
            next = t.order[min(base + 32, end - 16) + i16];
        }
    }
}

// f = M_a (C M_b)
template <bool Few>
__global__ void __launch_bounds__(256) k_string_bra(const SlotDesc* __restrict__ slots, TopoDesc topo, int tiles,
                                                    int tiles_j) {
    int x, z, ti, tj;
    problem_block(x, z);
    const SlotDesc& sd = slots[z];
    if (!string_slot(sd)) return;
    const int na = topo.str.a.N, nb = topo.str.b.N, sym = topo.str.sym;
    const int at = Few ? x * 4 + (int)(threadIdx.x >> 6) : x;
    if (at >= tiles) return;
    product_tile(at, tiles_j, sym, ti, tj);
    const auto M = to_global(static_cast<const double*>(sd.sw.Ma)), CM = to_global(static_cast<const double*>(sd.Sdet));
    if (Few) string_product_few(M, na, CM, nb, to_global(sd.Hdet), nb, na, nb, na, ti, tj, sym);
    else string_product(M, na, CM, nb, to_global(sd.Hdet), nb, na, nb, na, ti, tj, sym);
}

// (C M_b)[a][y] = sum over the determinants of alpha string a of w c_d M_b[b_d][y], into Sdet
__global__ void __launch_bounds__(256) k_string_ket(const SlotDesc* __restrict__ slots, TopoDesc topo, int state) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const StringTopo& t = topo.str;
    const int y = blockIdx.x * blockDim.x + threadIdx.x, a = blockIdx.y, nb = t.b.N;
    if (y >= nb) return;
    const auto c = to_global(sd.dcoef) + (size_t)state * topo.n_det;
    const double w = topo.n_states > 1 ? topo.state_w[state] : 1.0;
    double acc = 0.0;
    for (int i = t.aoff[a]; i < t.aoff[a + 1]; ++i) {
        const int d = t.adet[i];
        acc += w * c[d] * to_global(sd.sw.Mb)[(size_t)t.brank[d] * nb + y];
    }
    to_global(sd.Sdet)[(size_t)a * nb + y] = acc;
}

// ---- sigma -------------------------------------------------------------------------------------------

// Row x of sigma = (Ht - lambda) c, one wavefront per row, the row in LDS. The determinants one alpha
// replacement away are taken 64 at a time (one per lane) and walked in order; the lanes run over the
// single replacements of the determinant's beta string and, in lane noff, the string itself, whose
// targets are distinct, so each step is a plain read-add-write of the row. The table and gt reads of
// eight determinants are issued together: their latency bounds the kernel (192 problems of 10 orbitals: 250 us
// one determinant at a time).
__global__ void k_string_sigma(const SlotDesc* __restrict__ slots, TopoDesc topo, int state) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    extern __shared__ double lds[];
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n, na = t.a.N, nb = t.b.N, J = t.b.J, noff = t.b.noff;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x = bx * (blockDim.x >> 6) + wave;
    if (x >= na) return;
    double* row = lds + (size_t)wave * nb;
    const auto c = to_global(sd.dcoef) + (size_t)state * topo.n_det;
    const auto gt = to_global(static_cast<const double*>(sd.sw.gt));
    const auto Ja = to_global(static_cast<const double*>(sd.sw.Ja)) + (size_t)x * n2;
    const auto Jb = to_global(static_cast<const double*>(sd.sw.Jb));
    const auto Ha = to_global(static_cast<const double*>(sd.sw.Ha)) + (size_t)x * na;
    const auto Hb = to_global(static_cast<const double*>(sd.sw.Hb));
    const double lambda = topo.n_states > 1 ? to_global(sd.state_energy)[state] : to_global(sd.energy)[0];
    const uint32_t xmask = t.a.mask[x];
    const int own0 = t.aoff[x], own1 = t.aoff[x + 1];
    for (int y = lane; y < nb; y += 64) {
        double v = 0.0;
        for (int i = t.boff[y]; i < t.boff[y + 1]; ++i) {
            const int e = t.bdet[i];
            v += Ha[t.arank[e]] * c[e];
        }
        for (int i = own0; i < own1; ++i) {
            const int e = t.adet[i], b = t.brank[e];
            v += c[e] * (Hb[(size_t)y * nb + b] - (b == y ? lambda : 0.0));
        }
        row[y] = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int slot = min(lane, noff);
    const bool single = lane < noff;
    constexpr int kAhead = 8;
    // the row's own determinants (no alpha replacement) stand last in its list
    const int last = t.soff[x + 1] - (own1 - own0);
    for (int base = t.soff[x]; base < last; base += 64) {
        const int cnt = min(64, last - base);
        int code = 0, b = 0;
        double ce = 0.0;
        if (lane < cnt) {
            const StringLink s = t.slink[base + lane];
            code = (int)(s.to & 0xffff);
            b = t.brank[s.det];
            ce = signed_value(c[s.det], s.to);
        }
        for (int k0 = 0; k0 < cnt; k0 += kAhead) {
            uint32_t e[kAhead];
            double g[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                e[u] = t.b.e1[(size_t)__builtin_amdgcn_readlane(b, min(k0 + u, cnt - 1)) * J + slot];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int k = min(k0 + u, cnt - 1);
                const int kc = __builtin_amdgcn_readlane(code, k), kb = __builtin_amdgcn_readlane(b, k);
                const auto at = single ? gt + kc * n2 + (e[u] >> 16 & 0xff) : Jb + (size_t)kb * n2 + kc;
                g[u] = *at;
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int k = min(k0 + u, cnt - 1);
                const double kv = k0 + u < cnt ? wave_bcast(ce, k) : 0.0;
                // the entry in lane noff is q == l of the string itself: its rank, even parity
                if (lane <= noff) row[e[u] & 0xffff] += signed_value(kv * g[u], e[u]);
            }
        }
    }
    for (int i = own0; i < own1; ++i) {
        const int d = t.adet[i], b = t.brank[d];
        const uint32_t e = t.b.e1[(size_t)b * J + slot];
        double g = 0.0;
        if (single) g = Ja[e >> 16 & 0xff];
        else
            for (uint32_t m = xmask; m; m &= m - 1) g += Jb[(size_t)b * n2 + __builtin_ctz(m) * (n + 1)];
        if (lane <= noff) row[e & 0xffff] += signed_value(c[d] * g, e);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const auto out = to_global(sd.Sdet) + (size_t)x * nb;
    for (int y = lane; y < nb; y += 64) out[y] = row[y];
}

// ---- densities ---------------------------------------------------------------------------------------

// Opposite-spin density: gpart[chunk][ql][q2l2] = sum over a chunk of 64 determinants whose alpha string
// allows l -> q of c_e f[a_e(l->q)][b_e(l2->q2)]. One wavefront per (ql, chunk): the determinants are
// loaded one per lane and walked in order, the lanes run over the replacements of the beta string
// (distinct targets in the wavefront's n^2 accumulators in LDS). Bound by the latency of the f reads,
// which are issued eight determinants ahead.
__global__ void __launch_bounds__(256) k_string_opposite(const SlotDesc* __restrict__ slots, TopoDesc topo, int state,
                                                         int accumulate) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    __shared__ double lds[4][kMaxN * kMaxN];
    const StringTopo& t = topo.str;
    const int n2 = topo.n * topo.n, nb = t.b.N, J = t.b.J;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int item = bx * 4 + wave;
    if (item >= n2 * t.gchunks) return;
    const int chunk = item / n2, X = item - chunk * n2;
    double* acc = lds[wave];
    for (int i = lane; i < n2; i += 64) acc[i] = 0.0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const auto c = to_global(sd.dcoef) + (size_t)state * topo.n_det;
    const auto f = to_global(static_cast<const double*>(sd.Hdet));
    const int base = t.goff[X] + chunk * 64, cnt = min(64, t.goff[X + 1] - base);
    int xr = 0, b = 0;
    double ce = 0.0;
    if (lane < cnt) {
        const StringLink s = t.glink[base + lane];
        xr = (int)(s.to & 0xffff);
        b = t.brank[s.det];
        ce = signed_value(c[s.det], s.to);
    }
    constexpr int kAhead = 8;
    for (int k0 = 0; k0 < cnt; k0 += kAhead) {
        uint32_t e[kAhead];
        double v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(k0 + u, cnt - 1);
            e[u] = t.b.e1[(size_t)__builtin_amdgcn_readlane(b, k) * J + min(lane, J - 1)];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(k0 + u, cnt - 1);
            v[u] = f[(size_t)__builtin_amdgcn_readlane(xr, k) * nb + (e[u] & 0xffff)];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(k0 + u, cnt - 1);
            const double kv = k0 + u < cnt ? wave_bcast(ce, k) : 0.0;
            if (lane < J) acc[e[u] >> 16 & 0xff] += signed_value(kv * v[u], e[u]);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const auto out = to_global(sd.sw.gpart) + (size_t)item * n2;
    for (int i = lane; i < n2; i += 64) out[i] = accumulate ? out[i] + acc[i] : acc[i];
}

// Same-spin density of one spin: wpart[chunk][(l < l2)][(q < q2)] = sum over a chunk of 64 determinants
// whose beta (alpha) string holds l and l2 of sign c_e f[a_e][b_e(l l2 -> q q2)]. One wavefront per (l l2,
// chunk); its halves take alternate determinants, lanes over the (q, q2), each half with accumulators of
// its own in LDS (summed at the end), so the elements of a step are distinct. The reads of eight steps
// are issued together. (One thread per element over all strings took 205 us for 192 problems of 10 orbitals:
// of 2,025 elements x 252 strings to test a tenth contribute.)
template <bool Alpha>
__global__ void __launch_bounds__(256) k_string_same(const SlotDesc* __restrict__ slots, TopoDesc topo, int state,
                                                     int first_chunk, int accumulate) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    constexpr int kPairs = kMaxN * (kMaxN - 1) / 2;
    __shared__ double lds[4][2][kPairs];
    const StringTopo& t = topo.str;
    const int n = topo.n, nc = n * (n - 1) / 2, nb = t.b.N, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int item = bx * 4 + wave;
    if (item >= nc * t.wchunks) return;
    const int chunk = item / nc, L = item - chunk * nc;
    const int nq = Alpha ? t.nq_a : t.nq_b, per = nq * (Alpha ? t.a.m * (t.a.m - 1) / 2 : t.b.m * (t.b.m - 1) / 2);
    const uint32_t* e2 = Alpha ? t.e2a : t.e2b;
    const int* off = Alpha ? t.w2off_a : t.w2off_b;
    const StringLink* link = Alpha ? t.w2link_a : t.w2link_b;
    const auto c = to_global(sd.dcoef) + (size_t)state * topo.n_det;
    const auto f = to_global(static_cast<const double*>(sd.Hdet));
    for (int i = lane; i < nc; i += 64) lds[wave][0][i] = lds[wave][1][i] = 0.0;
    wave_sync();
    const int base = off[L] + chunk * 64, cnt = min(64, off[L + 1] - base);
    // lane k: determinant k of the chunk: offset of its list, the fixed index of f, its coefficient
    int at = 0, fixed = 0;
    double ce = 0.0;
    if (lane < cnt) {
        const StringLink s = link[base + lane];
        const int a = t.arank[s.det], b = t.brank[s.det];
        at = (Alpha ? a : b) * per + (int)s.to * nq;
        fixed = Alpha ? b : a;
        ce = c[s.det];
    }
    const int half = lane >> 5, q = lane & 31;
    double* acc = lds[wave][half];
    constexpr int kAhead = 8;
    for (int k0 = 0; k0 < cnt; k0 += 2 * kAhead) {
        int atk[kAhead], fk[kAhead];
        double ck[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = k0 + 2 * u + half;
            atk[u] = __shfl(at, k & 63, 64);
            fk[u] = __shfl(fixed, k & 63, 64);
            const double cu = __shfl(ce, k & 63, 64);  // by every lane: the halves may disagree on k < cnt
            ck[u] = k < cnt ? cu : 0.0;
        }
        for (int q0 = 0; q0 < nq; q0 += 32) {
            const bool live = q0 + q < nq;
            uint32_t code[kAhead];
            double v[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) code[u] = e2[atk[u] + min(q0 + q, nq - 1)];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int r = (int)(code[u] & 0xfff);
                v[u] = Alpha ? f[(size_t)r * nb + fk[u]] : f[(size_t)fk[u] * nb + r];
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                if (live) acc[code[u] >> 12 & 0x7f] += signed_value(ck[u] * v[u], code[u]);
        }
    }
    wave_sync();
    const auto out = to_global(sd.sw.wpart) + ((size_t)(first_chunk + chunk) * nc + L) * nc;
    for (int i = lane; i < nc; i += 64) {
        const double s = lds[wave][0][i] + lds[wave][1][i];
        out[i] = accumulate ? out[i] + s : s;
    }
}

// ---- response ------------------------------------------------------------------------------------------

// zpart[block][ql] = sum over the block's rows x of f and sigma of
//   sum_w f_q[w] sigma_l[w],  f_q[w] = +-f[x][w with q added] over the strings w of one electron fewer:
// a product of n x n with the long summation (x, w) on the matrix cores (n <= 16: one tile). A lane's
// f and sigma operands have the same index, so one table entry and one 16-byte LDS read serve both; R rows
// share the table read. Bound by those LDS reads (gathers). One thread per (q, l) over lists of
// strings took 288 us for 192 problems of 10 orbitals and 1.77 ms for one of 14.
template <int R, typename P>
__device__ __forceinline__ void response_products(const f64x2* rows, P wtab, int nb, int nw, string_double4& acc) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
#pragma unroll 4
    for (int w0 = 4 * wave; w0 < nw; w0 += 16) {
        const int w = w0 + k4;
        const uint32_t code = wtab[(size_t)min(w, nw - 1) * 16 + i16];
        const int at = w < nw ? (int)(code & 0xfff) : nb;
        const uint32_t odd = code << 16;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const f64x2 v = rows[r * (nb + 1) + at];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(signed_value(v[0], odd), signed_value(v[1], odd), acc, 0, 0, 0);
        }
    }
}

// Element (q, l) = (threadIdx.x / 16, threadIdx.x % 16) of the four wavefronts' sums; lds: 4 x 256
__device__ __forceinline__ double response_sum(double* lds, const string_double4& acc) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) lds[wave * 256 + (4 * v + k4) * 16 + i16] = acc[v];
    __syncthreads();
    return (lds[threadIdx.x] + lds[256 + threadIdx.x]) + (lds[512 + threadIdx.x] + lds[768 + threadIdx.x]);
}

template <int R>
__global__ void __launch_bounds__(256) k_string_response(const SlotDesc* __restrict__ slots, TopoDesc topo,
                                                         int accumulate) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    extern __shared__ double lds[];
    const StringTopo& t = topo.str;
    const int n = topo.n, na = t.a.N, nb = t.b.N;
    f64x2* rows = reinterpret_cast<f64x2*>(lds);  // [R][nb + 1]: (f, sigma), zeros at nb
    const auto f = to_global(static_cast<const double*>(sd.Hdet));
    const auto sg = to_global(static_cast<const double*>(sd.Sdet));
    string_double4 acc = string_double4{0.0, 0.0, 0.0, 0.0};
    const int last = min(na, (bx + 1) * kStringRowsZ);
    for (int x = bx * kStringRowsZ; x < last; x += R) {
        __syncthreads();
        for (int r = 0; r < R; ++r)
            for (int i = threadIdx.x; i <= nb; i += 256) {
                const bool live = i < nb && x + r < last;
                const size_t at = (size_t)min(x + r, last - 1) * nb + min(i, nb - 1);
                rows[r * (nb + 1) + i] = live ? f64x2{f[at], sg[at]} : f64x2{0.0, 0.0};
            }
        __syncthreads();
        response_products<R>(rows, t.wtab, nb, t.nw, acc);
    }
    const double s = response_sum(lds, acc);
    const int q = threadIdx.x >> 4, l = threadIdx.x & 15;
    if (q < n && l < n) {
        const auto out = to_global(sd.sw.zpart) + (size_t)bx * n * n + q * n + l;
        *out = accumulate ? *out + s : s;
    }
}

// The alpha part for determinant coefficients without spin-exchange symmetry:
// zalpha[x J + j] = sign f[x_j] . sigma[x], one workgroup per alpha string, a wavefront per replacement.
__global__ void __launch_bounds__(256) k_string_response_alpha(const SlotDesc* __restrict__ slots, TopoDesc topo,
                                                               int offset, int accumulate) {
    int x, bz;
    problem_block(x, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    extern __shared__ double lds[];
    const StringTopo& t = topo.str;
    const int nb = t.b.N, J = t.a.J;
    const auto f = to_global(static_cast<const double*>(sd.Hdet));
    const auto sg = to_global(static_cast<const double*>(sd.Sdet)) + (size_t)x * nb;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) lds[i] = sg[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const auto out = to_global(sd.sw.zpart) + offset + (size_t)x * J;
    for (int j = wave; j < J; j += 4) {
        const uint32_t e = t.a.e1[(size_t)x * J + j];
        const auto fr = f + (size_t)(e & 0xffff) * nb;
        double acc = 0.0;
#pragma unroll 4
        for (int y = lane; y < nb; y += 64) acc += fr[y] * lds[y];
        acc = signed_value(wave_sum(acc), e);
        if (lane == 0) out[j] = accumulate ? out[j] + acc : acc;
    }
}

// ---- listed pairs ------------------------------------------------------------------------------------------

// The densities above sum over all pairs; those of the listed ones, which the list kernels differentiate, are
// taken out again as one more chunk. One wavefront per (q, l) (opposite spin), then per (l < l2) of each
// spin (beta alone under spin-exchange symmetry), over the listed pairs in order, each pair both ways
// (d ket, e bra); lanes over the ket's replacements. Bound by the chain of dependent reads of a pair, about 1 us.
__global__ void __launch_bounds__(256) k_string_list_density(const SlotDesc* __restrict__ slots, TopoDesc topo) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    __shared__ double lds[4][kMaxN * kMaxN];
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n, nc = n * (n - 1) / 2, na = t.a.N, nb = t.b.N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int item = blockIdx.x * 4 + wave, listed = to_global(sd.flags)[FLAG_DEFERRED];
    if (listed == 0 || item >= n2 + (t.sym ? 1 : 2) * nc) return;
    const bool opposite = item < n2, alpha = item >= n2 + nc;
    const int L = item - n2 - (alpha ? nc : 0);
    int x = item / n, y = item - x * n;  // opposite spin: y -> x of the alpha string; same spin: the two replaced
    if (!opposite) {
        unpack_pair(L, x, y);
        ++y;
    }
    double* acc = lds[wave];
    const int len = opposite ? n2 : nc;
    for (int i = lane; i < len; i += 64) acc[i] = 0.0;
    wave_sync();
    const auto Ma = to_global(static_cast<const double*>(sd.sw.Ma)), Mb = to_global(static_cast<const double*>(sd.sw.Mb));
    const StringSpace& own = opposite || alpha ? t.a : t.b;  // the string that the wavefront's item selects
    for (int i = 0; i < listed; ++i) {
        int d, e;
        unpack_pair(to_global(sd.defer)[i], d, e);
        double w, unused;
        pair_weights(sd, topo, d, e, d, e, false, 1.0, w, unused);
        for (int way = 0; way < (d == e ? 1 : 2); ++way) {
            const int bra = way ? e : d, ket = way ? d : e;
            const int a = t.arank[ket], b = t.brank[ket], A = t.arank[bra], B = t.brank[bra];
            const uint32_t mask = own.mask[opposite || alpha ? a : b];
            if (opposite) {
                if (!(mask >> y & 1) || (x != y && (mask >> x & 1))) continue;
                const uint32_t left = mask ^ (1u << y);
                const double m = Ma[(size_t)A * na + t.rank[left | 1u << x]];
                const double u = -w * ((below(mask, y) + below(left, x)) & 1 ? -m : m);
                if (lane < t.b.J) {
                    const uint32_t code = t.b.e1[(size_t)b * t.b.J + lane];
                    acc[code >> 16 & 0xff] += signed_value(u * Mb[(size_t)B * nb + (code & 0xffff)], code);
                }
            } else {
                if (!(mask >> x & 1) || !(mask >> y & 1)) continue;
                const int k1 = below(mask, x), k2 = below(mask, y), pairs = own.m * (own.m - 1) / 2;
                const int nq = alpha ? t.nq_a : t.nq_b;
                const uint32_t* list = (alpha ? t.e2a : t.e2b) + ((size_t)(alpha ? a : b) * pairs + k2 * (k2 - 1) / 2 + k1) * nq;
                const auto M = alpha ? Ma + (size_t)A * na : Mb + (size_t)B * nb;
                const double u = -w * (alpha ? Mb[(size_t)B * nb + b] : Ma[(size_t)A * na + a]);
                for (int q = lane; q < nq; q += 64) acc[list[q] >> 12 & 0x7f] += signed_value(u * M[list[q] & 0xfff], list[q]);
            }
        }
    }
    wave_sync();
    const auto out = opposite ? to_global(sd.sw.gpart) + ((size_t)t.gchunks * n2 + item) * n2
                              : to_global(sd.sw.wpart) + ((size_t)((t.sym ? 1 : 2) * t.wchunks + (alpha ? 1 : 0)) * nc + L) * nc;
    for (int i = lane; i < len; i += 64) out[i] = acc[i];
}

// The listed pairs' response, rows zblocks.. of zpart: workgroup k takes k, k + kStringListRows, ... of them, both ways counted.
// Both rows of a pair are products of one vector per spin: f = M_a[d_a] M_b[d_b], and sigma = (Ht - E) e is
// contracted with the other spin's row of M, so that the beta part is the response of the strings
//   (M_b[d_b][y], t[y]),  t[y] = sum_x M_a[d_a][x] sigma[x][y]
// as one more row of k_string_response, and the alpha part (without spin-exchange symmetry) its mirror image.
__global__ void __launch_bounds__(256) k_string_list_response(const SlotDesc* __restrict__ slots, TopoDesc topo,
                                                              int zblocks) {
    const SlotDesc& sd = slots[blockIdx.z];
    const int listed = to_global(sd.flags)[FLAG_DEFERRED];
    if (!string_slot(sd) || (int)blockIdx.x >= 2 * listed) return;  // k_string_gather skips the row
    extern __shared__ __align__(16) double lds[];
    __shared__ double ua[64], ub[64], part[2][4];
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n, na = t.a.N, nb = t.b.N, Ja = t.a.J, Jb = t.b.J, tid = threadIdx.x;
    f64x2* rows = reinterpret_cast<f64x2*>(lds);  // (M_b[d_b][y], t[y]), zeros at nb
    double* ta = lds + 2 * (nb + 1);
    const auto Ma = to_global(static_cast<const double*>(sd.sw.Ma)), Mb = to_global(static_cast<const double*>(sd.sw.Mb));
    const auto Ha = to_global(static_cast<const double*>(sd.sw.Ha)), Hb = to_global(static_cast<const double*>(sd.sw.Hb));
    const auto gt = to_global(static_cast<const double*>(sd.sw.gt));
    string_double4 acc = string_double4{0.0, 0.0, 0.0, 0.0};
    double alpha = 0.0;  // element tid of the alpha part
    for (int i = blockIdx.x; i < 2 * listed; i += gridDim.x) {
        int d, e;
        unpack_pair(to_global(sd.defer)[i >> 1], d, e);
        if (d == e && (i & 1)) continue;
        double wH, wS;
        pair_weights(sd, topo, d, e, d, e, false, 1.0, wH, wS);
        const int bra = i & 1 ? e : d, ket = i & 1 ? d : e;
        const int a = t.arank[ket], b = t.brank[ket], A = t.arank[bra], B = t.brank[bra];
        const uint32_t* ea = t.a.e1 + (size_t)a * Ja;
        const uint32_t* eb = t.b.e1 + (size_t)b * Jb;
        const double ma = Ma[(size_t)A * na + a], mb = Mb[(size_t)B * nb + b];
        __syncthreads();  // the previous pair's rows have been read
        if (tid < Ja) ua[tid] = signed_value(Ma[(size_t)A * na + (ea[tid] & 0xffff)], ea[tid]);
        if (tid >= 64 && tid < 64 + Jb) ub[tid - 64] = signed_value(Mb[(size_t)B * nb + (eb[tid - 64] & 0xffff)], eb[tid - 64]);
        // K = M Ht of the pair, either spin
        double ka = 0.0, kb = 0.0;
        for (int x = tid; x < na; x += 256) ka += Ma[(size_t)A * na + x] * Ha[(size_t)x * na + a];
        for (int y = tid; y <= nb; y += 256) {
            const double m = y < nb ? Mb[(size_t)B * nb + y] : 0.0, h = y < nb ? Hb[(size_t)y * nb + b] : 0.0;
            kb += m * h;
            rows[y] = f64x2{m, wH * ma * h};
        }
        if (!t.sym)
            for (int x = tid; x < na; x += 256) ta[x] = wH * mb * Ha[(size_t)x * na + a];
        ka = wave_sum(ka);
        kb = wave_sum(kb);
        if ((tid & 63) == 0) {
            part[0][tid >> 6] = ka;
            part[1][tid >> 6] = kb;
        }
        __syncthreads();
        // opposite spin: wavefront 0 adds the beta targets, 1 the alpha ones (distinct but for the string itself)
        const bool beta = tid < 64;
        if (beta || (tid < 128 && !t.sym)) {
            const int j = tid & 63, J = beta ? Jb : Ja, J2 = beta ? Ja : Jb, noff = beta ? t.b.noff : t.a.noff;
            double v = 0.0;
            const uint32_t code = beta ? eb[min(j, J - 1)] : ea[min(j, J - 1)];
            const int own = (int)(code >> 16 & 0xff);
#pragma unroll 4
            for (int k = 0; k < J2; ++k) {
                const int other = (int)((beta ? ea[k] : eb[k]) >> 16 & 0xff);
                v += (beta ? ua[k] : ub[k]) * gt[beta ? other * n2 + own : own * n2 + other];
            }
            v = signed_value(wH * v, code);
            const double itself = wave_sum(j >= noff && j < J ? v : 0.0);
            if (j < noff) {
                if (beta) rows[code & 0xffff][1] += v;
                else ta[code & 0xffff] += v;
            }
            if (j == 0) {
                const double* p = part[beta ? 0 : 1];
                const double k = (p[0] + p[1]) + (p[2] + p[3]);
                const double s = itself + wH * k + wS * (beta ? ma : mb);
                if (beta) rows[b][1] += s;
                else ta[a] += s;
            }
        }
        __syncthreads();
        response_products<1>(rows, t.wtab, nb, t.nw, acc);
        if (!t.sym && tid < n2) {
#pragma unroll 8
            for (int k = 0; k < t.ak; ++k) {
                const uint32_t entry = t.alist[(size_t)k * n2 + tid], at = entry == ~0u ? 0u : entry;
                const uint32_t code = t.a.e1[at];
                const double v = signed_value(Ma[(size_t)A * na + (code & 0xffff)] * ta[at / Ja], code);
                alpha += entry == ~0u ? 0.0 : v;
            }
        }
    }
    const double s = response_sum(lds, acc);
    __syncthreads();
    lds[tid] = alpha;
    __syncthreads();
    const int q = tid >> 4, l = tid & 15;
    if (q < n && l < n) to_global(sd.sw.zpart)[(size_t)(zblocks + blockIdx.x) * n2 + q * n + l] = -(s + lds[q * n + l]);
}

// ---- adjoints ------------------------------------------------------------------------------------------

// gs = dgt + dgt^T from the chunks of the densities, the listed pairs' last: a workgroup takes the 16 x 16 tiles (X, Y) and (Y, X), both
// read along their rows and exchanged through LDS. The last workgroup forms dht and Z.
constexpr int kGatherTile = 16;
__global__ void __launch_bounds__(256) k_string_gather(const SlotDesc* __restrict__ slots, TopoDesc topo, int tiles,
                                                       int zblocks) {
    int bx, bz;
    problem_block(bx, bz);
    const SlotDesc& sd = slots[bz];
    if (!string_slot(sd)) return;
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n, nc = n * (n - 1) / 2;
    const size_t n4 = (size_t)n2 * n2;
    const auto gp = to_global(static_cast<const double*>(sd.sw.gpart));
    const int listed = to_global(sd.flags)[FLAG_DEFERRED];  // 0: no listed pairs' chunk
    const int gchunks = t.gchunks + (listed > 0), wchunks = (t.sym ? 1 : 2) * (t.wchunks + (listed > 0));
    if (bx < tiles) {
        __shared__ double up[kGatherTile][kGatherTile + 1], lo[kGatherTile][kGatherTile + 1];
        int tx, ty;
        unpack_pair(bx, tx, ty);  // tx <= ty
        const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
        const int X = tx * kGatherTile + i, Y = ty * kGatherTile + j;   // element of the upper tile
        const int X2 = ty * kGatherTile + i, Y2 = tx * kGatherTile + j;  // of the lower one
        double v = 0.0, v2 = 0.0;
        const size_t at = (size_t)min(X, n2 - 1) * n2 + min(Y, n2 - 1), at2 = (size_t)min(X2, n2 - 1) * n2 + min(Y2, n2 - 1);
#pragma unroll 4
        for (int k = 0; k < gchunks; ++k) {
            v += gp[k * n4 + at];
            v2 += gp[k * n4 + at2];
        }
        up[i][j] = v;
        lo[i][j] = v2;
        __syncthreads();
        v += lo[j][i];
        v2 += up[j][i];
        auto same_spin = [&](int x, int y) {
            const int q = x / n, l = x - q * n, q2 = y / n, l2 = y - q2 * n;
            if (q == q2 || l == l2) return 0.0;
            const int qa = min(q, q2), qb = max(q, q2), la = min(l, l2), lb = max(l, l2);
            const auto w = to_global(static_cast<const double*>(sd.sw.wpart)) + (size_t)(lb * (lb - 1) / 2 + la) * nc +
                           qb * (qb - 1) / 2 + qa;
            double s = 0.0;
            for (int k = 0; k < wchunks; ++k) s += w[(size_t)k * nc * nc];
            if (t.sym) s *= 2.0;
            return (q < q2) == (l < l2) ? s : -s;
        };
        const auto out = to_global(sd.sw.gs);
        if (X < n2 && Y < n2) out[at] = v + same_spin(X, Y);
        if (tx != ty && X2 < n2 && Y2 < n2) out[at2] = v2 + same_spin(X2, Y2);
        return;
    }
    // dht over both spins: a diagonal of the density counts every electron of the other spin
    for (int X = threadIdx.x; X < n2; X += 256) {
        double va = 0.0, vb = 0.0;
        for (int k = 0; k < gchunks; ++k)
            for (int l = 0; l < n; ++l) {
                va += gp[k * n4 + (size_t)X * n2 + l * (n + 1)];
                vb += gp[k * n4 + (size_t)l * (n + 1) * n2 + X];
            }
        to_global(sd.sw.hb)[X] = va / t.b.m + vb / t.a.m;
        const auto z = to_global(static_cast<const double*>(sd.sw.zpart));
        const int zrows = zblocks + min(kStringListRows, 2 * listed);
        double v = 0.0;
#pragma unroll 8
        for (int k = 0; k < zrows; ++k) v += z[(size_t)k * n2 + X];
        if (t.sym) v *= 2.0;
        else
            for (int k = 0; k < t.ak; ++k) {
                const uint32_t at = t.alist[(size_t)k * n2 + X];
                if (at != ~0u) v += z[(size_t)(zblocks + kStringListRows) * n2 + at];
            }
        to_global(sd.sw.Zt)[X] = v;
    }
}

// V[rl][Y] = sum_q S^-1_qr gs[ql][Y]; the last blocks: W_qp = sum_lY gs[ql][Y] gt[pl][Y] + dht_ql ht_pl,
// one workgroup per (q, p)
__global__ void __launch_bounds__(256) k_string_pullback(const SlotDesc* __restrict__ slots, int n, int vblocks) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const int n2 = n * n, n4 = n2 * n2, n3 = n2 * n;
    const auto gs = to_global(static_cast<const double*>(sd.sw.gs));
    if ((int)blockIdx.x < vblocks) {
        const int id = blockIdx.x * blockDim.x + threadIdx.x;
        if (id >= n4) return;
        const int X = id / n2, Y = id - X * n2, r = X / n, l = X - r * n;
        double v = 0.0;
        for (int q = 0; q < n; ++q) v += to_global(sd.sw.Sinv)[q * n + r] * gs[(q * n + l) * n2 + Y];
        to_global(sd.sw.V)[id] = v;
        return;
    }
    const int at = blockIdx.x - vblocks, q = at / n, p = at - q * n;
    const auto gt = to_global(static_cast<const double*>(sd.sw.gt));
    double acc = 0.0;
#pragma unroll 4
    for (int k = threadIdx.x; k < n3; k += 256) acc += gs[q * n3 + k] * gt[p * n3 + k];
    if ((int)threadIdx.x < n)
        acc += to_global(sd.sw.hb)[q * n + threadIdx.x] * to_global(sd.sw.ht)[p * n + threadIdx.x];
    __shared__ double part[4];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) to_global(sd.sw.W2)[at] = (part[0] + part[1]) + (part[2] + part[3]);
}

// dsum: the packed-kernel adjoint, then the S_act and h_act adjoints
__global__ void __launch_bounds__(256) k_string_adjoint(const SlotDesc* __restrict__ slots, int n, int ng) {
    const SlotDesc& sd = slots[blockIdx.z];
    if (!string_slot(sd)) return;
    const int n2 = n * n;
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    const auto Sinv = to_global(static_cast<const double*>(sd.sw.Sinv));
    const auto out = to_global(sd.dsum);
    if (id < ng) {
        int P, Q, r[2], s[2];
        unpack_pair(id, Q, P);  // Q <= P
        unpack_pair(P, r[0], r[1]);
        unpack_pair(Q, s[0], s[1]);
        const auto V = to_global(static_cast<const double*>(sd.sw.V));
        double v = 0.0;
        for (int i = 0; i < (r[0] == r[1] ? 1 : 2); ++i)
            for (int j = 0; j < (s[0] == s[1] ? 1 : 2); ++j)
                for (int q = 0; q < n; ++q)
                    v += Sinv[q * n + s[j]] * V[(r[i] * n + r[1 - i]) * n2 + q * n + s[1 - j]];
        out[id] = P == Q ? 0.5 * v : v;
    } else if (id < ng + n2) {
        const int r = (id - ng) % n, p = (id - ng) / n;
        double v = 0.0;
        for (int q = 0; q < n; ++q) v += Sinv[q * n + r] * (to_global(sd.sw.Zt)[q * n + p] - to_global(sd.sw.W2)[q * n + p]);
        out[id] = v;
    } else if (id < ng + 2 * n2) {
        const int r = (id - ng - n2) % n, l = (id - ng - n2) / n;
        double v = 0.0;
        for (int q = 0; q < n; ++q) v += Sinv[q * n + r] * to_global(sd.sw.hb)[q * n + l];
        out[id] = v;
    }
}

unsigned blocks_for(long long work, int threads = 256) { return (unsigned)((work + threads - 1) / threads); }

int z_blocks(const StringTopo& t) { return (t.a.N + kStringRowsZ - 1) / kStringRowsZ; }

template <int M>
void minors(hipStream_t st, const SlotDesc* slots, unsigned z, int n, const StringSpace& sp, bool beta) {
    if constexpr (M > 7) return;  // the lane kernels' shapes
    else if (sp.m == M) {
        hipLaunchKernelGGL(k_string_minors<M>, dim3(blocks_for(sp.N), (unsigned)((sp.N + kMinorRows - 1) / kMinorRows), z),
                           dim3(256), 0, st, slots, n, sp, beta);
        hipLaunchKernelGGL(k_string_condition<M>, dim3(blocks_for((long long)sp.N * (sp.N + 1) / 2, 256 * kConditionSteps), 1, z), dim3(256), 0, st,
                           slots, n, sp, beta);
    } else minors<M + 1>(st, slots, z, n, sp, beta);
}

}  // namespace

size_t string_work_carve(const TopoDesc& topo, double* base, StringWork& w) {
    const StringTopo& t = topo.str;
    const size_t n = topo.n, n2 = n * n, n4 = n2 * n2, nc = n * (n - 1) / 2, na = t.a.N, nb = t.b.N;
    const bool same = t.a.m == t.b.m;
    size_t at = 0;
    auto take = [&](double*& p, size_t count) {
        p = base + at;
        at += (count + 31) / 32 * 32;
    };
    take(w.Sinv, n2);
    take(w.ht, n2);
    take(w.U, n2 * topo.np);
    take(w.gt, n4);
    take(w.Ma, na * na);
    if (same) w.Mb = w.Ma;
    else take(w.Mb, nb * nb);
    take(w.Ja, na * n2);
    if (same) w.Jb = w.Ja;
    else take(w.Jb, nb * n2);
    take(w.Fa, na * n2);
    if (same) w.Fb = w.Fa;
    else take(w.Fb, nb * n2);
    take(w.Ha, na * na);
    if (same) w.Hb = w.Ha;
    else take(w.Hb, nb * nb);
    const size_t bytes_a = (na * na + 7) / 8, bytes_b = same ? 0 : (nb * nb + 7) / 8;
    double* near = nullptr;
    take(near, bytes_a + bytes_b);
    w.neara = reinterpret_cast<unsigned char*>(near);
    w.nearb = same ? w.neara : reinterpret_cast<unsigned char*>(near + bytes_a);
    const size_t shared = at;  // K is dead when the densities are formed
    take(w.Ka, na * na);
    if (same) w.Kb = w.Ka;
    else take(w.Kb, nb * nb);
    const size_t after_k = at;
    at = shared;
    take(w.gpart, (size_t)(t.gchunks + 1) * n4);
    take(w.wpart, (size_t)(t.wchunks + 1) * (t.sym ? 1 : 2) * nc * nc);
    take(w.zpart, (size_t)(z_blocks(t) + kStringListRows) * n2 + na * t.a.J);
    take(w.gs, n4);
    take(w.hb, n2);
    take(w.V, n4);
    take(w.W2, n2);
    take(w.Zt, n2);
    return std::max(at, after_k);
}

void launch_string_frame(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    hipLaunchKernelGGL(k_string_frame, dim3(1, 1, z), dim3(64), 0, st, slots, topo.n);
}

void launch_string_minors(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    const StringTopo& t = topo.str;
    minors<1>(st, slots, z, topo.n, t.a, false);
    if (t.a.m != t.b.m) minors<1>(st, slots, z, topo.n, t.b, true);
    hipLaunchKernelGGL(k_string_list, dim3((unsigned)std::min<long long>(256, (topo.n_lane_pairs + 255) / 256), 1, z),
                       dim3(256), 0, st, slots, topo);
}

void launch_string_integrals(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n;
    hipLaunchKernelGGL(k_string_half, dim3(blocks_for((long long)n2 * topo.np), 1, z), dim3(256), 0, st, slots, n, topo.np);
    hipLaunchKernelGGL(k_string_full, dim3(blocks_for((long long)n2 * n2), 1, z), dim3(256), 0, st, slots, n, topo.np);
    for (int beta = 0; beta < (t.a.m == t.b.m ? 1 : 2); ++beta) {
        const StringSpace& sp = beta ? t.b : t.a;
        hipLaunchKernelGGL(k_string_coulomb, dim3(blocks_for((long long)sp.N * n2), 1, z), dim3(256), 0, st, slots, n, sp,
                           beta != 0);
        hipLaunchKernelGGL(k_string_hamiltonian, dim3(blocks_for(sp.N), (unsigned)sp.N, z), dim3(256), 0, st, slots, n, sp,
                           beta != 0);
    }
}

namespace {

template <int KK>
void string_pairs(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo, int need) {
    if constexpr (KK > 13) return;  // 49 replacements of 7 electrons in 14 orbitals
    else if (need <= KK)
        hipLaunchKernelGGL(k_string_pairs<KK>, dim3((unsigned)((topo.str.npitem + 3) / 4), 1, z), dim3(256), 0, st, slots, topo);
    else string_pairs<KK + 1>(st, slots, z, topo, need);
}

}  // namespace

void launch_string_forward(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    const StringTopo& t = topo.str;
    for (int beta = 0; beta < (t.a.m == t.b.m ? 1 : 2); ++beta) {
        const StringSpace& sp = beta ? t.b : t.a;
        const auto tri = [](int k) { return k * (k + 1) / 2; };
        const int big = (sp.N + kProductTile - 1) / kProductTile, small = (sp.N + 15) / 16;
        if ((long long)tri(big) * z >= kProductTilesFew)
            hipLaunchKernelGGL(k_string_same_spin<false>, dim3((unsigned)tri(big), 1, z), dim3(256), 0, st, slots, sp.N, big,
                               beta != 0);
        else
            hipLaunchKernelGGL(k_string_same_spin<true>, dim3((unsigned)(tri(small) + 3) / 4, 1, z), dim3(256), 0, st, slots,
                               sp.N, small, beta != 0);
    }
    string_pairs<2>(st, slots, z, topo, (std::max(t.a.noff, t.b.noff) + 4) / 4);
}

void launch_string_backward(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    const StringTopo& t = topo.str;
    const int n = topo.n, n2 = n * n, nc = n * (n - 1) / 2, na = t.a.N, nb = t.b.N;
    const int wc = t.wchunks, zb = z_blocks(t);
    const dim3 w_grid((unsigned)((nc * wc + 3) / 4), 1, z);
    const int ti = (na + kProductTile - 1) / kProductTile, tj = (nb + kProductTile - 1) / kProductTile;
    const int row_waves = nb > 1000 ? 2 : 4;  // two wavefronts' rows of 3432 strings leave two workgroups per CU
    for (int s = 0; s < topo.n_states; ++s) {
        const int add = s > 0;
        hipLaunchKernelGGL(k_string_ket, dim3(blocks_for(nb), (unsigned)na, z), dim3(256), 0, st, slots, topo, s);
        const int big = t.sym ? ti * (ti + 1) / 2 : ti * tj;
        if ((long long)big * z >= kProductTilesFew) {
            hipLaunchKernelGGL(k_string_bra<false>, dim3((unsigned)big, 1, z), dim3(256), 0, st, slots, topo, big, tj);
        } else {
            const int si = (na + 15) / 16, sj = (nb + 15) / 16, few = t.sym ? si * (si + 1) / 2 : si * sj;
            hipLaunchKernelGGL(k_string_bra<true>, dim3((unsigned)(few + 3) / 4, 1, z), dim3(256), 0, st, slots, topo, few, sj);
        }
        hipLaunchKernelGGL(k_string_sigma, dim3((unsigned)((na + row_waves - 1) / row_waves), 1, z), dim3(64 * row_waves),
                           sizeof(double) * row_waves * nb, st, slots, topo, s);
        hipLaunchKernelGGL(k_string_opposite, dim3((unsigned)((n2 * t.gchunks + 3) / 4), 1, z), dim3(256), 0, st, slots,
                           topo, s, add);
        if (wc > 0) hipLaunchKernelGGL(k_string_same<false>, w_grid, dim3(256), 0, st, slots, topo, s, 0, add);
        // rows staged together: as many as leave several workgroups per CU
        const size_t row_lds = 2 * sizeof(double) * (nb + 1), least = 4 * 256 * sizeof(double);
        if (nb <= 512)
            hipLaunchKernelGGL(k_string_response<4>, dim3((unsigned)zb, 1, z), dim3(256), std::max(4 * row_lds, least), st,
                               slots, topo, add);
        else if (nb <= 1024)
            hipLaunchKernelGGL(k_string_response<2>, dim3((unsigned)zb, 1, z), dim3(256), std::max(2 * row_lds, least), st,
                               slots, topo, add);
        else
            hipLaunchKernelGGL(k_string_response<1>, dim3((unsigned)zb, 1, z), dim3(256), std::max(row_lds, least), st,
                               slots, topo, add);
        if (!t.sym) {
            if (wc > 0) hipLaunchKernelGGL(k_string_same<true>, w_grid, dim3(256), 0, st, slots, topo, s, wc, add);
            hipLaunchKernelGGL(k_string_response_alpha, dim3((unsigned)na, 1, z), dim3(256), sizeof(double) * nb, st, slots,
                               topo, (zb + kStringListRows) * n2, add);
        }
    }
    hipLaunchKernelGGL(k_string_list_density, dim3((unsigned)((n2 + (t.sym ? 1 : 2) * nc + 3) / 4), 1, z), dim3(256), 0, st,
                       slots, topo);
    hipLaunchKernelGGL(k_string_list_response, dim3(kStringListRows, 1, z), dim3(256),
                       sizeof(double) * std::max<size_t>(2 * (nb + 1) + (t.sym ? 0 : na), 4 * 256), st, slots, topo, zb);
    const long long n4 = (long long)n2 * n2;
    const int gt = (n2 + kGatherTile - 1) / kGatherTile, gtiles = gt * (gt + 1) / 2;
    hipLaunchKernelGGL(k_string_gather, dim3((unsigned)gtiles + 1, 1, z), dim3(256), 0, st, slots, topo, gtiles, zb);
    const unsigned vb = blocks_for(n4);
    hipLaunchKernelGGL(k_string_pullback, dim3(vb + n2, 1, z), dim3(256), 0, st, slots, n, (int)vb);
    hipLaunchKernelGGL(k_string_adjoint, dim3(blocks_for(topo.ng + 2 * n2), 1, z), dim3(256), 0, st, slots, n, topo.ng);
}

hipError_t configure_strings() {
    for (const void* k : {reinterpret_cast<const void*>(&k_string_sigma),
                          reinterpret_cast<const void*>(&k_string_response<1>),
                          reinterpret_cast<const void*>(&k_string_response<2>),
                          reinterpret_cast<const void*>(&k_string_response<4>),
                          reinterpret_cast<const void*>(&k_string_list_response)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace xmvb_amd
