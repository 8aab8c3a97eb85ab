// Dense eigensolve of structure spaces beyond one wavefront (n_str > 64), one selected state that is the
// lowest root: Cholesky of the metric in LDS, the explicit L^-1, and the lowest eigenpair of
// A = L^-1 H L^-T by Lanczos with full reorthogonalisation
// (GeneralizedEigensolver::solve_dense semantics, linalg/eigensolver.cpp:365-387).
//
// Lanczos with every new vector orthogonalised against all earlier ones is the tridiagonalisation of
// the dense solve built one column at a time: after n steps it is a full orthogonal reduction. Its
// lowest eigenpair converges long before that, and the reduction stops when the residual of the
// Ritz vector, beta_k |s_k|, is below rounding (kRitzTolerance of the largest row sum of T), which is
// the backward error of the full reduction. Householder steps cost n launches or n block-wide
// steps over the whole trailing matrix whatever the root wanted.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace xmvb_amd {

namespace {

// ---- Cholesky in LDS ------------------------------------------------------------------------------------

constexpr int kCholTile = 16;
constexpr int kCholThreads = 512;  // 256 registers each: at 1024 threads the unrolled tile steps spill

typedef double chol_double4 __attribute__((ext_vector_type(4)));

// Diagonal tile of T columns, jb of them in the matrix, on one wavefront: row `lane` in r becomes the row of L (what
// stands above the diagonal or past the matrix is never read), the reciprocal diagonal goes to rl. false: a
// pivot is not positive.
template <int T>
__device__ __forceinline__ bool chol_tile(double (&r)[T], int jb, double* rl, int lane) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < T; ++k) {
        const double piv = k < jb ? wave_bcast(r[k], k) : 1.0;
        ok = ok && piv > 0.0;
        const double inv = 1.0 / sqrt(piv);
        r[k] *= inv;
        if (lane == 0) rl[k] = inv;
#pragma unroll
        for (int j = k + 1; j < T; ++j) r[j] -= r[k] * wave_bcast(r[k], j);
        __builtin_amdgcn_sched_barrier(0);  // one column at a time: the broadcasts of several spill scalar registers
    }
    return ok;
}

// x L_tile^T = the row x, tile_t[k][t] = L_tile[t][k]
template <int T>
__device__ __forceinline__ void chol_row_solve(double (&x)[T], const double (*tile_t)[T], const double* rl) {
#pragma unroll
    for (int k = 0; k < T; ++k) {
        x[k] *= rl[k];
#pragma unroll
        for (int t = k + 1; t < T; ++t) x[t] -= x[k] * tile_t[k][t];
        __builtin_amdgcn_sched_barrier(0);
    }
}

// S = L L^T (S symmetrised in the workspace) with the lower triangle packed by columns in LDS, one workgroup per
// problem: panels of 16 columns (diagonal tile in the registers of one wavefront, one thread per row
// below it, trailing update by v_mfma_f64_16x16x4 tiles). The chain of pivots bounds it. The
// column-at-a-time form in global memory took 557 us at 175 structures (two block barriers and a
// pass over the trailing matrix in the L2 per column), this one 93.
__global__ void __launch_bounds__(kCholThreads) k_gep_chol_lds(const SlotDesc* __restrict__ slots, int n) {
    const SlotDesc& sd = slots[blockIdx.z];
    extern __shared__ double a[];
    __shared__ double tile_t[kCholTile][kCholTile], rl[kCholTile];
    __shared__ int bad;
    const auto Lm = to_global(sd.gep);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, k4 = lane >> 4;
    constexpr int kWaves = kCholThreads / 64, kRowBlocks = (kCholLdsMaxN + 63) / 64;
    auto col = [n](int j) { return j * n - j * (j + 1) / 2; };  // element (i, j), i >= j, at col(j) + i
    if (tid == 0) bad = 0;
    for (int j0 = wave; j0 < n; j0 += 4 * kWaves) {
        double v[4][kRowBlocks];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int b = 0; b < kRowBlocks; ++b)
                v[u][b] = Lm[min(64 * b + lane, n - 1) + (size_t)n * min(j0 + kWaves * u, n - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int b = 0; b < kRowBlocks; ++b) {
                const int i = 64 * b + lane, j = j0 + kWaves * u;
                if (i >= j && i < n) a[col(j) + i] = v[u][b];
            }
    }
    __syncthreads();
    for (int j0 = 0; j0 < n; j0 += kCholTile) {
        const int jb = min(kCholTile, n - j0);
        if (wave == 0) {
            double r[kCholTile];
            const int row = min(lane, jb - 1);
#pragma unroll
            for (int k = 0; k < kCholTile; ++k) {
                const int kc = min(k, row);
                r[k] = a[col(j0 + kc) + j0 + row];
            }
            if (!chol_tile<kCholTile>(r, jb, rl, lane) && lane == 0) bad = 1;
            if (lane < kCholTile)
#pragma unroll
                for (int k = 0; k < kCholTile; ++k) tile_t[k][lane] = r[k];
        }
        __syncthreads();
        if (bad) {  // uniform; the later kernels run on meaningless values the host discards
            if (tid == 0) to_global(sd.flags)[FLAG_METRIC] = 1;
            return;
        }
        if (tid < 256) {
            const int i = tid & 15, k = tid >> 4;
            if (k <= i && i < jb) a[col(j0 + k) + j0 + i] = tile_t[k][i];
        }
        if (j0 + jb >= n) break;
        for (int i = j0 + jb + tid; i < n; i += kCholThreads) {  // a full panel: jb == kCholTile here
            double x[kCholTile];
#pragma unroll
            for (int k = 0; k < kCholTile; ++k) x[k] = a[col(j0 + k) + i];
            chol_row_solve<kCholTile>(x, tile_t, rl);
#pragma unroll
            for (int k = 0; k < kCholTile; ++k) a[col(j0 + k) + i] = x[k];
        }
        __syncthreads();
        const int r0 = j0 + jb, tiles = (n - r0 + 15) / 16;
        int ti = 0, tj = wave;  // wavefront's tiles of the lower triangle, row by row
        for (;; tj += kWaves) {
            while (tj > ti) tj -= ++ti;
            if (ti >= tiles) break;
            const int i = r0 + 16 * ti, j = r0 + 16 * tj, ic = min(i + i16, n - 1), jc = min(j + i16, n - 1);
            chol_double4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int t = 0; t < kCholTile; t += 4) {
                const double* p = a + col(j0 + t + k4);
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(p[ic], p[jc], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int ir = i + 4 * v + k4, jr = j + i16;
                if (ir < n && jr <= ir) a[col(jr) + ir] -= acc[v];
            }
        }
        __syncthreads();
    }
    __syncthreads();
    for (int j = wave; j < n; j += kWaves)
        for (int i = j + lane; i < n; i += 64) Lm[i + (size_t)n * j] = a[col(j) + i];
}

// Panel of the blocked Cholesky for spaces beyond it (launches of few problems): every workgroup factors the
// diagonal tile in the registers of its first wavefront and solves its rows below it against it, one row per
// thread. The factored tile goes to a scratch area (`last`: in place; no other workgroup reads it then),
// from where k_chol_syrk of the panel puts it into L. 18 us per panel of 32 columns, the chain of pivots;
// a tile kernel with three barriers a column and a solve kernel of its own took 38.
__global__ void __launch_bounds__(256) k_chol_panel(const SlotDesc* __restrict__ slots, int n, int j0, int jb, int last) {
    const SlotDesc& sd = slots[blockIdx.z];
    const auto L = to_global(sd.gep);
    const auto scratch = L + 3 * (size_t)n * n + 9 * (size_t)n;  // gep_core_doubles: free until L^-1 is formed
    __shared__ double tile_t[kCholPanel][kCholPanel], rl[kCholPanel];
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 64) {
        double r[kCholPanel];
        const int row = min(lane, jb - 1);
#pragma unroll
        for (int k = 0; k < kCholPanel; ++k) {
            r[k] = L[(size_t)(j0 + row) + (size_t)n * (j0 + min(k, row))];
        }
        if (!chol_tile<kCholPanel>(r, jb, rl, lane) && lane == 0)
            to_global(sd.flags)[FLAG_METRIC] = 1;  // the solve goes on with values the host discards
        if (lane < kCholPanel)
#pragma unroll
            for (int k = 0; k < kCholPanel; ++k) tile_t[k][lane] = r[k];
    }
    __syncthreads();
    if (blockIdx.x == 0)
        for (int idx = tid; idx < kCholPanel * kCholPanel; idx += 256) {
            const int r = idx % kCholPanel, k = idx / kCholPanel;
            if (k > r || r >= jb) continue;
            if (last) L[(size_t)(j0 + r) + (size_t)n * (j0 + k)] = tile_t[k][r];
            else scratch[r * kCholPanel + k] = tile_t[k][r];
        }
    const int i = j0 + jb + blockIdx.x * 256 + tid;
    if (last || i >= n) return;  // a panel with rows below it is full: jb == kCholPanel
    double x[kCholPanel];
#pragma unroll
    for (int k = 0; k < kCholPanel; ++k) x[k] = L[(size_t)i + (size_t)n * (j0 + k)];
    chol_row_solve<kCholPanel>(x, tile_t, rl);
#pragma unroll
    for (int k = 0; k < kCholPanel; ++k) L[(size_t)i + (size_t)n * (j0 + k)] = x[k];
}

// ---- L^-1 -----------------------------------------------------------------------------------------------

// Column j of L^-1 by columns of L, one wavefront per column: x_k = x_k / L_kk, then x -= L[:, k] x_k, the
// column in registers (lane r: rows r, r + 64, ...). The columns of L are read with unit stride and do
// not depend on x, so the next ones are in flight while these are used; a sum over each row of L instead
// reads L with stride n (117 us at 175 structures, now 48).
template <int R>
__global__ void __launch_bounds__(256) k_gep_linv_cols(const SlotDesc* __restrict__ slots, int n) {
    const SlotDesc& sd = slots[blockIdx.z];
    const auto L = to_global(static_cast<const double*>(sd.gep));
    const auto V = to_global(sd.gep) + 2 * (size_t)n * n;
    const int lane = threadIdx.x & 63, j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= n) return;
    double x[R], rd[R];  // rd: 1 / L_ii of the lane's rows
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = min(lane + 64 * r, n - 1);
        x[r] = lane + 64 * r == j ? 1.0 : 0.0;
        rd[r] = 1.0 / L[i + (size_t)n * i];
    }
    constexpr int kAhead = R <= 4 ? 8 : R <= 7 ? 4 : R <= 16 ? 2 : 1;
    auto fetch = [&](double (&c)[kAhead][R], int k0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) c[u][r] = L[min(lane + 64 * r, n - 1) + (size_t)n * min(k0 + u, n - 1)];
    };
    double c[kAhead][R], next[kAhead][R];
    fetch(c, j);
    for (int k0 = j; k0 < n; k0 += kAhead) {
        fetch(next, k0 + kAhead);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = k0 + u;
            if (k < n) {
                double xk = 0.0;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (k >> 6 == r) xk = wave_bcast(x[r] * rd[r], k & 63);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int i = lane + 64 * r;
                    x[r] = i == k ? xk : i > k ? x[r] - c[u][r] * xk : x[r];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) c[u][r] = next[u][r];
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (lane + 64 * r < n) V[lane + 64 * r + (size_t)n * j] = x[r];
}

// ---- lowest eigenpair of a tridiagonal in LDS --------------------------------------------------------------

constexpr double kRitzTolerance = 4.0e-16;

// Lowest eigenpair of the tridiagonal (d, e) of order k on one wavefront, as tridiag_lowest_wave but with the
// rows in LDS: de[i] = (d_i, e_{i-1}^2) for i < k + 4 (zeros past k), e[i] = T[i+1, i]. f: scratch of k + 4 pairs;
// y: the unit vector (k + 4 entries). Returns the eigenvalue; norm receives the largest Gershgorin bound.
__device__ double tridiag_lowest_lds(int k, const double2* de, const double* e, double2* f, double* y, double& norm) {
    const int lane = threadIdx.x & 63;
    double lo = 1e300, hi = -1e300;
    for (int i = lane; i < k; i += 64) {
        const double rad = (i > 0 ? fabs(e[i - 1]) : 0.0) + (i + 1 < k ? fabs(e[i]) : 0.0);
        lo = fmin(lo, de[i].x - rad);
        hi = fmax(hi, de[i].x + rad);
    }
    lo = -wave_max(-lo);
    hi = wave_max(hi);
    norm = fmax(fabs(lo), fabs(hi));
    const double pad = 1e-12 * norm + 1e-300;
    lo -= pad;
    hi += pad;
    double unused = 0.0;
    for (int it = 0; it < 64; ++it) {
        if (!(hi - lo > 1e-10 * fmax(fabs(lo), fabs(hi)))) break;
        const double x = lo + (hi - lo) * (double)(lane + 1) / 64.0;
        const uint64_t hit = __ballot(sturm_count<false>(lane, k, de, x, unused) >= 1);
        const int f = hit ? __builtin_ctzll(hit) : 64;
        const double nlo = f == 0 ? lo : lo + (hi - lo) * (double)f / 64.0;
        const double nhi = f >= 64 ? hi : lo + (hi - lo) * (double)(f + 1) / 64.0;
        lo = nlo;
        hi = nhi;
    }
    // T - lo I = L D L^T, positive definite: the pivots are ratios of the Sturm sequence at lo, whose
    // product form has no division on the chain; (p_{i+1}, p_i) of every row go to f
    {
        double pm = 1.0, pc = de[0].x - lo;
        if (!(pc > 0.0)) pc = 1e-300;  // rounding at a bracket end that touches an eigenvalue
        if (lane == 0) f[0] = make_double2(pc, 1.0);
        for (int i = 1; i < k; i += 4) {
            double2 v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = de[i + t];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                double pn = (i + t < k ? v[t].x - lo : 1.0) * pc - v[t].y * pm;
                if (!(pn > 0.0)) pn = 1e-300;
                if (lane == 0 && i + t < k) f[i + t] = make_double2(pn, pc);
                pm = pc;
                pc = pn;
            }
            if ((i & 7) == 5) {
                const int ex = ilogb(fmax(pc, pm));
                pc = ldexp(pc, -ex);
                pm = ldexp(pm, -ex);
            }
        }
    }
    wave_sync();
    // rows: f[i] = (l_{i-1}, 1 / q_i), l_i = e_i / q_i the unit lower factor
    for (int i = lane; i < k; i += 64) y[i] = f[i].y / f[i].x;
    wave_sync();
    for (int i = lane; i < k; i += 64) {
        f[i].y = y[i];
        f[i + 1].x = i + 1 < k ? e[i] * y[i] : 0.0;
    }
    if (lane < 4) f[k + lane] = make_double2(0.0, 0.0);
    if (lane == 0) f[0].x = 0.0;
    for (int i = lane; i < k + 4; i += 64) y[i] = i < k ? 1.0 : 0.0;
    wave_sync();
    for (int iter = 0; iter < 2; ++iter) {
        double cur = 0.0;
        for (int i = 0; i < k; i += 4) {  // z_i = y_i - l_{i-1} z_{i-1}, then times 1 / q_i
            double2 v[4];
            double b[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v[t] = f[i + t];
                b[t] = y[i + t];
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                cur = b[t] - v[t].x * cur;
                if (lane == 0) y[i + t] = cur * v[t].y;  // rows past k: zero
            }
        }
        wave_sync();
        cur = 0.0;
        int i = k - 1;
        for (; i >= 3; i -= 4) {  // y_i = z_i / q_i - l_i y_{i+1}
            double l[4], b[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                l[t] = f[i - t + 1].x;
                b[t] = y[i - t];
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                cur = b[t] - l[t] * cur;
                if (lane == 0) y[i - t] = cur;
            }
        }
        for (; i >= 0; --i) {
            cur = y[i] - f[i + 1].x * cur;
            if (lane == 0) y[i] = cur;
        }
        wave_sync();
        double s = 0.0, big = 0.0;
        for (int r = lane; r < k; r += 64) big = fmax(big, fabs(y[r]));
        big = wave_max(big);
        const double scale = big > 0.0 ? 1.0 / big : 1.0;  // the squares of a nearly singular solve overflow
        for (int r = lane; r < k; r += 64) s += (y[r] * scale) * (y[r] * scale);
        s = scale / sqrt(wave_sum(s));
        for (int r = lane; r < k; r += 64) y[r] *= s;
        wave_sync();
    }
    double r = 0.0;
    for (int i = lane; i < k; i += 64)
        r += y[i] * (de[i].x * y[i] + 2.0 * (i + 1 < k ? e[i] * y[i + 1] : 0.0));
    return wave_sum(r);
}

// ---- Lanczos -----------------------------------------------------------------------------------------------

constexpr int kLanczosThreads = 1024;
constexpr int kLanczosMaxN = 1024;   // rows a pass of the workgroup covers
constexpr int kLanczosFirst = 24, kLanczosEvery = 12;  // basis sizes at which the Ritz pair is tested

size_t lanczos_vector_doubles(int n) { return 2 * (size_t)kLanczosThreads + 10 * (size_t)n + 64; }
// basis vectors kept in LDS (the rest, if the basis grows past them, behind the core workspace)
int lanczos_basis_in_lds(int n) {
    const size_t doubles = (160 * 1024 - 4096) / sizeof(double) - lanczos_vector_doubles(n);
    return (int)std::min<size_t>(n, doubles / n);
}

// sum over the workgroup, the wavefronts' parts in order; red: one double per wavefront
__device__ __forceinline__ double lanczos_sum(double v, double* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kLanczosThreads / 64; ++w) s += red[w];
    return s;
}

// One workgroup per problem; the basis in LDS as far as it fits, A read from the L2 with 16-byte loads (two
// rows a lane). Per step: w = A q (the columns split over the wavefronts, partial sums added in
// order), the three-term recurrence, one classical Gram-Schmidt pass over the whole basis. The loads of A
// bound it: a compute unit's address path takes about as long for a 16-byte load as for an 8-byte one, and
// with 8-byte loads a step at 429 structures took 56,000 cycles (2.09 ms in all, now 1.40). 175
// structures 0.68 ms; A in registers spills at 128 a thread (1.09 ms), A in LDS to 132 structures 0.75 against
// 0.54 ms for 32 problems. Householder before: 132 structures, 32 problems 1.70 ms on one workgroup each;
// 429 structures 4.9 ms in 427 launches and a serial tail.
__global__ void __launch_bounds__(kLanczosThreads) k_gep_lanczos(const SlotDesc* __restrict__ slots, TopoDesc topo, int cap) {
    const SlotDesc& sd = slots[blockIdx.z];
    const int n = topo.n_str, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int kWaves = kLanczosThreads / 64;
    const auto Ag = to_global(static_cast<const double*>(sd.gep)) + (size_t)n * n;
    const auto Linv = Ag + (size_t)n * n;
    const auto Qg = to_global(sd.gep) + 3 * (size_t)n * n + 9 * (size_t)n;  // gep_core_doubles
    extern __shared__ __align__(16) double lds[];
    __shared__ double red[kWaves], scalar[4];
    double2* de = reinterpret_cast<double2*>(lds);  // n + 8 rows
    double2* f2 = de + n + 8;                        // n + 8 rows
    double* e = reinterpret_cast<double*>(f2 + n + 8);
    double* qv = e + n;       // the newest basis vector
    double* w = qv + n;
    double* h = w + n;        // basis products
    double* s = h + n;        // eigenvector of T (n + 8)
    double* part = s + n + 8; // two partial sums per thread
    double* Q = part + 2 * kLanczosThreads;
    // wavefront: rows 128 (wave % row_waves) .., two per lane, of its share of the columns
    const int row_waves = (n + 127) / 128, parts = kWaves / row_waves, stride = 128 * row_waves;
    const int my_part = wave / row_waves, row = (wave - my_part * row_waves) * 128 + 2 * lane;
    const int rc = min(row, n - 2);  // n > 64; a lane at the odd end reads one row lower and shifts
    const bool active = my_part < parts, odd_end = row == n - 1;
    const int col0 = n * min(my_part, parts) / parts, col1 = n * min(my_part + 1, parts) / parts;
    for (int t = tid; t < n + 8; t += kLanczosThreads) de[t] = make_double2(0.0, 0.0);
    auto put_basis = [&](int k, int i, double v) {
        if (k < cap) Q[k * n + i] = v;
        else Qg[(size_t)n * k + i] = v;
    };
    // a fixed start with a component along every direction
    double norm2 = 0.0;
    for (int i = tid; i < n; i += kLanczosThreads) {
        uint32_t x = (uint32_t)i * 2654435761u + 12345u;
        x ^= x >> 16;
        x *= 0x45d9f3bu;
        x ^= x >> 16;
        const double v = (0.5 + (double)(x & 0xffff) / 65536.0) * (x >> 31 ? -1.0 : 1.0);
        qv[i] = v;
        norm2 += v * v;
    }
    norm2 = lanczos_sum(norm2, red);
    {
        const double f = 1.0 / sqrt(norm2);
        for (int i = tid; i < n; i += kLanczosThreads) {
            qv[i] *= f;
            put_basis(0, i, qv[i]);
        }
    }
    __syncthreads();
    // part[p][i]: sum over the p-th share of the columns j of A(i, j) qv[j]
    auto store_part = [&](double a0, double a1) {
        if (active) {
            part[my_part * stride + row] = odd_end ? a1 : a0;
            part[my_part * stride + row + 1] = a1;
        }
        __syncthreads();
    };
    auto apply = [&]() {
        double a0 = 0.0, a1 = 0.0;
        if (active) {
            const auto p = Ag + rc;
#pragma unroll 16
            for (int j = col0; j < col1; ++j) {
                const f64x2u v = *reinterpret_cast<gptr<const f64x2u>>(p + (size_t)j * n);
                const double x = qv[j];
                a0 += v[0] * x;
                a1 += v[1] * x;
            }
        }
        store_part(a0, a1);
    };
    // part[p][i]: sum over the p-th share of the first `count` basis vectors of coefficient_j q_j(i)
    auto combine = [&](int count, const double* coefficient) {
        double a0 = 0.0, a1 = 0.0;
        if (active) {
            const int j0 = count * my_part / parts, j1 = count * (my_part + 1) / parts, jl = min(j1, cap);
            int j = j0;
#pragma unroll 4
            for (; j < jl; ++j) {
                a0 += Q[j * n + rc] * coefficient[j];
                a1 += Q[j * n + rc + 1] * coefficient[j];
            }
#pragma unroll 8
            for (; j < j1; ++j) {
                const f64x2u v = *reinterpret_cast<gptr<const f64x2u>>(Qg + (size_t)n * j + rc);
                a0 += v[0] * coefficient[j];
                a1 += v[1] * coefficient[j];
            }
        }
        store_part(a0, a1);
    };
    auto collect = [&](int i) {
        double v = 0.0;
        for (int p = 0; p < parts; ++p) v += part[p * stride + i];
        return v;
    };
    double beta = 0.0;
    int k = 0, next_test = min(n, kLanczosFirst), last_k = 0;
    double last_left = 0.0;
    for (;;) {
        apply();
        // w = A q - beta q_prev - alpha q
        double dot = 0.0;
        for (int i = tid; i < n; i += kLanczosThreads) {
            double v = collect(i);
            if (k > 0) v -= beta * (k - 1 < cap ? Q[(k - 1) * n + i] : Qg[(size_t)n * (k - 1) + i]);
            w[i] = v;
            dot += v * qv[i];
        }
        const double alpha = lanczos_sum(dot, red);
        for (int i = tid; i < n; i += kLanczosThreads) w[i] -= alpha * qv[i];
        __syncthreads();
        // h_j = q_j . w, w -= sum_j h_j q_j over the whole basis
        for (int j = wave; j <= k; j += kWaves) {
            double v = 0.0;
            if (j < cap)
                for (int i = lane; i < n; i += 64) v += Q[j * n + i] * w[i];
            else
                for (int i = lane; i < n; i += 64) v += Qg[(size_t)n * j + i] * w[i];
            v = wave_sum(v);
            if (lane == 0) h[j] = v;
        }
        __syncthreads();
        combine(k + 1, h);
        double sq = 0.0;
        for (int i = tid; i < n; i += kLanczosThreads) {
            const double v = w[i] - collect(i);
            w[i] = v;
            sq += v * v;
        }
        const double nb = sqrt(lanczos_sum(sq, red));
        if (tid == 0) de[k] = make_double2(alpha + h[k], k > 0 ? beta * beta : 0.0);
        ++k;
        // a vanishing remainder (or a NaN): the basis is invariant, T is complete
        const bool invariant = !(nb > 1e-14 * fabs(alpha) && nb > 1e-280);
        if (tid == 0) e[k - 1] = invariant || k == n ? 0.0 : nb;
        if (invariant || k == n || k == next_test) {
            __syncthreads();
            if (wave == 0) {
                double norm;
                const double theta = tridiag_lowest_lds(k, de, e, f2, s, norm);
                if (lane == 0) {
                    scalar[0] = theta;
                    scalar[1] = nb * fabs(s[k - 1]) / norm;
                }
            }
            __syncthreads();
            if (invariant || k == n || scalar[1] <= kRitzTolerance) break;
            // the residual falls geometrically: the next test where the last two put the tolerance
            const double left = log(scalar[1] / kRitzTolerance), fall = last_left - left;
            const double guess = last_k > 0 && fall > 0.0 ? left / fall * (k - last_k) + 1.0 : kLanczosEvery;
            last_left = left;
            last_k = k;
            next_test = min(n, k + (int)fmin(fmax(guess, 3.0), 2.0 * kLanczosEvery));
        }
        beta = nb;
        const double f = 1.0 / nb;
        for (int i = tid; i < n; i += kLanczosThreads) {
            const double v = w[i] * f;
            qv[i] = v;
            put_basis(k, i, v);
        }
        __syncthreads();
    }
    // y = sum_j s_j q_j, normalised; lambda = y . A y
    combine(k, s);
    {
        double sq = 0.0;
        for (int i = tid; i < n; i += kLanczosThreads) {
            const double v = collect(i);
            w[i] = v;
            sq += v * v;
        }
        const double f = 1.0 / sqrt(lanczos_sum(sq, red));
        for (int i = tid; i < n; i += kLanczosThreads) qv[i] = w[i] * f;
        __syncthreads();
    }
    apply();
    double dot = 0.0;
    for (int i = tid; i < n; i += kLanczosThreads) dot += collect(i) * qv[i];
    const double lambda = lanczos_sum(dot, red);
    // c = L^-T y
    for (int i = wave; i < n; i += kWaves) {
        double v = 0.0;
        for (int j = i + lane; j < n; j += 64) v += Linv[(size_t)n * i + j] * qv[j];
        v = wave_sum(v);
        if (lane == 0) w[i] = v;
    }
    __syncthreads();
    for (int i = tid; i < n; i += kLanczosThreads) to_global(sd.coef)[i] = w[i];
    if (tid == 0) {
        to_global(sd.energy)[0] = lambda;
        to_global(sd.energy)[1] = lambda + sd.e_nuc;
    }
    // determinant coefficients for the backward weights
    for (int d = tid; d < topo.n_det; d += kLanczosThreads) {
        double v = 0.0;
        for (long long t = topo.off[d]; t < topo.off[d + 1]; ++t) v += topo.tc[t] * w[topo.ts[t]];
        to_global(sd.dcoef)[d] = v;
    }
}

}  // namespace

void launch_chol_panel(hipStream_t st, const SlotDesc* slots, unsigned z, int n, int j0, int jb) {
    const int rest = n - j0 - jb;
    hipLaunchKernelGGL(k_chol_panel, dim3((unsigned)std::max(1, (rest + 255) / 256), 1, z), dim3(256), 0, st, slots, n, j0, jb,
                       rest == 0 ? 1 : 0);
}

void launch_gep_chol_lds(hipStream_t st, const SlotDesc* slots, unsigned z, int n) {
    hipLaunchKernelGGL(k_gep_chol_lds, dim3(1, 1, z), dim3(kCholThreads), sizeof(double) * ((size_t)n * (n + 1) / 2), st, slots, n);
}

bool launch_gep_linv_cols(hipStream_t st, const SlotDesc* slots, unsigned z, int n) {
    const dim3 grid((unsigned)((n + 3) / 4), 1, z), block(256);
    if (n <= 64) hipLaunchKernelGGL(k_gep_linv_cols<1>, grid, block, 0, st, slots, n);
    else if (n <= 128) hipLaunchKernelGGL(k_gep_linv_cols<2>, grid, block, 0, st, slots, n);
    else if (n <= 192) hipLaunchKernelGGL(k_gep_linv_cols<3>, grid, block, 0, st, slots, n);
    else if (n <= 256) hipLaunchKernelGGL(k_gep_linv_cols<4>, grid, block, 0, st, slots, n);
    else if (n <= 448) hipLaunchKernelGGL(k_gep_linv_cols<7>, grid, block, 0, st, slots, n);
    else if (n <= 1024) hipLaunchKernelGGL(k_gep_linv_cols<16>, grid, block, 0, st, slots, n);
    else if (n <= 2048) hipLaunchKernelGGL(k_gep_linv_cols<32>, grid, block, 0, st, slots, n);
    else return false;
    return true;
}

bool launch_gep_lanczos(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo) {
    const int n = topo.n_str;
    if (n > kLanczosMaxN) return false;
    const int cap = lanczos_basis_in_lds(n);
    const size_t lds = (lanczos_vector_doubles(n) + (size_t)cap * n) * sizeof(double);
    hipLaunchKernelGGL(k_gep_lanczos, dim3(1, 1, z), dim3(kLanczosThreads), lds, st, slots, topo, cap);
    return true;
}

hipError_t configure_gep_large() {
    for (const void* k : {reinterpret_cast<const void*>(&k_gep_chol_lds), reinterpret_cast<const void*>(&k_gep_lanczos)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 4096);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace xmvb_amd
