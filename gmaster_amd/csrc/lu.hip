// Dense FP64 LU of the binned mode-coupling matrix and its triangular solves (the
// decoupling step: jnp.linalg.solve(mcm_binned, binned) in gmaster/workspaces.py:2106-2147).
//
// The binned coupling matrix is close to the identity for the masks MASTER is used with, so
// partial pivoting almost never exchanges rows.  gm_lu_factor therefore factors without
// pivoting (A = L U, L unit lower, in place) and raises a device flag when a pivot is zero
// or some |L_ij| > 1: that is exactly when partial pivoting would have chosen another row
// (at step j it takes the largest |A(j)_ij|, i >= j, the first one on ties, and
// L_ij = A(j)_ij / A(j)_jj), so without the flag the factors are the partially pivoted
// ones with identity permutation.  The caller uses a pivoting LU when the flag is set.
//
// Right-looking blocked algorithm, panels of kNB = 64 columns, three launches per panel:
//   k_lu_diag    the 64 x 64 diagonal block, factored by one workgroup in registers;
//   k_lu_panel   L21 = A21 U11^-1 and U12 = L11^-1 A12, 64 rows / columns per workgroup;
//   k_lu_update  A22 -= L21 U12 in 64 x 64 tiles on v_mfma_f64_16x16x4f64 (operands
//                staged in LDS; each wave a 32 x 32 quarter, 2 x 2 MFMA blocks).
// gm_lu_solve: B <- U^-1 L^-1 B for row-major B (n x nrhs), one workgroup per group of
// up to kSolveR right-hand sides, 64-row blocks: the sums over the solved blocks from the transposed
// factors (coalesced), then the block's diagonal system.
#include "common.h"

namespace gm {
namespace {

constexpr int kNB = 64;
constexpr int kSolveR = 4;
typedef double d4 __attribute__((ext_vector_type(4)));

__global__ void k_lu_clear(int* __restrict__ flag) {
    if (threadIdx.x == 0) *flag = 0;
}

// Lane r's value in every lane.
__device__ __forceinline__ double lane_value(double x, int r) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(v.x, r), __builtin_amdgcn_readlane(v.y, r)));
}

// Divisor of many quotients: a / d = q + (a - q d) y with q = a y, y = 1 / d to a unit in the
// last place (Newton's steps from the hardware's estimate).  Outside 2^-1000 .. 2^1000, where y or
// a step could leave the range, and for an infinite or NaN q, the plain quotient.
struct Divisor {
    double d, y;
    bool plain;
    __device__ __forceinline__ explicit Divisor(double v) : d(v) {
        const double m = fabs(v);
        plain = !(m > 0x1p-1000 && m < 0x1p1000);
        double r = __builtin_amdgcn_rcp(v);
        r = fma(fma(-v, r, 1.0), r, r);
        r = fma(fma(-v, r, 1.0), r, r);
        y = r;
    }
    __device__ __forceinline__ double quotient(double a) const {
        const double q = a * y;
        const double e = fma(-q, d, a);
        return fabs(q) < INFINITY ? fma(e, y, q) : q;
    }
};

// 64 elimination steps over 64 vectors of 64 columns, one workgroup of 16 waves: lane i holds vector
// i, wave w its columns 16 k + w in registers.  Step j takes l_j, the vector's multiplier of column
// j, from LDS (published one step ahead) and subtracts l_j u_jc from the columns c > j:
//   kDiag    the vectors are the block's rows; u is row j itself (readlane), l = a / pivot below it
//   kRows    rows of L21 (x U11 = a): u is U11's row j, l = x / U11[j][j] = the unknown
//   kCols    columns of U12 (L11 y = a): u is L11's column j, l = the unknown
// The owner of column j + 1 updates that column first and publishes l_{j+1} before its others, so a
// step is one barrier.  Bound: the chain of 64 steps (LDS read, fma, pivot, reciprocal, LDS write,
// barrier); 16 waves keep the other columns' updates out of it (four waves of 16 columns: 21 us for
// the diagonal block, one wave of 64 unknowns: 35 us for a panel).  |L_ij| > 1 exactly when
// |a_ij| > |pivot|: the smallest quotient above 1 does not round to 1.
//
// MI355X: diagonal block 60 - 65 us before (4 x 4 elements per thread, pivot row and column through
// LDS, an IEEE quotient in every thread) -> 19 us; panel 39 - 43 us (four rows per LDS port,
// 64 unknowns per lane) -> 17 us.
enum { kDiag, kRows, kCols };

template <int MODE>
__device__ __forceinline__ void lu_publish(double& t, int j, int i, const Divisor* own, double* lcol, bool& bad) {
    if constexpr (MODE == kCols) {
        lcol[i] = t;
    } else {
        const double a = t;
        const Divisor dv = MODE == kDiag ? Divisor(lane_value(a, j)) : *own;
        double l = dv.quotient(a);
        if (__builtin_amdgcn_readfirstlane(dv.plain)) l = a / dv.d;
        if (MODE == kRows || i > j) {
            bad = bad || fabs(a) > fabs(dv.d);
            t = l;
        } else {
            l = 0.0;
        }
        if (MODE == kDiag && dv.d == 0.0) bad = true;
        lcol[i] = l;
    }
}

template <int MODE, int KJ>
__device__ __forceinline__ void lu_steps(double (&t)[4], int w, int i, const double (*T)[kNB + 1], const Divisor* own,
                                         double (*lcol)[kNB], bool& bad) {
#pragma unroll
    for (int wj = 0; wj < 16; ++wj) {
        const int j = 16 * KJ + wj;
        double u[4];
        if constexpr (MODE != kDiag) {
#pragma unroll
            for (int k = KJ; k < 4; ++k) u[k] = T[j][16 * k + w];
        }
        __syncthreads();
        const double l = lcol[wj & 1][i];
        auto update = [&](int k) { t[k] = fma(-l, MODE == kDiag ? lane_value(t[k], j) : u[k], t[k]); };
        if (w > wj) update(KJ);
        if (w == wj + 1) lu_publish<MODE>(t[KJ], j + 1, i, own + KJ, lcol[(wj + 1) & 1], bad);
        if constexpr (KJ < 3) {
            update(KJ + 1);
            if (w == 0 && wj == 15) lu_publish<MODE>(t[KJ + 1], j + 1, i, own + KJ + 1, lcol[0], bad);
        }
#pragma unroll
        for (int k = KJ + 2; k < 4; ++k) update(k);
    }
}

template <int MODE>
__device__ __forceinline__ void lu_block(double (&t)[4], int b, int w, int i, const double (*T)[kNB + 1],
                                         const Divisor* own, double (*lcol)[kNB], bool& bad) {
    if (w == 0) lu_publish<MODE>(t[0], 0, i, own, lcol[0], bad);
    lu_steps<MODE, 0>(t, w, i, T, own, lcol, bad);
    if (b > 16) lu_steps<MODE, 1>(t, w, i, T, own, lcol, bad);
    if (b > 32) lu_steps<MODE, 2>(t, w, i, T, own, lcol, bad);
    if (b > 48) lu_steps<MODE, 3>(t, w, i, T, own, lcol, bad);
    __syncthreads();
}

// Rows and columns past the matrix are those of the identity.
__global__ __launch_bounds__(1024) void k_lu_diag(double* __restrict__ A, int n, int k0, int* __restrict__ flag) {
    __shared__ double lcol[2][kNB], S[kNB][kNB + 1];
    const int b = min(kNB, n - k0);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = threadIdx.x & 63;
    double* blk = A + (int64_t)k0 * n + k0;
#pragma unroll
    for (int r = w; r < kNB; r += 16) S[i][r] = r < b && i < b ? blk[(int64_t)r * n + i] : (r == i ? 1.0 : 0.0);
    __syncthreads();
    double t[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = S[16 * k + w][i];
    bool bad = false;
    lu_block<kDiag>(t, b, w, i, S, nullptr, lcol, bad);
#pragma unroll
    for (int k = 0; k < 4; ++k) S[16 * k + w][i] = t[k];
    __syncthreads();
#pragma unroll
    for (int r = w; r < kNB; r += 16)
        if (r < b && i < b) blk[(int64_t)r * n + i] = S[i][r];
    if (bad) atomicOr(flag, 1);
}

__global__ __launch_bounds__(1024) void k_lu_panel(double* __restrict__ A, int n, int k0, int nrb,
                                                   int* __restrict__ flag) {
    __shared__ double lcol[2][kNB], T[kNB][kNB + 1], S[kNB][kNB + 1];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = threadIdx.x & 63;
    const bool rows = (int)blockIdx.x < nrb;
    const int m0 = k0 + kNB + ((int)blockIdx.x - (rows ? 0 : nrb)) * kNB;
    bool bad = false;
    double t[4];
    if (rows) {
        Divisor own[4] = {Divisor(A[(int64_t)(k0 + w) * n + k0 + w]), Divisor(A[(int64_t)(k0 + 16 + w) * n + k0 + 16 + w]),
                          Divisor(A[(int64_t)(k0 + 32 + w) * n + k0 + 32 + w]),
                          Divisor(A[(int64_t)(k0 + 48 + w) * n + k0 + 48 + w])};
#pragma unroll
        for (int r = w; r < kNB; r += 16) {
            T[r][i] = A[(int64_t)(k0 + r) * n + k0 + i];
            S[i][r] = m0 + r < n ? A[(int64_t)(m0 + r) * n + k0 + i] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = S[16 * k + w][i];
        lu_block<kRows>(t, kNB, w, i, T, own, lcol, bad);
#pragma unroll
        for (int k = 0; k < 4; ++k) S[16 * k + w][i] = t[k];
        __syncthreads();
#pragma unroll
        for (int r = w; r < kNB; r += 16)
            if (m0 + r < n) A[(int64_t)(m0 + r) * n + k0 + i] = S[i][r];
        if (bad) atomicOr(flag, 1);
    } else {
        const bool in = m0 + i < n;
#pragma unroll
        for (int r = w; r < kNB; r += 16) T[i][r] = A[(int64_t)(k0 + r) * n + k0 + i];
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = in ? A[(int64_t)(k0 + 16 * k + w) * n + m0 + i] : 0.0;
        __syncthreads();
        lu_block<kCols>(t, kNB, w, i, T, nullptr, lcol, bad);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (in) A[(int64_t)(k0 + 16 * k + w) * n + m0 + i] = t[k];
    }
}

// A22 -= L21 U12 for the 64 x 64 tile (blockIdx.y, blockIdx.x) of the trailing matrix.
// Bound: latency (one load round, then 64 MFMAs per wave): 12 - 16 us with the staging loop's loads
// one after the other behind their bounds checks, now 5 - 8 us (n = 188, 1024).
// MFMA 16x16x4 f64: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]; accumulator
// register v holds D[4 v + l / 16][l % 16].
__global__ __launch_bounds__(256) void k_lu_update(double* __restrict__ A, int n, int k0) {
    __shared__ double As[kNB][kNB + 1];  // -L21 rows of the tile, columns k0 .. k0 + 63
    __shared__ double Bs[kNB][kNB + 1];  // U12 rows k0 .. k0 + 63, columns of the tile
    const int first = k0 + kNB;
    const int r0 = first + blockIdx.y * kNB, c0 = first + blockIdx.x * kNB;
    const int tid = threadIdx.x;
    const int w = tid >> 6, l = tid & 63;
    const int wr = 32 * (w >> 1), wc = 32 * (w & 1);
    const int lr = l & 15, lk = l >> 4;
    // all loads (clamped, not branched around) are in flight together: 16 rows of each operand per
    // wave and the wave's part of the tile
    double ar[16], br[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int r = 4 * u + w;
        ar[u] = A[(int64_t)min(r0 + r, n - 1) * n + k0 + l];
        br[u] = A[(int64_t)(k0 + r) * n + min(c0 + l, n - 1)];
    }
    d4 acc[2][2];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = r0 + wr + 16 * bi + 4 * v + lk, c = c0 + wc + 16 * bj + lr;
                acc[bi][bj][v] = A[(int64_t)min(r, n - 1) * n + min(c, n - 1)];
            }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        As[4 * u + w][l] = -ar[u];
        Bs[4 * u + w][l] = br[u];
    }
    __syncthreads();
#pragma unroll 4
    for (int kk = 0; kk < kNB; kk += 4) {
        double a[2], bb[2];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi) a[bi] = As[wr + 16 * bi + lr][kk + lk];
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) bb[bj] = Bs[kk + lk][wc + 16 * bj + lr];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
                acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[bi], bb[bj], acc[bi][bj], 0, 0, 0);
    }
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = r0 + wr + 16 * bi + 4 * v + lk, c = c0 + wc + 16 * bj + lr;
                if (r < n && c < n) A[(int64_t)r * n + c] = acc[bi][bj][v];
            }
}

// One pass over the 64-row blocks (UP: U from the last block up; else unit L from the first) for
// right-hand sides c0 .. c0 + nr - 1 <= c0 + R - 1, by one workgroup of 16 waves, lane = row of the
// block.  Per block, between two barriers each:
//   A  every wave adds four columns of the block solved just before (their factors are in
//      registers already) to its partial sums, which meet in LDS with the diagonal block;
//   B  wave q < nr solves right-hand side q (64 steps of readlane and fma; no shuffle through
//      LDS) while the other 12 waves sum the columns of the blocks before that for the next block,
//      and the loads of the next A are issued.
// The factors are read transposed, LUT[c][i], so that a wave's 64 rows are one 512-byte read.
template <int R, bool UP>
__device__ __forceinline__ void lu_pass(const double* __restrict__ LUT, int n, double* B, int nrhs, int c0, int nr,
                                        double (*T)[kNB + 1], double* D, double (*P)[R][kNB], double (*xl)[kNB]) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), s = threadIdx.x & 63;
    const int nblk = (n + kNB - 1) / kNB;
    auto block = [&](int k) { return (UP ? nblk - 1 - k : k) * kNB; };
    // rows and columns past the matrix read its last: nothing uses such rows' sums, and such
    // columns meet zeros
    auto factor = [&](int i, int c) { return LUT[(int64_t)min(c, n - 1) * n + min(i, n - 1)]; };
    double tr[4], la[4], acc[R], x = 0.0;
    // right-hand side, diagonal block and the last block's columns 4 w .. 4 w + 3 for block k
    auto fetch = [&](int k) {
        const int j0 = block(k);
        if (w < nr) x = j0 + s < n ? B[(int64_t)(j0 + s) * nrhs + c0 + w] : 0.0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            tr[u] = factor(j0 + s, j0 + 4 * w + u);
            la[u] = factor(j0 + s, block(max(k - 1, 0)) + 4 * w + u);
        }
    };
#pragma unroll
    for (int q = 0; q < R; ++q) acc[q] = 0.0;
    if (w < R) xl[w][s] = 0.0;
    fetch(0);
    __syncthreads();
    for (int k = 0; k < nblk; ++k) {
        const int j0 = block(k);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = 4 * w + u;
            T[s][c] = (UP ? c > s && j0 + c < n : c < s) ? tr[u] : 0.0;
            if (UP && c == s) D[s] = j0 + s < n ? tr[u] : 1.0;
            if (k > 0) {
#pragma unroll
                for (int q = 0; q < R; ++q) acc[q] = fma(la[u], xl[q][c], acc[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) P[w][q][s] = acc[q];
        const double b = x;
        __syncthreads();
        if (k + 1 < nblk) fetch(k + 1);
#pragma unroll
        for (int q = 0; q < R; ++q) acc[q] = 0.0;
        if (w < nr) {
            double sum = 0.0;
#pragma unroll
            for (int v = 0; v < 16; ++v) sum += P[v][w][s];
            const double y = j0 + s < n ? b - sum : 0.0;
            double z = y;
            // T is zero on and beyond the diagonal, so every lane takes every step ...
            const Divisor dv(UP ? D[s] : 1.0);
            bool redo = UP && dv.plain;
            if constexpr (UP) {
#pragma unroll 16
                for (int r = kNB - 1; r > 0; --r) {
                    const double q = z * dv.y;
                    z = fma(-T[s][r], lane_value(fma(fma(-q, dv.d, z), dv.y, q), r), z);
                }
                const double q = z * dv.y;
                z = fma(fma(-q, dv.d, z), dv.y, q);
            } else {
#pragma unroll 16
                for (int r = 0; r < kNB - 1; ++r) z = fma(-T[s][r], lane_value(z, r), z);
            }
            redo = redo || !(fabs(z) < INFINITY);
            // ... unless a value is not finite (0 times it) or a pivot far out of range
            if (__ballot(redo)) {
                z = y;
                for (int e = 0; e < kNB; ++e) {
                    const int r = UP ? kNB - 1 - e : e;
                    if (UP && s == r) z = z / dv.d;
                    const double zr = __shfl(z, r);
                    if (UP ? s < r : s > r) z = fma(-T[s][r], zr, z);
                }
            }
            xl[w][s] = z;
            if (j0 + s < n) B[(int64_t)(j0 + s) * nrhs + c0 + w] = z;
        } else if (w >= 4 && k + 1 < nblk) {
            // blocks 0 .. k - 1 of the pass: units of four columns, unit u to wave 4 + u % 12
            const int i = block(k + 1) + s;
#pragma unroll 4
            for (int u = w - 4; u < 16 * k; u += 12) {
                const int c = block(u >> 4) + 4 * (u & 15);
                const int e = s & (4 * R - 1);  // lane e: column e / R of the unit, right-hand side e % R
                double xe = B[(int64_t)min(c + e / R, n - 1) * nrhs + c0 + min(e % R, nr - 1)];
                if (c + e / R >= n || e % R >= nr) xe = 0.0;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const double f = factor(i, c + v);
#pragma unroll
                    for (int q = 0; q < R; ++q) acc[q] = fma(f, lane_value(xe, v * R + q), acc[q]);
                }
            }
        }
        __syncthreads();
    }
}

// B <- L^-1 B then U^-1 B for the right-hand sides R * blockIdx.x .. + R - 1.  Bound: the chain of
// 2 n / 64 diagonal solves while the matrix is small, the one CU's reads of the factors when large.
// MI355X, one right-hand side, n = 188: 75 us before (shuffles through LDS, one thread per row of
// the update) -> 14 us; n = 1024: 734 -> 180 us.
template <int R>
__global__ __launch_bounds__(1024) void k_lu_solve(const double* __restrict__ LUT, int n, double* B, int nrhs) {
    __shared__ double T[kNB][kNB + 1];
    __shared__ double P[16][R][kNB];
    __shared__ double xl[R][kNB], D[kNB];
    const int c0 = blockIdx.x * R, nr = min(R, nrhs - c0);
    lu_pass<R, false>(LUT, n, B, nrhs, c0, nr, T, D, P, xl);
    lu_pass<R, true>(LUT, n, B, nrhs, c0, nr, T, D, P, xl);
}

}  // namespace
}  // namespace gm

using namespace gm;

extern "C" int gm_lu_factor(double* A, int64_t n, int32_t* flag, void* stream) {
    if (!A || !flag) return fail(GM_E_ARG, "gm_lu_factor: null pointer");
    if (n < 1 || n > (1 << 20)) return fail(GM_E_ARG, "gm_lu_factor: bad size %lld", (long long)n);
    hipStream_t st = (hipStream_t)stream;
    const int nn = (int)n;
    hipLaunchKernelGGL(k_lu_clear, dim3(1), dim3(64), 0, st, flag);
    for (int k0 = 0; k0 < nn; k0 += kNB) {
        hipLaunchKernelGGL(k_lu_diag, dim3(1), dim3(1024), 0, st, A, nn, k0, flag);
        const int m = nn - k0 - kNB;
        if (m <= 0) break;
        const int nt = (m + kNB - 1) / kNB;
        hipLaunchKernelGGL(k_lu_panel, dim3(2 * nt), dim3(1024), 0, st, A, nn, k0, nt, flag);
        hipLaunchKernelGGL(k_lu_update, dim3(nt, nt), dim3(256), 0, st, A, nn, k0);
    }
    return check_launch("gm_lu_factor");
}

extern "C" int gm_lu_solve(const double* LU, const double* LUT, int64_t n, double* B, int64_t nrhs, void* stream) {
    if (!LU || !LUT || !B) return fail(GM_E_ARG, "gm_lu_solve: null pointer");
    if (n < 1 || n > (1 << 20) || nrhs < 1 || nrhs > (1 << 26))
        return fail(GM_E_ARG, "gm_lu_solve: bad sizes n=%lld nrhs=%lld", (long long)n, (long long)nrhs);
    // one right-hand side alone carries no sums of three others (n = 188: 16.3 us, 18.9 in
    // the kernel for four; n = 1024: 184 and 269)
    if (nrhs == 1)
        hipLaunchKernelGGL(k_lu_solve<1>, dim3(1), dim3(1024), 0, (hipStream_t)stream, LUT, (int)n, B, 1);
    else
        hipLaunchKernelGGL(k_lu_solve<kSolveR>, dim3((unsigned)((nrhs + kSolveR - 1) / kSolveR)), dim3(1024), 0,
                           (hipStream_t)stream, LUT, (int)n, B, (int)nrhs);
    return check_launch("gm_lu_solve");
}
