// Power spectra and binning on gfx950, FP64: coupled pseudo-C_ell of healpy-packed alms
// (HBM-bound segmented reduction over m), binned spectra and binned coupling blocks.
#include <mutex>

#include "common.h"

namespace gm {
namespace {

constexpr int kClMChunk = 32;  // orders per partial in the coupled-C_ell reduction

// partial[mc][pair][l] = sum_{m in chunk mc, m <= l} c_m Re(a_lm conj b_lm)
// Bound: HBM for large lmax, else latency: the loads of kClStep orders are in flight together (one
// order at a time behind run-time component loops before: 24 us for 2 x 2 components at
// lmax 767, now 8 us).  Orders past l read order l and are dropped.
constexpr int kClStep = 8;

template <int N1, int N2>
__global__ __launch_bounds__(256) void k_cl_partial(const double2* __restrict__ a, const double2* __restrict__ b,
                                                    int64_t stride, int L, double* __restrict__ part) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    const int mc = blockIdx.y;
    const int m0 = mc * kClMChunk;
    if (l >= L || m0 > l) return;
    const int lmax = L - 1;
    double acc[N1 * N2];
#pragma unroll
    for (int p = 0; p < N1 * N2; ++p) acc[p] = 0.0;
    for (int ms = m0; ms < min(m0 + kClMChunk, l + 1); ms += kClStep) {
        double2 x[kClStep][N1], y[kClStep][N2];
#pragma unroll
        for (int u = 0; u < kClStep; ++u) {
            const int64_t ia = alm_index(l, min(ms + u, l), lmax);
#pragma unroll
            for (int i = 0; i < N1; ++i) x[u][i] = a[i * stride + ia];
#pragma unroll
            for (int j = 0; j < N2; ++j) y[u][j] = b[j * stride + ia];
        }
#pragma unroll
        for (int u = 0; u < kClStep; ++u) {
            const double w = ms + u ? 2.0 : 1.0;
            if (ms + u <= l) {
#pragma unroll
                for (int i = 0; i < N1; ++i)
#pragma unroll
                    for (int j = 0; j < N2; ++j)
                        acc[i * N2 + j] += w * (x[u][i].x * y[u][j].x + x[u][i].y * y[u][j].y);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < N1 * N2; ++p) part[((int64_t)mc * (N1 * N2) + p) * L + l] = acc[p];
}

__global__ void k_cl_final(const double* __restrict__ part, int np, int L, double* __restrict__ cl) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    const int p = blockIdx.y;
    if (l >= L) return;
    const int nmc = l / kClMChunk + 1;
    double s = 0.0;
    for (int ms = 0; ms < nmc; ms += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = part[((int64_t)min(ms + u, nmc - 1) * np + p) * L + l];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (ms + u < nmc) s += v[u];
    }
    cl[(int64_t)p * L + l] = s / (2.0 * l + 1.0);
}

__global__ void k_bin_cell(const double* __restrict__ cl, int64_t ld, const int* __restrict__ ells,
                           const int* __restrict__ bstart, int nb, const double* __restrict__ w,
                           double* __restrict__ out) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = blockIdx.y;
    if (b >= nb) return;
    double s = 0.0;
    for (int e = bstart[b]; e < bstart[b + 1]; ++e) s += w[e] * cl[c * ld + ells[e]];
    out[(int64_t)c * nb + b] = s;
}

// Binned coupling matrix: for each block M and its slots (c1, c2, sign),
//   out[b1 ncls + c1][b2 ncls + c2] = sign sum_{e1 in b1, e2 in b2} wout[e1] M[ells[e1]][ells[e2]] tin[e2].
// blockIdx.z = block of the list, blockIdx.x = nbw bins b2.  One thread per column: its sum over
// the rows of b1 (eight rows in flight), then the columns' products meet in LDS and one thread
// per bin adds its own, 256 columns at a time.  Bound: HBM for wide matrices, else latency.  One
// thread per bin read a cache line per column (16 degrees a bin: ten times the matrix's bytes,
// 1.7 ms a block at lmax 12287 -> 0.21) and one row after the other (26 us for a 3000 x 3000
// block, 4 degrees a bin -> 16; 106 -> 16 with 16 a bin).  All blocks and slots are one launch: eight slots
// of two blocks were 2 + 16 launches.
constexpr int kBinSlots = 16;  // of one launch
template <int N> struct Rows { static constexpr int value = N; };

struct BinBlocks {
    const double* M[kBinSlots];
    int nslots;
    signed char block[kBinSlots], c1[kBinSlots], c2[kBinSlots], sign[kBinSlots];
};

// NB1 bins b1 per workgroup (blockIdx.y): their rows' loads, LDS words and barriers run together.
template <int NB1>
__global__ __launch_bounds__(256) void k_bin_blocks(BinBlocks bb, int L, const int* __restrict__ ells,
                                                    const int* __restrict__ bstart, int nb,
                                                    const double* __restrict__ wout, const double* __restrict__ tin,
                                                    int ncls, int nbw, double* __restrict__ out) {
    __shared__ double val[NB1][256];
    const int tid = threadIdx.x;
    const int b10 = blockIdx.y * NB1, z = blockIdx.z;
    const int first = blockIdx.x * nbw, b2 = first + tid;
    const bool mine = tid < nbw && b2 < nb;
    const double* __restrict__ M = bb.M[z];
    const int lo = mine ? bstart[b2] : 0, hi = mine ? bstart[b2 + 1] : 0;
    const int c_end = bstart[min(first + nbw, nb)];
    int row[NB1 + 1];  // bins past the last are empty
#pragma unroll
    for (int q = 0; q <= NB1; ++q) row[q] = bstart[min(b10 + q, nb)];
    double s[NB1];
#pragma unroll
    for (int q = 0; q < NB1; ++q) s[q] = 0.0;
    for (int c0 = bstart[first]; c0 < c_end; c0 += 256) {
        const int e2 = c0 + tid;
        double v[NB1];
#pragma unroll
        for (int q = 0; q < NB1; ++q) v[q] = 0.0;
        if (e2 < c_end) {
            const int c = ells[e2];
#pragma unroll
            for (int q = 0; q < NB1; ++q) {
                auto rows = [&](auto n, int e1) {
                    double m[n.value];
#pragma unroll
                    for (int u = 0; u < n.value; ++u) m[u] = M[(int64_t)ells[e1 + u] * L + c];
#pragma unroll
                    for (int u = 0; u < n.value; ++u) v[q] = fma(wout[e1 + u], m[u], v[q]);
                };
                const int end = row[q + 1];
                int e1 = row[q];
                for (; e1 + 8 <= end; e1 += 8) rows(Rows<8>{}, e1);
                if (e1 + 4 <= end) {
                    rows(Rows<4>{}, e1);
                    e1 += 4;
                }
                for (; e1 < end; ++e1) rows(Rows<1>{}, e1);
            }
            const double t = tin[e2];
#pragma unroll
            for (int q = 0; q < NB1; ++q) v[q] *= t;
        }
#pragma unroll
        for (int q = 0; q < NB1; ++q) val[q][tid] = v[q];
        __syncthreads();
        for (int e = max(lo, c0); e < min(hi, c0 + 256); ++e)
#pragma unroll
            for (int q = 0; q < NB1; ++q) s[q] += val[q][e - c0];
        __syncthreads();
    }
    if (!mine) return;
    for (int k = 0; k < bb.nslots; ++k)
        if (bb.block[k] == z)
#pragma unroll
            for (int q = 0; q < NB1; ++q)
                if (b10 + q < nb)
                    out[((int64_t)(b10 + q) * ncls + bb.c1[k]) * ((int64_t)nb * ncls) + (int64_t)b2 * ncls + bb.c2[k]] =
                        bb.sign[k] < 0 ? -s[q] : s[q];
}

}  // namespace
}  // namespace gm

using namespace gm;

extern "C" int64_t gm_cl_work_size(int64_t lmax, int64_t npairs) {
    const int64_t L = lmax + 1;
    return ((L + kClMChunk - 1) / kClMChunk) * npairs * L;
}

extern "C" int gm_coupled_cell(const double* alm1, int64_t n1, const double* alm2, int64_t n2, int64_t alm_stride,
                               int64_t lmax, double* cl, double* work, void* stream) {
    if (!alm1 || !alm2 || !cl || !work) return fail(GM_E_ARG, "gm_coupled_cell: null pointer");
    if (lmax < 0) return fail(GM_E_ARG, "gm_coupled_cell: lmax < 0");
    if (n1 < 1 || n1 > 2 || n2 < 1 || n2 > 2) return fail(GM_E_ARG, "gm_coupled_cell: 1 or 2 components per field");
    const int64_t L = lmax + 1, nelem = L * (L + 1) / 2;
    if ((n1 > 1 || n2 > 1) && alm_stride < nelem) return fail(GM_E_SHAPE, "gm_coupled_cell: alm stride too small");
    const int nmc = (int)((L + kClMChunk - 1) / kClMChunk);
    const int np = (int)(n1 * n2);
    hipStream_t st = (hipStream_t)stream;
    const auto kernel = n1 == 1 ? (n2 == 1 ? &k_cl_partial<1, 1> : &k_cl_partial<1, 2>)
                                : (n2 == 1 ? &k_cl_partial<2, 1> : &k_cl_partial<2, 2>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((L + 255) / 256), nmc), dim3(256), 0, st,
                       reinterpret_cast<const double2*>(alm1), reinterpret_cast<const double2*>(alm2), alm_stride,
                       (int)L, work);
    hipLaunchKernelGGL(k_cl_final, dim3((unsigned)((L + 255) / 256), np), dim3(256), 0, st, work, np, (int)L, cl);
    return check_launch("gm_coupled_cell");
}

// ------------------------------------------------------------------ no-allocation variant
// The partial sums of gm_coupled_cell live in a file-scope device array instead of a
// caller's workspace.  Each GPU holds its own copy for the life of the process; host code
// uses the per-device address returned by hipGetSymbolAddress, never the symbol itself.
namespace gm {
namespace {
constexpr int64_t kClScratchDoubles = int64_t(1) << 23;  // 64 MiB: lmax <= 8191 for 4 pairs
__device__ __align__(256) double scratch[kClScratchDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

// Address of the current device's scratch array (resolved once per device).
int scratch_for_current_device(double** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(GM_E_LAUNCH, "gm_coupled_cell_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(GM_E_ARG, "gm_coupled_cell_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(GM_E_LAUNCH, "gm_coupled_cell_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<double*>(p);
    }
    *out = g_scratch_ptr[dev];
    return GM_OK;
}
}  // namespace
}  // namespace gm

extern "C" int64_t gm_coupled_cell_noalloc_max_work(void) { return kClScratchDoubles; }

extern "C" int gm_coupled_cell_noalloc(const double* alm1, int64_t n1, const double* alm2, int64_t n2,
                                       int64_t alm_stride, int64_t lmax, double* cl, void* stream) {
    if (!alm1 || !alm2 || !cl) return fail(GM_E_ARG, "gm_coupled_cell_noalloc: null pointer");
    if (lmax < 0) return fail(GM_E_ARG, "gm_coupled_cell_noalloc: lmax < 0");
    if (n1 < 1 || n1 > 2 || n2 < 1 || n2 > 2)
        return fail(GM_E_ARG, "gm_coupled_cell_noalloc: 1 or 2 components per field");
    const int64_t need = gm_cl_work_size(lmax, n1 * n2);
    if (need > kClScratchDoubles)
        return fail(GM_E_SHAPE,
                    "gm_coupled_cell_noalloc: lmax %lld with %lld pairs needs %lld scratch doubles, the maximum is "
                    "%lld (use gm_coupled_cell with a workspace)",
                    (long long)lmax, (long long)(n1 * n2), (long long)need, (long long)kClScratchDoubles);
    double* work = nullptr;
    const int rc = scratch_for_current_device(&work);
    if (rc != GM_OK) return rc;
    // every partial the final pass reads is written by the partial pass: nothing to clear
    return gm_coupled_cell(alm1, n1, alm2, n2, alm_stride, lmax, cl, work, stream);
}

extern "C" int gm_bin_cell(const double* cl, int64_t ncl, int64_t ld, const int32_t* ells, const int32_t* band_start,
                           int64_t nbands, const double* w, double* out, void* stream) {
    if (!cl || !ells || !band_start || !w || !out) return fail(GM_E_ARG, "gm_bin_cell: null pointer");
    if (ncl < 1 || nbands < 1) return fail(GM_E_ARG, "gm_bin_cell: empty input");
    hipLaunchKernelGGL(k_bin_cell, dim3((unsigned)((nbands + 127) / 128), (unsigned)ncl), dim3(128), 0,
                       (hipStream_t)stream, cl, ld, ells, band_start, (int)nbands, w, out);
    return check_launch("gm_bin_cell");
}

extern "C" int gm_bin_blocks(const double* const* blocks, int64_t nblocks, int64_t lmax, const int32_t* ells,
                             const int32_t* band_start, int64_t nbands, const double* wout, const double* tin,
                             int64_t ncls, const int32_t* slots, int64_t nslots, double* out, void* stream) {
    if (!blocks || !ells || !band_start || !wout || !tin || !slots || !out)
        return fail(GM_E_ARG, "gm_bin_blocks: null pointer");
    if (lmax < 0 || nbands < 1 || ncls < 1 || ncls > 127) return fail(GM_E_ARG, "gm_bin_blocks: bad sizes");
    if (nblocks < 1 || nslots < 1) return fail(GM_E_ARG, "gm_bin_blocks: bad sizes");
    for (int64_t k = 0; k < nblocks; ++k)
        if (!blocks[k]) return fail(GM_E_ARG, "gm_bin_blocks: null pointer");
    for (int64_t k = 0; k < nslots; ++k) {
        const int32_t* v = slots + 4 * k;
        if (v[0] < 0 || v[0] >= nblocks || v[1] < 0 || v[1] >= ncls || v[2] < 0 || v[2] >= ncls || (v[3] != 1 && v[3] != -1))
            return fail(GM_E_ARG, "gm_bin_blocks: bad slot %lld", (long long)k);
    }
    // 256 columns a workgroup: 64 bins of three degrees or more, 256 narrower ones (lmax 3071, bins of
    // one degree: 128 us in 64s, 46 in 256s).  Bins below 3.5 degrees whose workgroups of one bin b1
    // would fill the chip more than once (8 of them a CU) go two b1 to a workgroup, which is all
    // latency: lmax 3000, 1 / 2 / 3 degrees a bin 42 / 23 / 23 us with one, 33 / 22 / 16 with
    // two, 31 / 23 / 20 with four (6000: 215 / 108 / 114, 181 / 91 / 78, 155 / 90 / 73); fewer
    // workgroups are slower in pairs (lmax 1000, 3 a bin: 4.5 us in 64s, 6.8).
    const bool pairs = 7 * nbands > 2 * (lmax + 1) && nbands * ((nbands + 255) / 256) > 2048;
    const int nbw = pairs || 3 * nbands > lmax + 1 ? 256 : 64, nb1 = pairs ? 2 : 1;
    // kBinSlots slots a launch: every layout of the workspaces but one block per channel pair of a
    // joint TEB workspace (49) is one launch
    for (int64_t k0 = 0; k0 < nslots; k0 += kBinSlots) {
        BinBlocks bb{};
        int used = 0;
        bb.nslots = (int)(nslots - k0 < kBinSlots ? nslots - k0 : kBinSlots);
        for (int k = 0; k < bb.nslots; ++k) {
            const int32_t* v = slots + 4 * (k0 + k);
            int b = 0;
            while (b < used && bb.M[b] != blocks[v[0]]) ++b;
            if (b == used) bb.M[used++] = blocks[v[0]];
            bb.block[k] = (signed char)b;
            bb.c1[k] = (signed char)v[1];
            bb.c2[k] = (signed char)v[2];
            bb.sign[k] = (signed char)v[3];
        }
        hipLaunchKernelGGL(pairs ? &k_bin_blocks<2> : &k_bin_blocks<1>,
                           dim3((unsigned)((nbands + nbw - 1) / nbw), (unsigned)((nbands + nb1 - 1) / nb1), (unsigned)used),
                           dim3(256), 0, (hipStream_t)stream, bb, (int)(lmax + 1), ells, band_start, (int)nbands, wout, tin,
                           (int)ncls, nbw, out);
    }
    return check_launch("gm_bin_blocks");
}

extern "C" int gm_bin_block(const double* M, int64_t lmax, const int32_t* ells, const int32_t* band_start,
                            int64_t nbands, const double* wout, const double* tin, double* out, void* stream) {
    if (!M || !ells || !band_start || !wout || !tin || !out) return fail(GM_E_ARG, "gm_bin_block: null pointer");
    if (lmax < 0 || nbands < 1) return fail(GM_E_ARG, "gm_bin_block: bad sizes");
    const int32_t slot[4] = {0, 0, 0, 1};
    return gm_bin_blocks(&M, 1, lmax, ells, band_start, nbands, wout, tin, 1, slot, 1, out, stream);
}

// ------------------------------------------------------------------ content fingerprint
namespace gm {
namespace {

// splitmix64 finaliser (Steele, Lea & Flood 2014): a bijective 64-bit mixer.
__device__ inline uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__global__ void k_fingerprint_clear(unsigned long long* out) {
    if (threadIdx.x < 2) out[threadIdx.x] = 0ull;
}

// Two order-independent 64-bit sums of position-keyed word hashes; any change of one word
// changes both sums unless two independent 64-bit hashes collide.
// Bound: HBM and the hashes' multiplications for large buffers.  The sums meet in two words, so
// a workgroup adds once, and at most kFingerBlocks workgroups run: one atomic per wave of 2048
// workgroups queued up on them for 200 us at any size above 4 MiB (Nside 64, 384 KiB: 21 -> 4;
// Nside 1024, 96 MiB: 208 -> 33).
constexpr int kFingerThreads = 1024, kFingerBlocks = 256;

__global__ __launch_bounds__(kFingerThreads) void k_fingerprint(const uint64_t* __restrict__ w, int64_t nwords, const unsigned char* __restrict__ tail,
                              int ntail, unsigned long long* out) {
    uint64_t s1 = 0, s2 = 0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < nwords; i0 += 4 * stride) {
        uint64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = w[i0 + u * stride < nwords ? i0 + u * stride : i0];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = i0 + u * stride;
            if (i < nwords) {
                const uint64_t h = mix64(v[u] ^ mix64((uint64_t)i + 0x9e3779b97f4a7c15ull));
                s1 += h;
                s2 += mix64(h ^ 0x632be59bd9b4e019ull);
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && ntail > 0) {
        uint64_t t = 0;
        for (int k = 0; k < ntail; ++k) t |= (uint64_t)tail[k] << (8 * k);
        const uint64_t h = mix64(t ^ mix64((uint64_t)nwords + 0x9e3779b97f4a7c15ull) ^ 0xff51afd7ed558ccdull);
        s1 += h;
        s2 += mix64(h ^ 0x632be59bd9b4e019ull);
    }
    for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_down(s1, off);
        s2 += __shfl_down(s2, off);
    }
    __shared__ uint64_t part[2][kFingerThreads / 64];
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = s1;
        part[1][threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        uint64_t t = 0;
        for (int k = 0; k < kFingerThreads / 64; ++k) t += part[threadIdx.x][k];
        atomicAdd(&out[threadIdx.x], (unsigned long long)t);
    }
}

}  // namespace
}  // namespace gm

extern "C" int gm_fingerprint(const void* data, int64_t nbytes, uint64_t* out, void* stream) {
    if (!out || (nbytes > 0 && !data)) return fail(GM_E_ARG, "gm_fingerprint: null pointer");
    if (nbytes < 0) return fail(GM_E_ARG, "gm_fingerprint: nbytes < 0");
    if (reinterpret_cast<uintptr_t>(data) & 7) return fail(GM_E_ARG, "gm_fingerprint: data not 8-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    auto* o = reinterpret_cast<unsigned long long*>(out);
    hipLaunchKernelGGL(k_fingerprint_clear, dim3(1), dim3(64), 0, st, o);
    const int64_t nwords = nbytes / 8;
    const int ntail = (int)(nbytes - nwords * 8);
    int64_t blocks = (nwords + kFingerThreads - 1) / kFingerThreads;
    if (blocks > kFingerBlocks) blocks = kFingerBlocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_fingerprint, dim3((unsigned)blocks), dim3(kFingerThreads), 0, st,
                       reinterpret_cast<const uint64_t*>(data), nwords,
                       reinterpret_cast<const unsigned char*>(data) + nwords * 8, ntail, o);
    return check_launch("gm_fingerprint");
}
