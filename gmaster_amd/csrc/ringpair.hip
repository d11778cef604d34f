// Ring FFTs of two real rings as one complex transform (FP64): Q and U of a ring for spin 2,
// the north and south ring of one |z| for spin 0.  The complex ring z = a + i b of nphi = n
// pixels needs no real-to-complex post-processing: Q + iU's spectrum is F+ itself, and the two
// spin-0 spectra are the conjugate-even and -odd parts of Z.
//
// A polar-cap ring (n = 4 q, any q up to kRingPairQ) is one radix-4 step and four q-point DFTs,
// each a Bluestein convolution (chirp z: j k = (j^2 + k^2 - (j - k)^2) / 2) of power-of-two length
// M >= 2 q, so that every ring of a size class costs the same -- a direct DFT pass over a prime
// factor p costs O(n p) and its ring held up the whole launch.  A belt ring (n = 4 nside) is one
// n-point FFT.
//
// FFT: M / 16 threads hold 16 points each; in-place radix-16 passes through LDS
// (M = 16 x 16 x M / 256, one padding word per 16 so that every stride is conflict-free),
// decimation in frequency forward and in time back, so that no pass reorders: the convolution
// multiplies the spectra in digit-reversed order.  A thread's twiddle bases depend on its index
// only and are computed once per ring.  Up to M = 2048 the four sub-transforms run side by side
// in four groups of threads, at M = 4096 two at a time (LDS: 136 KiB, and 16 KiB of chirp).
//
// Bounds: the ring's passes are a chain of barriers with 8 to 16 waves per CU (LDS holds one or two
// rings), so LDS latency and, below Nside 512, the launch.  MI355X, lmax = 3 Nside - 1, spin 2,
// microseconds, forward / inverse, before (direct passes over prime factors, Q and U separate) ->
// now; in brackets the time of the map and the spectrum at the card's copy rate:
//   Nside   64    40 /   53 ->   13 /   13    (1)
//   Nside  256   119 /  217 ->   27 /   32    (8)
//   Nside  512   352 /  632 ->   61 /   75   (32)
//   Nside 1024  1020 / 1756 ->  257 /  330  (128)
//   Nside 2048  3154 / 4942 -> 1309 / 1652  (514; the M = 4096 classes spill 0.9 KB per thread)
#include "common.h"
#include "ringpair.h"

namespace gm {
namespace {

__device__ __forceinline__ int pad(int a) { return a + (a >> 4); }

__device__ inline double2 cis_pi(int num, int den, double sgn) {  // e^{sgn i pi num / den}
    double s, c;
    sincospi(sgn * (double)num / (double)den, &s, &c);
    return make_double2(c, s);
}

__device__ inline double2 cis_minus(double x) {  // e^{-i pi x}
    double s, c;
    sincospi(x, &s, &c);
    return make_double2(c, -s);
}

template <bool INV>
__device__ __forceinline__ double2 mul_i(double2 a) {  // times -i (forward) or i (inverse)
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

template <bool INV>
__device__ __forceinline__ void dft4(double2& a, double2& b, double2& c, double2& d) {
    const double2 s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = mul_i<INV>(csub(b, d));
    a = cadd(s0, s2);
    c = csub(s0, s2);
    b = cadd(s1, s3);
    d = csub(s1, s3);
}

// DFTs of R points, natural order in and out.
template <int R, bool INV>
__device__ __forceinline__ void dft(double2* v) {
    if constexpr (R == 2) {
        const double2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        dft4<INV>(v[0], v[2], v[4], v[6]);
        dft4<INV>(v[1], v[3], v[5], v[7]);
        const double h = 0.70710678118654752440;
        const double sg = INV ? 1.0 : -1.0;
        const double2 w1 = make_double2(h, sg * h), w3 = make_double2(-h, sg * h);
        const double2 o0 = v[1], o1 = cmul(v[3], w1), o2 = mul_i<INV>(v[5]), o3 = cmul(v[7], w3);
        const double2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, o1);
        v[5] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[6] = csub(e2, o2);
        v[3] = cadd(e3, o3);
        v[7] = csub(e3, o3);
    } else {
        static_assert(R == 16, "radix");
        constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, h = 0.70710678118654752440;
        const double sg = INV ? 1.0 : -1.0;
#pragma unroll
        for (int b = 0; b < 4; ++b) dft4<INV>(v[b], v[4 + b], v[8 + b], v[12 + b]);
        // v[4 j1 + b] holds y_b[j1]; times W16^{b j1}
        v[5] = cmul(v[5], make_double2(c1, sg * s1));
        v[6] = cmul(v[6], make_double2(h, sg * h));
        v[7] = cmul(v[7], make_double2(s1, sg * c1));
        v[9] = cmul(v[9], make_double2(h, sg * h));
        v[10] = mul_i<INV>(v[10]);
        v[11] = cmul(v[11], make_double2(-h, sg * h));
        v[13] = cmul(v[13], make_double2(s1, sg * c1));
        v[14] = cmul(v[14], make_double2(-h, sg * h));
        v[15] = cmul(v[15], make_double2(-c1, -sg * s1));
#pragma unroll
        for (int j = 0; j < 4; ++j) dft4<INV>(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
        // v[4 j1 + j2] holds X[j1 + 4 j2]
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = a + 1; b < 4; ++b) {
                const double2 t = v[4 * a + b];
                v[4 * a + b] = v[4 * b + a];
                v[4 * b + a] = t;
            }
    }
}

// v[j] *= w^j (j < 16), w^j as w4^a w^b.
__device__ __forceinline__ void twiddle16(double2 (&v)[16], double2 w, double2 w2, double2 w3, double2 w4) {
    v[1] = cmul(v[1], w);
    v[2] = cmul(v[2], w2);
    v[3] = cmul(v[3], w3);
    double2 b = w4;
#pragma unroll
    for (int a = 1; a < 4; ++a) {
        v[4 * a] = cmul(v[4 * a], b);
        v[4 * a + 1] = cmul(v[4 * a + 1], cmul(b, w));
        v[4 * a + 2] = cmul(v[4 * a + 2], cmul(b, w2));
        v[4 * a + 3] = cmul(v[4 * a + 3], cmul(b, w3));
        if (a < 3) b = cmul(b, w4);
    }
}

__device__ __forceinline__ void twiddle16(double2 (&v)[16], double2 w) {
    const double2 w2 = cmul(w, w), w3 = cmul(w2, w), w4 = cmul(w2, w2);
    twiddle16(v, w, w2, w3, w4);
}

__device__ __forceinline__ void twiddle16(double2 (&v)[16], double2 w, double2 w4) {
    const double2 w2 = cmul(w, w);
    twiddle16(v, w, w2, cmul(w2, w), w4);
}

// One M-point transform by T = M / 16 threads over z (padded, M + M / 16 words).  BELT: the fourth
// powers of the twiddle bases are evaluated, not squared twice, so w^15 carries 6 times a base's
// rounding instead of 15 times: rms error of the belt's spectra and pixels 3.9 - 5.6e-16 -> 2.2 -
// 4.5e-16 at Nside 64 - 2048 (single rings 2.3 - 4.6e-16), 1% of the launch.  A cap's convolution
// (6 - 11e-16, its single ring's direct passes 20 - 220e-16) has no registers to spare for it.
template <int M, bool BELT = false>
struct Fft {
    static constexpr int T = M / 16;
    static constexpr int kWords = M + M / 16;
    static constexpr int L2 = M / 16;                    // length after the first pass
    static constexpr int R3 = M > 256 ? M / 256 : 16;     // last length (no twiddles); 256: two passes
    static constexpr bool kMid = M > 256;                 // a middle radix-16 pass over length L2
    double2 wa, wb;  // twiddle bases
    int t;

    __device__ void init(int tid) {
        t = tid;
        wa = cis_pi(2 * t, M, -1.0);
        wb = kMid ? cis_pi(2 * (t % (L2 / 16)), L2, -1.0) : make_double2(1.0, 0.0);
    }
    // Twiddles of the first pass and of the middle one.
    template <bool INV>
    __device__ __forceinline__ void twiddle_a(double2 (&v)[16]) const {
        twiddle<INV>(v, wa, t * (2.0 / M));
    }
    template <bool INV>
    __device__ __forceinline__ void twiddle_b(double2 (&v)[16]) const {
        twiddle<INV>(v, wb, (t % (L2 / 16)) * (2.0 / L2));
    }
    template <bool INV>
    __device__ __forceinline__ static void twiddle(double2 (&v)[16], double2 w, double x) {  // w = e^{-i pi x}
        if constexpr (INV) w = cconj(w);
        if constexpr (BELT) {
            const double2 w4 = cis_minus(4.0 * x);
            twiddle16(v, w, INV ? cconj(w4) : w4);
        } else {
            twiddle16(v, w);
        }
    }
    // Position of spectrum entry k after the forward passes.
    __device__ static int pos(int k) {
        if constexpr (M == 256) return (k & 15) * 16 + (k >> 4);
        else if constexpr (R3 <= 16) return (k & 15) * L2 + ((k >> 4) & 15) * R3 + (k >> 8);
        else return (k & 15) * L2 + ((k >> 4) & 15) * R3 + ((k >> 8) & 15) * 2 + (k >> 12);
    }
    // v: points t + T i, natural order.
    __device__ __forceinline__ void first(double2 (&v)[16], double2* z) const {
        dft<16, false>(v);
        twiddle_a<false>(v);
#pragma unroll
        for (int j = 0; j < 16; ++j) z[pad(t + T * j)] = v[j];
    }
    __device__ __forceinline__ void last_inv(double2 (&v)[16], const double2* z) const {
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = z[pad(t + T * j)];
        twiddle_a<true>(v);
        dft<16, true>(v);
    }
    __device__ __forceinline__ int mid_base() const { return (t / (L2 / 16)) * L2 + t % (L2 / 16); }
    __device__ __forceinline__ void mid(double2* z) const {
        double2 v[16];
        const int b = mid_base();
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = z[pad(b + (L2 / 16) * i)];
        dft<16, false>(v);
        twiddle_b<false>(v);
#pragma unroll
        for (int i = 0; i < 16; ++i) z[pad(b + (L2 / 16) * i)] = v[i];
    }
    __device__ __forceinline__ void mid_inv(double2* z) const {
        double2 v[16];
        const int b = mid_base();
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = z[pad(b + (L2 / 16) * i)];
        twiddle_b<true>(v);
        dft<16, true>(v);
#pragma unroll
        for (int i = 0; i < 16; ++i) z[pad(b + (L2 / 16) * i)] = v[i];
    }
    // The last lengths: thread t owns the 16 consecutive words 16 t .. 16 t + 15 (16 / R3 transforms).
    __device__ __forceinline__ void tail_load(double2 (&v)[16], const double2* z) const {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = z[17 * t + i];
    }
    __device__ __forceinline__ void tail_store(const double2 (&v)[16], double2* z) const {
#pragma unroll
        for (int i = 0; i < 16; ++i) z[17 * t + i] = v[i];
    }
    template <bool INV>
    __device__ __forceinline__ static void tail(double2 (&v)[16]) {
        static_assert(R3 <= 16, "longer tails take their own passes");
#pragma unroll
        for (int b = 0; b < 16 / R3; ++b) dft<R3, INV>(v + b * R3);
    }
};

// c <- conv(c, filter): v holds the points t + 8-halves (only i < 8 are non-zero on entry, and
// only those are meant on return); f the filter's spectrum in tail order, over M.
template <int M>
__device__ __forceinline__ void convolve(const Fft<M>& F, bool act, double2 (&v)[16], const double2 (&f)[16],
                                         double2* z) {
    if (act) F.first(v, z);
    __syncthreads();
    if constexpr (Fft<M>::kMid) {
        if (act) F.mid(z);
        __syncthreads();
    }
    if (act) {
        F.tail_load(v, z);
        Fft<M>::template tail<false>(v);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = cmul(v[i], f[i]);
        Fft<M>::template tail<true>(v);
        F.tail_store(v, z);
    }
    __syncthreads();
    if constexpr (Fft<M>::kMid) {
        if (act) F.mid_inv(z);
        __syncthreads();
    }
    if (act) F.last_inv(v, z);
    __syncthreads();  // z may be overwritten
}

// e^{i pi j^2 / q}, 0 <= j < q, from ct[j], j <= q / 2: (q - j)^2 = j^2 mod 2q up to q^2.
__device__ __forceinline__ double2 chirp_at(const double2* ct, int j, int q) {
    const bool hi = 2 * j > q;
    double2 c = ct[hi ? q - j : j];
    if (hi && (q & 1)) c = make_double2(-c.x, -c.y);
    return c;
}

__device__ __forceinline__ void chirp_table(double2* ct, int q) {
    for (int j = threadIdx.x; 2 * j <= q; j += blockDim.x) ct[j] = cis_pi((j * j) % (2 * q), q, 1.0);
    __syncthreads();
}

template <bool INV>  // e^{-i pi j^2 / q} (forward), its conjugate (inverse)
__device__ __forceinline__ double2 chirp(const double2* ct, int j, int q) {
    const double2 c = chirp_at(ct, j, q);
    return INV ? c : cconj(c);
}

// Spectrum of the conjugate chirp, |j| < q, wrapped into M points, over M.
template <int M, bool INV>
__device__ __forceinline__ void chirp_spectrum(const Fft<M>& F, bool act, double2 (&f)[16], double2* z,
                                               const double2* ct, int q) {
    if (act) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = F.t + Fft<M>::T * i;
            const int k = j < q ? j : (j > M - q ? M - j : -1);
            f[i] = k >= 0 ? cconj(chirp<INV>(ct, k, q)) : make_double2(0.0, 0.0);
        }
        F.first(f, z);
    }
    __syncthreads();
    if constexpr (Fft<M>::kMid) {
        if (act) F.mid(z);
        __syncthreads();
    }
    if (act) {
        F.tail_load(f, z);
        Fft<M>::template tail<false>(f);
#pragma unroll
        for (int i = 0; i < 16; ++i) f[i] = cscale(f[i], 1.0 / M);
    }
    __syncthreads();
}

// Groups of M / 16 threads side by side (LDS bounds them) and words of a cap ring: the groups'
// buffers and the chirp table.
template <int M> struct Cap {
    static constexpr int G = M <= 2048 ? 4 : 2;
    static constexpr int kRounds = 4 / G;
    static constexpr int kActive = G * Fft<M>::T;
    static constexpr int kBuf = G * Fft<M>::kWords;
    static constexpr int kLds = kBuf + M / 4 + 1;
};

struct RingPair {
    int n;               // pixels
    int rn, rs;          // ring rows (rs < 0: none)
    int64_t on, os;      // first pixels
    int num;             // phi0 = pi num / n
};

// Spin 0: ring i (1 .. 2 nside from the north pole) and its mirror; spin 2: one ring.
template <bool SP2>
__device__ inline RingPair ring_pair(int nside, int i, bool south) {
    RingPair p;
    const int nring = 4 * nside - 1;
    const int r = SP2 && south ? nring - i : i - 1;
    const Ring g = ring_info(nside, r);
    p.n = g.nphi;
    p.num = g.phi0_num;
    p.rn = r;
    p.on = g.offset;
    p.rs = -1;
    p.os = g.offset;
    if (!SP2 && i < 2 * nside) {
        p.rs = nring - i;
        p.os = ring_info(nside, p.rs).offset;
    }
    return p;
}

// Spectrum rows from Z (natural index k at word at(k)): out[m] = w e^{-i m phi0} Z[m mod n].
template <bool SP2, typename At>
__device__ __forceinline__ void put_rows(const double2* z, At at, const RingPair& p, int nside, int L,
                                         double2* __restrict__ spec, int64_t ld) {
    const int n = p.n, step = blockDim.x;
    const double w = 4.0 * M_PI / (12.0 * (double)nside * (double)nside);
    const int m0 = SP2 ? (int)threadIdx.x - (L - 1) : (int)threadIdx.x;
    double2 ph = cscale(phase_pi(m0, p.num, n, -1.0), w);
    const double2 rot = phase_pi(step, p.num, n, -1.0);
    int k = m0 % n;
    if (k < 0) k += n;
    const int dk = step % n;
    double2* out = spec + (int64_t)p.rn * ld + (SP2 ? L - 1 : 0);
    double2* out_s = p.rs >= 0 ? spec + (int64_t)p.rs * ld : nullptr;
    for (int m = m0; m < L; m += step) {
        const double2 a = z[at(k)];
        if constexpr (SP2) {
            out[m] = cmul(ph, a);
        } else {
            const double2 b = z[at(k ? n - k : 0)];
            out[m] = cmul(ph, make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y)));
            if (out_s) out_s[m] = cmul(ph, make_double2(0.5 * (a.y + b.y), 0.5 * (b.x - a.x)));
        }
        ph = cmul(ph, rot);
        k += dk;
        if (k >= n) k -= n;
    }
}

// Alias sums of the spectrum rows: Z[k] = sum_{m = k mod n} F[m] e^{i m phi0} (spin 0: F[-m] =
// conj F[m], north + i south), k natural at word at(k).  Rings with fewer residues than threads
// split each residue over blockDim / n threads (partial sums at words part + thread).
template <bool SP2, typename At>
__device__ __forceinline__ void take_rows(double2* z, At at, int part, const RingPair& p, int L,
                                          const double2* __restrict__ spec, int64_t ld) {
    const int n = p.n, nt = blockDim.x;
    const double2* F = spec + (int64_t)p.rn * ld + (SP2 ? L - 1 : 0);
    const double2* S = p.rs >= 0 ? spec + (int64_t)p.rs * ld : nullptr;
    const bool alt = p.num != 0;
    // sum over m = k + j n in (-L, L), j = j0 + u, j0 + u + tpc, ...
    auto sum = [&](int k, int u, int tpc) {
        double2 s = make_double2(0.0, 0.0);
        const int j0 = -((L - 1 + k) / n);
#pragma unroll 8
        for (int j = j0 + u; k + j * n < L; j += tpc) {
            const int m = k + j * n;
            double2 v;
            if constexpr (SP2) {
                v = F[m];
            } else {
                const int am = m < 0 ? -m : m;
                const double2 a = F[am];
                const double2 b = S ? S[am] : make_double2(0.0, 0.0);
                // m < 0: conj F_N + i conj F_S
                v = m < 0 ? make_double2(a.x + b.y, b.x - a.y) : make_double2(a.x - b.y, a.y + b.x);
                if (m == 0) v = make_double2(a.x, b.x);
            }
            const double sg = alt && (j & 1) ? -1.0 : 1.0;
            s.x = fma(sg, v.x, s.x);
            s.y = fma(sg, v.y, s.y);
        }
        return s;
    };
    // Im F[0], zero for a real map, is Nyquist's -Im as in the transforms of single rings, and stays
    // with its own ring.
    auto done = [&](int k, double2 v) {
        if (!SP2 && 2 * k == n) {
            v.x -= F[0].y;
            if (S) v.y -= S[0].y;
        }
        z[at(k)] = v;
    };
    const int tpc = n < nt ? nt / n : 1;
    if (tpc == 1) {
        double2 ph = phase_pi(threadIdx.x, p.num, n, 1.0);
        const double2 rot = phase_pi(nt, p.num, n, 1.0);
        for (int k = threadIdx.x; k < n; k += nt) {
            done(k, cmul(sum(k, 0, 1), ph));
            ph = cmul(ph, rot);
        }
    } else {
        const int k = threadIdx.x / tpc, u = threadIdx.x % tpc;
        z[part + threadIdx.x] = k < n ? sum(k, u, tpc) : make_double2(0.0, 0.0);
        __syncthreads();
        double2 s = make_double2(0.0, 0.0);
        if ((int)threadIdx.x < n)
            for (int i = 0; i < tpc; ++i) s = cadd(s, z[part + threadIdx.x * tpc + i]);  // fixed order
        __syncthreads();
        if ((int)threadIdx.x < n) done(threadIdx.x, cmul(s, phase_pi(threadIdx.x, p.num, n, 1.0)));
    }
    __syncthreads();
}

// ------------------------------------------------------------------ polar caps
// Radix-4 step over the rows of z (word r q + k), in place.
template <bool INV>
__device__ __forceinline__ void radix4_rows(double2* z, int q) {
    for (int k = threadIdx.x; k < q; k += blockDim.x) {
        double2 u0 = z[k], u1 = z[q + k], u2 = z[2 * q + k], u3 = z[3 * q + k];
        dft4<INV>(u0, u1, u2, u3);
        z[k] = u0;
        z[q + k] = u1;
        z[2 * q + k] = u2;
        z[3 * q + k] = u3;
    }
    __syncthreads();
}

// Ring q's transforms: r = 0 .. 3 of length q, y[rd][i] of the group's r = g + G rd at t + T i.
// Forward: x[4 j + r] -> c_k e^{-2 pi i r k / n} Y_r[k]; inverse: the transpose.
template <int M, bool SP2, bool INV>
__device__ __forceinline__ void cap_ring(const RingArgs& a, int q, bool south, int map, double2* z) {
    typedef Cap<M> C;
    constexpr int T = Fft<M>::T;
    const int tid = threadIdx.x;
    const RingPair p = ring_pair<SP2>(a.nside, q, south);
    const double* xa = a.a + (SP2 ? 0 : map * a.mstride) + p.on;
    const double* xb = SP2 ? a.b + p.on : a.a + map * a.mstride + p.os;
    double2* spec = a.spec + (SP2 ? 0 : map * a.smap);
    const bool act = tid < C::kActive;
    const int g = act ? tid / T : 0;
    Fft<M> F;
    F.init(act ? tid % T : 0);
    double2* zg = z + g * Fft<M>::kWords;
    double2* ct = z + C::kBuf;
    chirp_table(ct, q);
    double2 f[16], v[16], y[C::kRounds][8];
    if constexpr (INV) {
        take_rows<SP2>(z, [](int k) { return k; }, 4 * q, p, a.L, spec, a.ld);
        radix4_rows<true>(z, q);
#pragma unroll
        for (int rd = 0; rd < C::kRounds; ++rd)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int k = F.t + T * i;
                y[rd][i] = act && k < q ? z[(g + C::G * rd) * q + k] : make_double2(0.0, 0.0);
            }
        __syncthreads();
    }
    chirp_spectrum<M, INV>(F, act, f, zg, ct, q);
#pragma unroll
    for (int rd = 0; rd < C::kRounds; ++rd) {
        const int r = g + C::G * rd;
        // e^{-+ 2 pi i r k / n} at k = t + T i: advanced by the rotation of T
        double2 w = phase_pi((int64_t)r * F.t, 1, 2 * q, INV ? 1.0 : -1.0);
        const double2 rot = phase_pi((int64_t)r * T, 1, 2 * q, INV ? 1.0 : -1.0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = F.t + T * i;
            v[i] = make_double2(0.0, 0.0);
            if (i < 8 && j < q && act) {
                const double2 c = chirp<INV>(ct, j, q);
                if constexpr (INV) v[i] = cmul(cmul(y[rd][i & 7], c), w);
                else v[i] = cmul(make_double2(xa[4 * j + r], xb[4 * j + r]), c);
            }
            if (INV && i < 7) w = cmul(w, rot);
        }
        convolve<M>(F, act, v, f, zg);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = F.t + T * i;
            y[rd][i] = make_double2(0.0, 0.0);
            if (k < q && act) {
                y[rd][i] = cmul(v[i], chirp<INV>(ct, k, q));
                if constexpr (!INV) y[rd][i] = cmul(y[rd][i], w);
            }
            if (!INV && i < 7) w = cmul(w, rot);
        }
    }
    if (act) {
#pragma unroll
        for (int rd = 0; rd < C::kRounds; ++rd)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int k = F.t + T * i, r = g + C::G * rd;
                if (k < q) z[INV ? 4 * k + r : r * q + k] = y[rd][i];
            }
    }
    __syncthreads();
    if constexpr (INV) {
        for (int j = tid; j < 4 * q; j += blockDim.x) {
            const_cast<double*>(xa)[j] = z[j].x;
            const_cast<double*>(xb)[j] = z[j].y;
        }
    } else {
        radix4_rows<false>(z, q);
        put_rows<SP2>(z, [](int k) { return k; }, p, a.nside, a.L, spec, a.ld);
    }
}

// ------------------------------------------------------------------ belt
// The middle and last passes of the belt's transform (M = 8192: 16 x 16 x 16 x 2).
template <int M, bool INV>
__device__ __forceinline__ void belt_tail(const Fft<M, true>& F, bool act, double2* z) {
    double2 v[16];
    if constexpr (M <= 4096) {
        if (act) {
            F.tail_load(v, z);
            Fft<M, true>::template tail<INV>(v);
            F.tail_store(v, z);
        }
    } else {
        // (every thread is active) length 32 = 16 x 2: butterfly t takes the words
        // 32 (t / 2) + t % 2 + 2 i, twiddles W32^(t % 2)
        const int base = 32 * (F.t >> 1) + (F.t & 1);
        const double2 w = cis_pi(F.t & 1, 16, -1.0), w4 = cis_pi(F.t & 1, 4, -1.0);
        if constexpr (!INV) {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = z[pad(base + 2 * i)];
            dft<16, false>(v);
            twiddle16(v, w, w4);
#pragma unroll
            for (int i = 0; i < 16; ++i) z[pad(base + 2 * i)] = v[i];
            __syncthreads();
            F.tail_load(v, z);
#pragma unroll
            for (int i = 0; i < 8; ++i) dft<2, false>(v + 2 * i);
            F.tail_store(v, z);
        } else {
            F.tail_load(v, z);
#pragma unroll
            for (int i = 0; i < 8; ++i) dft<2, true>(v + 2 * i);
            F.tail_store(v, z);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = z[pad(base + 2 * i)];
            twiddle16(v, cconj(w), cconj(w4));
            dft<16, true>(v);
#pragma unroll
            for (int i = 0; i < 16; ++i) z[pad(base + 2 * i)] = v[i];
        }
    }
    __syncthreads();
}

// Belt ring i0 = nside .. 3 nside (spin 2), nside .. 2 nside and its mirror (spin 0).
template <int M, bool SP2, bool INV>
__device__ __forceinline__ void belt_ring(const RingArgs& a, int i0, int map, double2* z) {
    constexpr int T = Fft<M, true>::T;
    const int tid = threadIdx.x;
    const bool south = SP2 && i0 > 2 * a.nside;
    const RingPair p = ring_pair<SP2>(a.nside, south ? 4 * a.nside - i0 : i0, south);
    const double* xa = a.a + (SP2 ? 0 : map * a.mstride) + p.on;
    const double* xb = SP2 ? a.b + p.on : a.a + map * a.mstride + p.os;
    double2* spec = a.spec + (SP2 ? 0 : map * a.smap);
    const bool two = SP2 || p.rs >= 0;
    const bool act = tid < T;
    Fft<M, true> F;
    F.init(act ? tid : 0);
    auto at = [](int k) { return pad(Fft<M, true>::pos(k)); };
    double2 v[16];
    if constexpr (!INV) {
        if (act) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int j = tid + T * i;
                v[i] = make_double2(xa[j], two ? xb[j] : 0.0);
            }
            F.first(v, z);
        }
        __syncthreads();
        if constexpr (Fft<M, true>::kMid) {
            if (act) F.mid(z);
            __syncthreads();
        }
        belt_tail<M, false>(F, act, z);
        put_rows<SP2>(z, at, p, a.nside, a.L, spec, a.ld);
    } else {
        take_rows<SP2>(z, at, 0, p, a.L, spec, a.ld);  // n >= blockDim: no partial words
        belt_tail<M, true>(F, act, z);
        if constexpr (Fft<M, true>::kMid) {
            if (act) F.mid_inv(z);
            __syncthreads();
        }
        if (act) {
            F.last_inv(v, z);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int j = tid + T * i;
                const_cast<double*>(xa)[j] = v[i].x;
                if (two) const_cast<double*>(xb)[j] = v[i].y;
            }
        }
    }
}

// ------------------------------------------------------------------ kernels
// Two launches at most, cap rings in descending q, then the belt: 512 threads for cap rings of
// M = 4096 and 2048 and the belt of 8192 points, 256 for the smaller (two of their workgroups fit
// a CU).  Rings of all sizes share a launch because each class alone leaves the chip part empty:
// one launch per class measured 50 / 54 us at Nside 256 and 361 / 433 at 1024 (spin 2).
template <bool SP2, bool INV>
__global__ __launch_bounds__(256, 2) void k_rings_256(RingArgs a, int qhi, int nbelt) {
    extern __shared__ double2 z[];
    int b = blockIdx.x;
    const int ncap = SP2 ? 2 * qhi : qhi;
    if (b < ncap) {
        const int q = qhi - (SP2 ? b >> 1 : b);
        const bool south = SP2 && (b & 1);
        if (q > 256) cap_ring<1024, SP2, INV>(a, q, south, blockIdx.y, z);
        else if (q > 128) cap_ring<512, SP2, INV>(a, q, south, blockIdx.y, z);
        else cap_ring<256, SP2, INV>(a, q, south, blockIdx.y, z);
        return;
    }
    const int i0 = a.nside + b - ncap;
    switch (nbelt ? 4 * a.nside : 0) {
        case 256: belt_ring<256, SP2, INV>(a, i0, blockIdx.y, z); break;
        case 512: belt_ring<512, SP2, INV>(a, i0, blockIdx.y, z); break;
        case 1024: belt_ring<1024, SP2, INV>(a, i0, blockIdx.y, z); break;
        case 2048: belt_ring<2048, SP2, INV>(a, i0, blockIdx.y, z); break;
        case 4096: belt_ring<4096, SP2, INV>(a, i0, blockIdx.y, z); break;
        default: break;
    }
}

template <bool SP2, bool INV>
__global__ __launch_bounds__(512, 2) void k_rings_512(RingArgs a, int qhi, int ncap) {
    extern __shared__ double2 z[];
    const int b = blockIdx.x;
    if (b < ncap) {
        const int q = qhi - (SP2 ? b >> 1 : b);
        const bool south = SP2 && (b & 1);
        if (q > 1024) cap_ring<4096, SP2, INV>(a, q, south, blockIdx.y, z);
        else cap_ring<2048, SP2, INV>(a, q, south, blockIdx.y, z);
        return;
    }
    belt_ring<8192, SP2, INV>(a, a.nside + b - ncap, blockIdx.y, z);
}

constexpr int kSmallQ = 512;  // cap rings of the 256-thread launch

template <bool SP2, bool INV>
int ring_pairs(const RingArgs& r) {
    const int qmax = r.nside - 1 < kRingPairQ ? r.nside - 1 : kRingPairQ;
    const int rings = SP2 ? 2 * r.nside + 1 : r.nside + 1;  // belt workgroups
    const unsigned maps = SP2 ? 1 : (unsigned)r.nmaps;
    const int n = 4 * r.nside;
    const bool belt = ring_pair_belt(r.nside);
    const int big = (qmax > kSmallQ ? qmax - kSmallQ : 0) * (SP2 ? 2 : 1), bbig = belt && n == 8192 ? rings : 0;
    if (big + bbig > 0) {
        size_t words = 0;
        if (qmax > 1024) words = Cap<4096>::kLds;
        else if (big) words = Cap<2048>::kLds;
        if (bbig && words < (size_t)Fft<8192>::kWords) words = Fft<8192>::kWords;
        const size_t lds = words * sizeof(double2);
        if (int e = ring_set_lds(reinterpret_cast<const void*>(&k_rings_512<SP2, INV>), lds)) return e;
        hipLaunchKernelGGL((k_rings_512<SP2, INV>), dim3(big + bbig, maps), dim3(512), lds, r.stream, r, qmax, big);
    }
    const int qs = qmax < kSmallQ ? qmax : kSmallQ, bsmall = belt && n < 8192 ? rings : 0;
    const int blocks = qs * (SP2 ? 2 : 1) + bsmall;
    if (blocks > 0) {
        size_t words = qs > 256 ? Cap<1024>::kLds : qs > 128 ? Cap<512>::kLds : Cap<256>::kLds;
        if (bsmall && words < (size_t)(n + n / 16)) words = n + n / 16;
        const size_t lds = words * sizeof(double2);
        if (int e = ring_set_lds(reinterpret_cast<const void*>(&k_rings_256<SP2, INV>), lds)) return e;
        hipLaunchKernelGGL((k_rings_256<SP2, INV>), dim3(blocks, maps), dim3(256), lds, r.stream, r, qs, bsmall);
    }
    return GM_OK;
}

}  // namespace

int ring_pairs_fwd(const RingArgs& r, bool spin2) { return spin2 ? ring_pairs<true, false>(r) : ring_pairs<false, false>(r); }
int ring_pairs_inv(const RingArgs& r, bool spin2) { return spin2 ? ring_pairs<true, true>(r) : ring_pairs<false, true>(r); }

}  // namespace gm
