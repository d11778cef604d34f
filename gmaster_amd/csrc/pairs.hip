// FP64 latitudinal kernels on folded ring pairs: one or two spin-0 maps, or one spin-2 field,
// through the spin-0 recurrence lambda_lm (two FP64 operations per degree and ring pair).
//
// Spin 0: a lane carries R ring pairs (north and south ring of one |z|); even l + m contract
// with E = N + S, odd with O = N - S.
//
// Spin 2 on the same rows.  With s^2 = sin^2(theta) the spin-2 rows W_l, X_l of orders +-m
// are combinations of lambda_{l-2} .. lambda_{l+1} (the HEALPix F1/F2 functions, Gorski et
// al. 2005), and s^2 lambda_j = lambda_j - x^2 lambda_j is a combination of lambda_{j-2},
// lambda_j, lambda_{j+2}, so every term can carry the weight 1/s^2: an analysis needs only
//     S_j(Q), S_j(U) = sum_r lambda_j(theta_r) G_r / s_r^2
// of the ring spectra of Q and U -- two spin-0 maps -- and the finish kernel forms E and B
// from degrees l - 2 .. l + 2; a synthesis is two spin-0 maps with per-degree coefficients,
// divided by s^2 at the end.  That is 6 FP64 operations per (degree, ring pair) where the
// spin-2 recurrence on every ring takes 12.  The 1/s^2 amplifies rounding towards the
// poles, so ring pairs with s^2 below the caller's split run the spin-2 recurrence instead
// (the "polar" blocks of the same launch).  In the orders m < kLowOrders the amplified rounding is
// not hidden by the rows themselves -- at m = 0 the spin-2 rows fall as s^2 towards the pole while
// the rounding of their 1/s^2 terms grows as 1/s^2, at m >= 2 both stay alike -- and those orders
// take the spin-0 rows in the belt only (s^2 >= 5/9).
// Syntheses of a field with power at l <= m + 10, Nside 64, rms error against long double over that of
// the spin-2 recurrence on every ring: orders 0 - 3 3.4 when split at 1/64 like the others, 1.0 with
// the belt alone; orders 4 - 7 1.4, 1.0; orders 8 - 15 (split at 1/64) 1.0; spectra as (l + 1)^-2
// 1.5, 1.0; 1.1, 1.0; 1.04.  The low orders' caps cost 1% of a transform (three iterations at
// Nside 1024 17.8 -> 18.0 ms, a synthesis at 2048 17.2 -> 17.3 ms, an analysis at 512 308 -> 311 us).
//
// Analysis reduction over rings: every degree each lane writes its 2K partial sums to LDS as
// 16-byte words, and once per 8 degrees the workgroup's threads sum them (T 4K reads), so the
// LDS traffic per degree is 2K words in, 2K out, against R (2 + 2K) FP64 operations.
#include "common.h"
#include "pairs.h"
#include "recurrence.h"

namespace gm {
namespace {

constexpr int kDeg = 8;  // degrees per reduction

template <int CTRL>
__device__ inline double dpp_get(double v) {
    int2 u = __builtin_bit_cast(int2, v);
    u.x = __builtin_amdgcn_update_dpp(0, u.x, CTRL, 15, 15, true);
    u.y = __builtin_amdgcn_update_dpp(0, u.y, CTRL, 15, 15, true);
    return __builtin_bit_cast(double, u);
}

// Sum of a double2 over N consecutive lanes (N = 4, 8, 16, 32; aligned): lane 0 of the group
// returns the sum of .x, lane 1 of .y.
template <int N>
__device__ inline double group_sum(double2 s) {
    const bool odd = threadIdx.x & 1;
    double v = odd ? s.y : s.x;
    v += dpp_get<0xB1>(odd ? s.x : s.y);  // quad_perm 1 0 3 2
    v += dpp_get<0x4E>(v);                // quad_perm 2 3 0 1
    if constexpr (N >= 32) v += __shfl_xor(v, 16);
    if constexpr (N >= 16) v += dpp_get<0x108>(v);  // row_shl 8: lane i takes lane i + 8
    if constexpr (N >= 8) v += dpp_get<0x104>(v);   // row_shl 4
    return v;
}

// Slot j of the rings ordered |z| ascending (0 = equator, 2u - 1 / 2u = north / south of pair u).
__device__ inline int slot_ring(int nside, int j) {
    if (j == 0) return 2 * nside - 1;
    const int u = (j + 1) / 2;
    return (j & 1) ? 2 * nside - 1 - u : 2 * nside - 1 + u;
}

// Orders m < n take the spin-0 rows for the ring pairs below j, their other ring slots in nb polar
// blocks.
constexpr int kLowOrders = 8;
struct Low {
    int n, j, nb;
    __device__ int pairs(int m, int jend) const { return m < n ? min(j, jend) : jend; }
};

struct Tables {
    const double* __restrict__ alpha;
    const double* __restrict__ gamma;
    const double* __restrict__ smant;
    const int* __restrict__ sexp;
    const int* __restrict__ nact;
    int L;  // degrees of the tables
};

// Seeds of R lanes' recurrences, lambda_M = smant 2^sexp sin^a(theta/2) cos^b(theta/2): with a = b
// (spin 0) one power of sin(theta) / 2.  The R binary powerings run in one loop (n is uniform),
// so their latencies overlap.
template <int R>
__device__ inline void pow_ext_r(const double (&x)[R], int n, double (&mant)[R], int (&e)[R]) {
    double b[R];
    int be[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        b[t] = frexp(x[t], &be[t]);
        mant[t] = 1.0;
        e[t] = 0;
    }
    while (n) {
        if (n & 1) {
#pragma unroll
            for (int t = 0; t < R; ++t) {
                int d;
                mant[t] = frexp(mant[t] * b[t], &d);
                e[t] += be[t] + d;
            }
        }
        n >>= 1;
        if (n) {
#pragma unroll
            for (int t = 0; t < R; ++t) {
                int d;
                b[t] = frexp(b[t] * b[t], &d);
                be[t] = 2 * be[t] + d;
            }
        }
    }
}

template <int R>
__device__ inline void seed_lanes(double smant, int sexp, int a, int b, const double (&shalf)[R],
                                  const double (&chalf)[R], double (&mu)[R], int (&k)[R]) {
    constexpr int thr = ExtExp<double>::thr, unit = ExtExp<double>::unit;
    double m1[R];
    int e1[R];
    if (a == b) {
        double x[R];
#pragma unroll
        for (int t = 0; t < R; ++t) x[t] = shalf[t] * chalf[t];
        pow_ext_r<R>(x, a, m1, e1);
    } else {
        double m2[R];
        int e2[R];
        pow_ext_r<R>(shalf, a, m1, e1);
        pow_ext_r<R>(chalf, b, m2, e2);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            m1[t] *= m2[t];
            e1[t] += e2[t];
        }
    }
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const double v = smant * m1[t];
        const int E = sexp + e1[t];
        const int kk = E >= thr ? 0 : (thr - E + unit - 1) / unit;
        k[t] = -kk;
        mu[t] = ldexp(v, E + unit * kk);
    }
}

// E and O combinations of ring pair j, order m (spin 2: the spectra of Q and U over s^2, from
// the +-m columns of Q + iU).
template <int K, bool SP2>
__device__ inline void load_pair(const double2* __restrict__ spec, int64_t ld, int64_t smap, int nside, int Lm, int m,
                                 int j, double sin, double2 (&e)[K], double2 (&o)[K]) {
    const int r = 2 * nside - 1 - j, rp = 2 * nside - 1 + j;
    if constexpr (!SP2) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const double2 a = spec[k * smap + (int64_t)r * ld + m];
            const double2 b = spec[k * smap + (int64_t)rp * ld + m];
            e[k] = j ? cadd(a, b) : a;
            o[k] = j ? csub(a, b) : make_double2(0.0, 0.0);
        }
    } else {
        static_assert(K == 2, "one spin-2 field is two maps");
        const double2* n = spec + (int64_t)r * ld + (Lm - 1);
        const double2* s = spec + (int64_t)rp * ld + (Lm - 1);
        const double2 np = n[m], nm = n[-m], sp = s[m], sm = s[-m];
        const double w = 0.5 / (sin * sin);
        // G_Q = (F(m) + conj F(-m)) / 2, G_U = (F(m) - conj F(-m)) / (2i)
        auto fold = [&](double2 p, double2 q, double2& gq, double2& gu) {
            gq = make_double2((p.x + q.x) * w, (p.y - q.y) * w);
            gu = make_double2((p.y + q.y) * w, (q.x - p.x) * w);
        };
        double2 nq, nu, sq, su;
        fold(np, nm, nq, nu);
        fold(sp, sm, sq, su);
        e[0] = j ? cadd(nq, sq) : nq;
        e[1] = j ? cadd(nu, su) : nu;
        o[0] = j ? csub(nq, sq) : make_double2(0.0, 0.0);
        o[1] = j ? csub(nu, su) : make_double2(0.0, 0.0);
    }
}

// One workgroup: order m, ring pairs (POL: ring slots) j0 .. j0 + 64 NW R - 1 below jhi.
// part: the partial slot's entries of order m, indexed by degree.  Degrees M .. L - 1 (blocks of
// 8 may write up to 7 entries of the order's padding).
template <int K, int R, int NW, bool SP2, bool POL>
__device__ __forceinline__ void ana_body(const double2* __restrict__ spec, int64_t ld, int64_t smap, int nside, int Lm,
                                         int spin, const Tables& tab, int m, int j0, int jhi, double* part,
                                         double2* lds) {
    constexpr int T = 64 * NW;
    constexpr int NO = kDeg * K;  // double2 outputs per reduction
    constexpr int TPO = T / NO;   // threads summing one output
    static_assert(TPO >= 4 && TPO <= 32 && T % NO == 0, "reduction layout");
    const int L = tab.L;
    const int M = POL ? (m > spin ? m : spin) : m;
    double x[R], mu0[R], mu1[R];
    int kx[R];
    constexpr int NP = POL ? 1 : 2;  // parity sets of contraction values
    double2 g[NP][R][K];
    double sh[R], ch[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int j = j0 + t * T + threadIdx.x;
        x[t] = mu1[t] = 0.0;
        sh[t] = ch[t] = 0.5;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int k = 0; k < K; ++k) g[p][t][k] = make_double2(0.0, 0.0);
        if (j < jhi) {
            const int r = POL ? slot_ring(nside, j) : 2 * nside - 1 - j;
            const Ring gr = ring_info(nside, r);
            x[t] = gr.z;
            sh[t] = gr.shalf;
            ch[t] = gr.chalf;
            if constexpr (POL) {
                g[0][t][0] = spec[(int64_t)r * ld + (Lm - 1) + m];
                if (m) g[0][t][K - 1] = spec[(int64_t)(4 * nside - 2 - r) * ld + (Lm - 1) - m];
            } else {
                load_pair<K, SP2>(spec, ld, smap, nside, Lm, m, j, gr.sin, g[0][t], g[NP - 1][t]);
            }
        }
    }
    seed_lanes<R>(tab.smant[m], tab.sexp[m], POL ? m + spin : m, POL ? (m > spin ? m - spin : spin - m) : m, sh, ch, mu0,
                  kx);
    bool anyinact = false;
#pragma unroll
    for (int t = 0; t < R; ++t) {
        if (j0 + t * T + threadIdx.x >= jhi) {
            mu0[t] = 0.0;
            kx[t] = 0;
        }
        anyinact = anyinact || (kx[t] < 0);
    }
    anyinact = __any(anyinact);

    const double* al = tab.alpha + table_base(m, L) - m;
    const double* ga = POL ? tab.gamma + table_base(m, L) - m : nullptr;
    double an[kDeg], gn[POL ? kDeg : 1];
#pragma unroll
    for (int i = 0; i < kDeg; ++i) {
        an[i] = al[M + i + 1];
        if constexpr (POL) gn[i] = ga[M + i + 1];
    }
    const int tid = threadIdx.x;
    const int o = tid / TPO, sl = tid % TPO;
    const double2* src = lds + o * T + sl;
    const int off = (o / K) * 2 * K + 2 * (o % K) + sl;  // output of lane sl (0: re, 1: im) of group o
    for (int l0 = M; l0 < L; l0 += kDeg) {
        double a[kDeg], gg[POL ? kDeg : 1];
        const int ln = l0 + kDeg < L ? l0 + kDeg : l0;  // the next block's coefficients stay inside the table
#pragma unroll
        for (int i = 0; i < kDeg; ++i) {
            a[i] = an[i];
            an[i] = al[ln + i + 1];
            if constexpr (POL) {
                gg[i] = gn[i];
                gn[i] = ga[ln + i + 1];
            }
        }
#pragma unroll
        for (int i = 0; i < kDeg; ++i) {
            double2 acc[K];
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] = make_double2(0.0, 0.0);
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const double cur = (i & 1) ? mu1[t] : mu0[t];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const double2 gv = g[(i & 1) ? NP - 1 : 0][t][k];
                    acc[k].x = fma(cur, gv.x, acc[k].x);
                    acc[k].y = fma(cur, gv.y, acc[k].y);
                }
                double c = x[t] * a[i];
                if constexpr (POL) c = fma(x[t], a[i], gg[i]);
                if (i & 1) mu0[t] = fma(c, mu1[t], -mu0[t]);
                else mu1[t] = fma(c, mu0[t], -mu1[t]);
            }
#pragma unroll
            for (int k = 0; k < K; ++k) lds[(i * K + k) * T + tid] = acc[k];
        }
        rescale<R, double>(mu0, mu1, kx, anyinact);
        __syncthreads();
        double2 s = make_double2(0.0, 0.0);
#pragma unroll
        for (int u = 0; u < NO; ++u) s = cadd(s, src[u * TPO]);
        const double v = group_sum<TPO>(s);
        if (sl < 2) part[(int64_t)l0 * (2 * K) + off] = v;
        __syncthreads();  // the next block overwrites the words
    }
}

// Sets of T ring pairs of an order's n live ones, dealt evenly to blocks of at most RMAX sets:
// block c runs sets [c spb, min((c + 1) spb, total)), and only those (a lane without a ring
// pair costs as much as one with).
struct Split {
    int total, spb;
    __device__ Split(int n, int T, int RMAX) {
        total = n > 0 ? (n + T - 1) / T : 0;
        const int nb = (total + RMAX - 1) / RMAX;
        spb = nb ? (total + nb - 1) / nb : 1;
    }
    __device__ int blocks() const { return (total + spb - 1) / spb; }
};

template <int N> struct Int { static constexpr int value = N; };

// body(Int<n>) for the block's number of sets n = 1 .. RMAX.
template <int RMAX, typename F>
__device__ __forceinline__ void with_sets(int n, F&& body) {
    if constexpr (RMAX > 1) {
        if (n < RMAX) {
            with_sets<RMAX - 1>(n, body);
            return;
        }
    }
    body(Int<RMAX>{});
}

// Grid (1-D): npol polar blocks (order-major; low.nb of each low order, nbp of the others), then
// nblk blocks of ring pairs per order, over the ring pairs jbeg .. jend - 1.  ppart: nbp slots of
// ptsize entries, then low.nb slots of the low orders'.
template <int K, int R, int NW, bool SP2, int RP>
__global__ __launch_bounds__(64 * NW, 2) void k_ana_pairs(const double2* __restrict__ spec, int64_t ld, int64_t smap,
                                                          int nside, int Lm, Tables tab, int jbeg, int jend, int nblk,
                                                          double* __restrict__ partial, Tables pol, int pbeg, int nbp,
                                                          int npol, Low low, double* __restrict__ ppart,
                                                          int64_t ptsize) {
    constexpr int T = 64 * NW;
    __shared__ double2 lds[kDeg * K * T];
    int b = blockIdx.x;
    if constexpr (SP2) {
        if (b < npol) {
            const int bl = b - low.n * low.nb;
            const bool lo = bl < 0;
            const int m = lo ? b / low.nb : low.n + bl / nbp, c = lo ? b % low.nb : bl % nbp;
            const int j0 = (lo ? 2 * low.j - 1 : pbeg) + c * T * RP;
            const int na = pol.nact[m];
            if (j0 >= na) return;
            const int64_t slot = lo ? nbp * ptsize + c * table_base(low.n, pol.L) : c * ptsize;
            double* part = ppart + (slot + table_base(m, pol.L) - m) * 4;
            ana_body<K, RP, NW, SP2, true>(spec, ld, smap, nside, Lm, 2, pol, m, j0, na, part, lds);
            return;
        }
        b -= npol;
    }
    const int m = b / nblk, c = b % nblk;
    if constexpr (SP2) jend = low.pairs(m, jend);
    const int jhi = min(tab.nact[m], jend);
    const Split sp(jhi - jbeg, T, R);
    const int n = min(sp.spb, sp.total - c * sp.spb);
    if (n <= 0) return;
    double* part = partial + ((int64_t)c * table_size(tab.L) + table_base(m, tab.L) - m) * (2 * K);
    with_sets<R>(n, [&](auto r) {
        ana_body<K, decltype(r)::value, NW, SP2, false>(spec, ld, smap, nside, Lm, 0, tab, m, jbeg + c * sp.spb * T, jhi,
                                                        part, lds);
    });
}

// ------------------------------------------------------------------ synthesis
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kStage = 32;  // degrees of coefficients staged per wave
// double2 words of LDS per wave: K per degree, and alpha (gamma) per degree
constexpr int stage_words(int K) { return kStage * K + kStage; }

// F+(+-m) of Q and U at one ring.
__device__ inline void put_spin2(double2* __restrict__ spec, int64_t ld, int Lm, int m, int ring, double2 q, double2 u) {
    double2* row = spec + (int64_t)ring * ld + (Lm - 1);
    row[m] = make_double2(q.x - u.y, q.y + u.x);
    if (m) row[-m] = make_double2(q.x + u.y, u.x - q.y);
}

// cf: the order's coefficients, K double2 per degree, indexed by degree (M .. L - 1 are read).
// Coefficients and alpha (POL: alpha, gamma) are staged in LDS, 32 degrees at a time per wave,
// and read back as broadcasts: scalar loads would share the wait counter with the LDS reads
// and expose their latency every few degrees.
template <int K, int R, int NW, bool SP2, bool POL>
__device__ __forceinline__ void syn_body(const double2* __restrict__ cf, int nside, int Lm, int spin, const Tables& tab,
                                         int m, int j0, int jhi, int jlim, double2* __restrict__ spec, int64_t ld,
                                         int64_t smap, double2* st) {
    constexpr int T = 64 * NW;
    const int L = tab.L;
    const int M = POL ? (m > spin ? m : spin) : m;
    constexpr int NP = POL ? 1 : 2;
    double x[R], mu0[R], mu1[R];
    int kx[R];
    double2 acc[NP][R][K];
    double sh[R], ch[R];
    bool anyact = false;
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int j = j0 + t * T + threadIdx.x;
        x[t] = mu1[t] = 0.0;
        sh[t] = ch[t] = 0.5;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int k = 0; k < K; ++k) acc[p][t][k] = make_double2(0.0, 0.0);
        if (j < jhi) {
            const Ring gr = ring_info(nside, POL ? slot_ring(nside, j) : 2 * nside - 1 - j);
            x[t] = gr.z;
            sh[t] = gr.shalf;
            ch[t] = gr.chalf;
            anyact = true;
        }
    }
    if (__any(anyact)) {
        seed_lanes<R>(tab.smant[m], tab.sexp[m], POL ? m + spin : m, POL ? (m > spin ? m - spin : spin - m) : m, sh, ch,
                      mu0, kx);
        bool anyinact = false;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            if (j0 + t * T + threadIdx.x >= jhi) {
                mu0[t] = 0.0;
                kx[t] = 0;
            }
            anyinact = anyinact || (kx[t] < 0);
        }
        anyinact = __any(anyinact);
        const double* al = tab.alpha + table_base(m, L) - m;
        const double* ga = POL ? tab.gamma + table_base(m, L) - m : nullptr;
        const int w = threadIdx.x >> 6, ln = threadIdx.x & 63;
        double2* my = st + w * stage_words(K);
        double* mya = reinterpret_cast<double*>(my + kStage * K);
        constexpr int NVL = (kStage * K + 63) / 64;  // coefficient words per lane and stage
        constexpr int NA = POL ? 2 : 1;
        // word e of the stage starting at degree lb (zero past the table)
        auto word = [&](int lb, int e) {
            return e < kStage * K && lb + e / K < L ? cf[(int64_t)lb * K + e] : make_double2(0.0, 0.0);
        };
        auto coef_a = [&](int lb) {  // lanes 0 .. 31: alpha_{lb + 1 + ln}; 32 .. 63: gamma
            const int l = lb + 1 + (ln & 31);
            double v = 0.0;
            if (l < L && (POL || ln < 32)) v = POL && ln >= 32 ? ga[l] : al[l];
            return v;
        };
        double2 pf[NVL];
#pragma unroll
        for (int v = 0; v < NVL; ++v) pf[v] = word(M, v * 64 + ln);
        double pa = coef_a(M);
        for (int lb = M; lb < L; lb += kStage) {
            wave_sync();  // the previous stage's reads are done
#pragma unroll
            for (int v = 0; v < NVL; ++v)
                if (v * 64 + ln < kStage * K) my[v * 64 + ln] = pf[v];
            if (ln < 32 * NA) mya[ln] = pa;
            wave_sync();
#pragma unroll
            for (int v = 0; v < NVL; ++v) pf[v] = word(lb + kStage, v * 64 + ln);
            pa = coef_a(lb + kStage);
            const int n4 = min(kStage / 4, (L - lb + 3) / 4);
#pragma unroll 1
            for (int i4 = 0; i4 < n4; ++i4) {
                double a[4], gg[POL ? 4 : 1];
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const double2 v = *reinterpret_cast<const double2*>(mya + 4 * i4 + i);
                    a[i] = v.x;
                    a[i + 1] = v.y;
                    if constexpr (POL) {
                        const double2 u = *reinterpret_cast<const double2*>(mya + 32 + 4 * i4 + i);
                        gg[i] = u.x;
                        gg[i + 1] = u.y;
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    double2 c[K];
#pragma unroll
                    for (int k = 0; k < K; ++k) c[k] = my[(4 * i4 + i) * K + k];
#pragma unroll
                    for (int t = 0; t < R; ++t) {
                        const double cur = (i & 1) ? mu1[t] : mu0[t];
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            double2& ac = acc[(i & 1) ? NP - 1 : 0][t][k];
                            ac.x = fma(cur, c[k].x, ac.x);
                            ac.y = fma(cur, c[k].y, ac.y);
                        }
                        double cc = x[t] * a[i];
                        if constexpr (POL) cc = fma(x[t], a[i], gg[i]);
                        if (i & 1) mu0[t] = fma(cc, mu1[t], -mu0[t]);
                        else mu1[t] = fma(cc, mu0[t], -mu1[t]);
                    }
                }
                if (i4 & 1) rescale<R, double>(mu0, mu1, kx, anyinact);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const int j = j0 + t * T + threadIdx.x;
        if (j >= jlim) continue;
        if constexpr (POL) {
            const int r = slot_ring(nside, j);
            spec[(int64_t)r * ld + (Lm - 1) + m] = acc[0][t][0];
            if (m) spec[(int64_t)(4 * nside - 2 - r) * ld + (Lm - 1) - m] = acc[0][t][K - 1];
        } else {
            // F_N = E + O, F_S = E - O (zero for rings beyond the polar-skip bound)
            const int r = 2 * nside - 1 - j, rp = 2 * nside - 1 + j;
            double2 n[K], s[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                n[k] = cadd(acc[0][t][k], acc[NP - 1][t][k]);
                s[k] = csub(acc[0][t][k], acc[NP - 1][t][k]);
            }
            if constexpr (SP2) {
                const Ring gr = ring_info(nside, r);
                const double rs = 1.0 / (gr.sin * gr.sin);
                put_spin2(spec, ld, Lm, m, r, cscale(n[0], rs), cscale(n[K - 1], rs));
                if (j) put_spin2(spec, ld, Lm, m, rp, cscale(s[0], rs), cscale(s[K - 1], rs));
            } else {
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    spec[k * smap + (int64_t)r * ld + m] = n[k];
                    if (j) spec[k * smap + (int64_t)rp * ld + m] = s[k];
                }
            }
        }
    }
}

// Grid (1-D): the polar blocks of orders m < mpol, the ring-pair blocks (live sets first, then
// the sets beyond the polar skip, whose outputs are zero), then the polar blocks of the other
// orders (zeros).
template <int K, int R, int NW, bool SP2, int RP>
__global__ __launch_bounds__(64 * NW, 2) void k_syn_pairs(const double2* __restrict__ coef, int nside, int Lm, Tables tab,
                                                          int jend, int nblk, const double2* __restrict__ pcoef,
                                                          Tables pol, int nbp, int npol, Low low,
                                                          double2* __restrict__ spec, int64_t ld, int64_t smap) {
    constexpr int T = 64 * NW;
    __shared__ __align__(16) double2 st[NW * stage_words(K)];
    int b = blockIdx.x;
    if constexpr (SP2) {
        const int npair = nblk * Lm;
        if (b < npol || b >= npol + npair) {
            const bool any = b < npol;
            if (!any) b -= npair;
            const int bl = b - low.n * low.nb;
            const bool lo = bl < 0;
            const int m = lo ? b / low.nb : low.n + bl / nbp, c = lo ? b % low.nb : bl % nbp;
            const int j0 = 2 * (lo ? low.j : jend) - 1 + c * T * RP;
            const double2* cf = pcoef + (table_base(m, pol.L) - m) * 2;
            syn_body<K, RP, NW, SP2, true>(cf, nside, Lm, 2, pol, m, j0, any ? pol.nact[m] : 0, 4 * nside - 1, spec, ld,
                                           smap, st);
            return;
        }
        b -= npol;
    }
    const int m = b / nblk, c = b % nblk;
    if constexpr (SP2) jend = low.pairs(m, jend);
    const int jhi = min(tab.nact[m], jend);
    const double2* cf = coef + (table_base(m, tab.L) - m) * K;
    const Split sp(jhi, T, R);
    const int n = min(sp.spb, sp.total - c * sp.spb);
    if (n > 0) {
        with_sets<R>(n, [&](auto r) {
            syn_body<K, decltype(r)::value, NW, SP2, false>(cf, nside, Lm, 0, tab, m, c * sp.spb * T, jhi, jend, spec, ld,
                                                            smap, st);
        });
    }
    // sets total, total + 1, ... hold zeros: dealt to all of the order's blocks
    for (int j = sp.total * T + c * T + threadIdx.x; j < jend; j += nblk * T) {
        const int r = 2 * nside - 1 - j, rp = 2 * nside - 1 + j;
        const double2 z = make_double2(0.0, 0.0);
        if constexpr (SP2) {
            put_spin2(spec, ld, Lm, m, r, z, z);
            if (j) put_spin2(spec, ld, Lm, m, rp, z, z);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                spec[k * smap + (int64_t)r * ld + m] = z;
                if (j) spec[k * smap + (int64_t)rp * ld + m] = z;
            }
        }
    }
}

// ------------------------------------------------------------------ spin-2 coefficients
__device__ inline double eps_lm(int j, int m) {
    if (j <= m || j <= 0) return 0.0;
    const double dj = j, dm = m;
    return sqrt((dj * dj - dm * dm) / (4.0 * dj * dj - 1.0));
}

// W_l = (w0 lambda_l + wm lambda_{l-2} + wp lambda_{l+2}) / s^2, X_l = (dX lambda_{l+1} + eX
// lambda_{l-1}) / s^2 (zero below max(m, 2)), the plain term of W_l folded into the 1/s^2 ones.
struct WX {
    double w0, wm, wp, dX, eX;
};
__device__ inline WX wx_fold(int l, int m) {
    WX c{0.0, 0.0, 0.0, 0.0, 0.0};
    if (l < 2 || l < m) return c;
    const double dl = l, dm = m, m2 = dm * dm;
    const double nrm = 2.0 / sqrt((dl + 2.0) * (dl + 1.0) * dl * (dl - 1.0));
    const double k = sqrt((2.0 * dl + 1.0) * (dl * dl - m2) / (2.0 * dl - 1.0));
    const double em = eps_lm(l - 1, m), e0 = eps_lm(l, m), e1 = eps_lm(l + 1, m), e2 = eps_lm(l + 2, m);
    const double b = -nrm * dl * (dl - 1.0) * 0.5;
    c.w0 = nrm * (m2 - dl + (dl * dl - m2) / (2.0 * dl - 1.0)) + b * (1.0 - e1 * e1 - e0 * e0);
    c.wm = nrm * k * em - b * em * e0;
    c.wp = -b * e1 * e2;
    c.dX = -nrm * dm * (dl - 1.0) * e1;
    c.eX = nrm * dm * (k - (dl - 1.0) * e0);
    return c;
}

// E, B of the spin-2 analysis: the ring-pair sums S (2 maps) of degrees l - 2 .. l + 2 and the
// polar blocks' direct / mirror sums.  mode 0 stores, 1 subtracts, 2 adds.
constexpr int kFin = 256;
__global__ __launch_bounds__(kFin) void k_finish_2(const double* __restrict__ partial, const double* __restrict__ ppart,
                                                   int T, int RMAX, int jbeg, int jend, int jsplit,
                                                   const int* __restrict__ nact,
                                                   const double* __restrict__ P, int nbp, int CHP, int mpol, Low low,
                                                   const int* __restrict__ nact2, const double* __restrict__ P2, int Lm,
                                                   int64_t ptsize, double2* __restrict__ ae, double2* __restrict__ ab,
                                                   int mode) {
    __shared__ double2 S[kFin + 4][2];
    const int Lt = Lm + 2;
    const int m = blockIdx.y, lb = m + blockIdx.x * kFin;
    if (lb >= Lm) return;
    const int nu = Split(min(nact[m], low.pairs(m, jend)) - jbeg, T, RMAX).blocks();
    const int64_t ts = table_size(Lt), pb = table_base(m, Lt) - m;
    const double2* p2 = reinterpret_cast<const double2*>(partial);
    for (int h = threadIdx.x; h < kFin + 4; h += kFin) {
        const int j = lb - 2 + h;
        double2 q = make_double2(0.0, 0.0), u = q;
        if (j >= m && j < Lt) {
            for (int c = 0; c < nu; ++c) {
                const double2* p = p2 + ((int64_t)c * ts + pb + j) * 2;
                q = cadd(q, p[0]);
                u = cadd(u, p[1]);
            }
            const double s = P[pb + j];
            q = cscale(q, s);
            u = cscale(u, s);
        }
        S[h][0] = q;
        S[h][1] = u;
    }
    __syncthreads();
    const int l = lb + threadIdx.x;
    if (l >= Lm) return;
    const int h = threadIdx.x + 2;
    const WX c = wx_fold(l, m);
    auto lin = [](double a, double2 x, double b, double2 y, double d, double2 z) {
        return make_double2(a * x.x + b * y.x + d * z.x, a * x.y + b * y.y + d * z.y);
    };
    const double2 z = make_double2(0.0, 0.0);
    const double2 wq = lin(c.w0, S[h][0], c.wm, S[h - 2][0], c.wp, S[h + 2][0]);
    const double2 wu = lin(c.w0, S[h][1], c.wm, S[h - 2][1], c.wp, S[h + 2][1]);
    const double2 xq = lin(c.dX, S[h + 1][0], c.eX, S[h - 1][0], 0.0, z);
    const double2 xu = lin(c.dX, S[h + 1][1], c.eX, S[h - 1][1], 0.0, z);
    // E = -(wq + i xu), B = i xq - wu
    double2 E = make_double2(-(wq.x - xu.y), -(wq.y + xu.x));
    double2 B = make_double2(-xq.y - wu.x, xq.x - wu.y);
    if (m < mpol && jbeg == 0 && l >= 2) {
        const bool lo = m < low.n;
        const int np = min(lo ? low.nb : nbp, (nact2[m] - (2 * (lo ? low.j : jsplit) - 1) + CHP - 1) / CHP);
        const int64_t qb = table_base(m, Lm) - m;
        const int64_t slots = lo ? nbp * ptsize : 0, stride = lo ? table_base(low.n, Lm) : ptsize;
        double2 d = z, mi = z;
        for (int k = 0; k < np; ++k) {
            const double2* p = reinterpret_cast<const double2*>(ppart) + (slots + k * stride + qb + l) * 2;
            d = cadd(d, p[0]);
            mi = cadd(mi, p[1]);
        }
        const double pl = P2[qb + l];
        const double2 plus = cscale(d, pl);
        const double2 am = m ? cscale(mi, (l & 1) ? -pl : pl) : plus;
        const double sg = (m & 1) ? -1.0 : 1.0;
        const double2 mn = make_double2(sg * am.x, -sg * am.y);  // (-1)^m conj a+_{l,-m}
        E = make_double2(E.x - 0.5 * (plus.x + mn.x), E.y - 0.5 * (plus.y + mn.y));
        B = make_double2(B.x - 0.5 * (plus.y - mn.y), B.y + 0.5 * (plus.x - mn.x));
    }
    if (l < 2) E = B = z;  // not zero times a sum that need not be finite
    const int64_t ia = alm_index(l, m, Lm - 1);
    ae[ia] = mode == 1 ? csub(ae[ia], E) : mode == 2 ? cadd(ae[ia], E) : E;
    ab[ia] = mode == 1 ? csub(ab[ia], B) : mode == 2 ? cadd(ab[ia], B) : B;
}

// Spin-2 synthesis coefficients times P: the ring-pair ones (Q, U per degree m .. L + 1; zero
// above) and, for orders m < mpol, the spin-2 recurrence's (direct, mirror).  The transpose of
// k_finish_2: GQ_j = -(w0_j E_j + wm_{j+2} E_{j+2} + wp_{j-2} E_{j-2} + i (dX_{j-1} B_{j-1} + eX_{j+1} B_{j+1})),
// GU_j = -(w0_j B_j + wm_{j+2} B_{j+2} + wp_{j-2} B_{j-2} - i (dX_{j-1} E_{j-1} + eX_{j+1} E_{j+1})).
__global__ __launch_bounds__(kFin) void k_prep_2(const double2* __restrict__ ae, const double2* __restrict__ ab,
                                                 const double* __restrict__ P, const double* __restrict__ P2, int Lm,
                                                 int mpol, double2* __restrict__ coef, double2* __restrict__ pcoef) {
    __shared__ double2 eb[kFin + 4][2];
    __shared__ WX wx[kFin + 4];
    const int Lt = Lm + 2;
    const int m = blockIdx.y, lb = m + blockIdx.x * kFin;
    if (lb >= Lt + GM_TABLE_PAD) return;
    for (int h = threadIdx.x; h < kFin + 4; h += kFin) {
        const int l = lb - 2 + h;
        double2 e = make_double2(0.0, 0.0), b = e;
        if (l >= m && l >= 2 && l < Lm) {
            const int64_t ia = alm_index(l, m, Lm - 1);
            e = ae[ia];
            b = ab[ia];
        }
        eb[h][0] = e;
        eb[h][1] = b;
        wx[h] = l < Lm ? wx_fold(l, m) : WX{0.0, 0.0, 0.0, 0.0, 0.0};
    }
    __syncthreads();
    const int l = lb + threadIdx.x, h = threadIdx.x + 2;
    if (l >= Lt + GM_TABLE_PAD) return;
    const int64_t pb = table_base(m, Lt) - m;
    const double pl = l < Lt ? P[pb + l] : 0.0;
    double2 w[2], x[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const double2 v0 = eb[h][c], vp = eb[h + 2][c], vm = eb[h - 2][c], v1 = eb[h - 1][c], v2 = eb[h + 1][c];
        w[c] = make_double2(wx[h].w0 * v0.x + wx[h + 2].wm * vp.x + wx[h - 2].wp * vm.x,
                            wx[h].w0 * v0.y + wx[h + 2].wm * vp.y + wx[h - 2].wp * vm.y);
        x[c] = make_double2(wx[h - 1].dX * v1.x + wx[h + 1].eX * v2.x, wx[h - 1].dX * v1.y + wx[h + 1].eX * v2.y);
    }
    // GQ = -(wE + i xB), GU = -(wB - i xE)
    coef[(pb + l) * 2] = make_double2(-(w[0].x - x[1].y) * pl, -(w[0].y + x[1].x) * pl);
    coef[(pb + l) * 2 + 1] = make_double2(-(w[1].x + x[0].y) * pl, -(w[1].y - x[0].x) * pl);
    if (m < mpol && l < Lm + GM_TABLE_PAD) {
        const int64_t qb = table_base(m, Lm) - m;
        double2 cd = make_double2(0.0, 0.0), cm = cd;
        if (l < Lm && l >= 2) {
            const double2 e = eb[h][0], b = eb[h][1];
            const double p2 = P2[qb + l], sg = (m & 1) ? -1.0 : 1.0, sl = (l & 1) ? -p2 : p2;
            cd = make_double2(-(e.x - b.y) * p2, -(e.y + b.x) * p2);
            cm = make_double2(-sg * (e.x + b.y) * sl, -sg * (b.x - e.y) * sl);
        }
        pcoef[(qb + l) * 2] = cd;
        pcoef[(qb + l) * 2 + 1] = cm;
    }
}

// alms of spin-0 maps: the partial slots of an order times P.
__global__ void k_finish_pairs(const double2* __restrict__ partial, int K, int T, int RMAX, int jbeg, int jend,
                               const int* __restrict__ nact, const double* __restrict__ P, int L,
                               double2* __restrict__ alm, int64_t astride, int mode) {
    const int m = blockIdx.y;
    const int nu = Split(min(nact[m], jend) - jbeg, T, RMAX).blocks();
    const int64_t pb = table_base(m, L) - m, ts = table_size(L);
    for (int l = m + blockIdx.x * blockDim.x + threadIdx.x; l < L; l += gridDim.x * blockDim.x) {
        const double p = P[pb + l];
        for (int k = 0; k < K; ++k) {
            double2 s = make_double2(0.0, 0.0);
            for (int c = 0; c < nu; ++c) s = cadd(s, partial[((int64_t)c * ts + pb + l) * K + k]);
            s = cscale(s, p);
            double2& a = alm[k * astride + alm_index(l, m, L - 1)];
            a = mode == 1 ? csub(a, s) : mode == 2 ? cadd(a, s) : s;
        }
    }
}

// ------------------------------------------------------------------ launch shapes
// R: sets of 64 NW ring pairs a workgroup carries at most.  Timed on MI355X per transform half
// (analysis with its finish, synthesis with its prep), lmax = 3 Nside - 1:
//   analysis, R 8: many pairs per lane amortise the reduction (Nside 2048, one spin-2 field:
//     8 x 4 waves 22.0 ms, 4 x 4 28.2 ms, 2 x 4 46.8 ms); at 1024 ring pairs one-wave
//     workgroups (0.46 ms against 0.61 ms with 4 waves, whose orders are too few to fill the
//     chip), at 512 and below 4-wave ones of up to 4 sets (0.13 ms against 0.15-0.16 ms), spin 2
//     one-wave ones (its polar blocks have few rings: 0.14 ms against 0.18 ms);
//   synthesis, R 6 (248 VGPRs): no reduction, so one-wave workgroups (Nside 2048, spin 2:
//     16.1 ms; R 4 16.7 ms, R 8 spills, 37 ms); one map holds fewer registers and is faster in
//     4-wave workgroups of 4 sets up to 2048 pairs (Nside 1024: 1.46-1.51 against 1.57 ms);
//     512 pairs and below: 2 x 4 waves (0.067 ms; 6 x 1 0.090 ms), spin 2 2 x 1.
struct Shape {
    int R, NW, CH;
};

Shape pair_shape(int64_t nside, int K, bool sp2, bool syn) {
    auto shape = [](int R, int NW) { return Shape{R, NW, 64 * R * NW}; };
    const int64_t np = 2 * nside;
    if (syn) {
        if (np <= 128) return shape(1, 2);
        if (np <= 512) return sp2 ? shape(2, 1) : shape(2, 4);
        return K == 1 && np <= 2048 ? shape(4, 4) : shape(6, 1);
    }
    if (np <= 128) return shape(2, 1);
    if (np <= 512) return sp2 ? shape(4, 1) : shape(4, 4);
    return np <= 1024 ? shape(8, 1) : shape(8, 4);
}

int npolar_slots(int64_t nside, int64_t jsplit) { return (int)(4 * nside - 1 - (2 * jsplit - 1)); }
constexpr int kRP = 2;

// Polar blocks of CHP ring slots beyond the ring pairs below j.
int polar_blocks(int64_t nside, int64_t j, int CHP) { return (npolar_slots(nside, j) + CHP - 1) / CHP; }

// (of a caller's m < mpol alone: its spin-2 tables need not reach further)
Low low_orders(int64_t nside, int64_t jsplit, int64_t mpol, int CHP) {
    const int64_t belt = nside + 1, j = belt < jsplit ? belt : jsplit;
    return Low{(int)(mpol < kLowOrders ? mpol : kLowOrders), (int)j, polar_blocks(nside, j, CHP)};
}

}  // namespace

int pairs_chunk(int64_t nside) { return pair_shape(nside, 1, false, false).CH; }

template <int K, bool SP2>
int launch_ana(const char* name, const double2* spec, int64_t ld, int64_t smap, int nside, int Lm, const Tables& tab,
               int jbeg, int jend, int nblk, double* partial, const Tables& pol, int pbeg, int nbp, int npol, const Low& low,
               double* ppart, int64_t ptsize, hipStream_t st) {
    const Shape s = pair_shape(nside, K, SP2, false);
    const dim3 grid((unsigned)(npol + nblk * Lm)), block(64 * s.NW);
#define GM_GO(RR, WW)                                                                                                  \
    if (s.R == RR && s.NW == WW) {                                                                                     \
        hipLaunchKernelGGL((k_ana_pairs<K, RR, WW, SP2, kRP>), grid, block, 0, st, spec, ld, smap, nside, Lm, tab, jbeg, \
                           jend, nblk, partial, pol, pbeg, nbp, npol, low, ppart, ptsize);                                 \
        return check_launch(name);                                                                                     \
    }
    GM_GO(2, 1)
    if constexpr (SP2) { GM_GO(4, 1) }
    else { GM_GO(4, 4) }
    GM_GO(8, 1)
    GM_GO(8, 4)
#undef GM_GO
    return fail(GM_E_LAUNCH, "%s: no kernel of shape R %d, NW %d", name, s.R, s.NW);
}

template <int K, bool SP2>
int launch_syn(const char* name, const double2* coef, int nside, int Lm, const Tables& tab, int jend, int nblk,
               const double2* pcoef, const Tables& pol, int nbp, int npol, int nzero, const Low& low, double2* spec,
               int64_t ld, int64_t smap, hipStream_t st) {
    const Shape s = pair_shape(nside, K, SP2, true);
    const dim3 grid((unsigned)(npol + nblk * Lm + nzero)), block(64 * s.NW);
#define GM_GO(RR, WW)                                                                                                \
    if (s.R == RR && s.NW == WW) {                                                                                   \
        hipLaunchKernelGGL((k_syn_pairs<K, RR, WW, SP2, kRP>), grid, block, 0, st, coef, nside, Lm, tab, jend, nblk, pcoef, \
                           pol, nbp, npol, low, spec, ld, smap);                                                     \
        return check_launch(name);                                                                                   \
    }
    GM_GO(1, 2)
    if constexpr (SP2) { GM_GO(2, 1) }
    else { GM_GO(2, 4) }
    if constexpr (K == 1) { GM_GO(4, 4) }
    GM_GO(6, 1)
#undef GM_GO
    return fail(GM_E_LAUNCH, "%s: no kernel of shape R %d, NW %d", name, s.R, s.NW);
}

int ana_pairs_s0(const char* name, const double* spec, int K, int64_t ld, int64_t smap, int64_t nside, int64_t L,
                 const double* alpha, const double* smant, const int32_t* sexp, const int32_t* nact, double* partial,
                 int jbeg, int jend, int nblk, void* stream) {
    const Tables tab{alpha, nullptr, smant, sexp, nact, (int)L};
    const auto* sp = reinterpret_cast<const double2*>(spec);
    hipStream_t st = (hipStream_t)stream;
    if (K == 1)
        return launch_ana<1, false>(name, sp, ld, smap, (int)nside, (int)L, tab, jbeg, jend, nblk, partial, tab, 0,
                                    1, 0, Low{0, 0, 1}, nullptr, 0, st);
    return launch_ana<2, false>(name, sp, ld, smap, (int)nside, (int)L, tab, jbeg, jend, nblk, partial, tab, 0, 1, 0,
                                Low{0, 0, 1}, nullptr, 0, st);
}

int finish_pairs_s0(const char* name, const double* partial, int K, int64_t nside, int64_t L, const int32_t* nact,
                    const double* P, double* alm, int64_t astride, int mode, int jbeg, int jend, void* stream) {
    const Shape s = pair_shape(nside, K, false, false);
    hipLaunchKernelGGL(k_finish_pairs, dim3((unsigned)((L + 255) / 256), (unsigned)L), dim3(256), 0, (hipStream_t)stream,
                       reinterpret_cast<const double2*>(partial), K, 64 * s.NW, s.R, jbeg, jend, nact, P, (int)L,
                       reinterpret_cast<double2*>(alm), astride, mode);
    return check_launch(name);
}

int syn_pairs_s0(const char* name, const double* coef, int K, int64_t nside, int64_t L, const double* alpha,
                 const double* smant, const int32_t* sexp, const int32_t* nact, double* spec, int64_t ld, int64_t smap,
                 void* stream) {
    const Tables tab{alpha, nullptr, smant, sexp, nact, (int)L};
    const auto* cf = reinterpret_cast<const double2*>(coef);
    auto* sp = reinterpret_cast<double2*>(spec);
    hipStream_t st = (hipStream_t)stream;
    const int CH = pair_shape(nside, K, false, true).CH;
    const int nblk = (int)((2 * nside + CH - 1) / CH);
    if (K == 1)
        return launch_syn<1, false>(name, cf, (int)nside, (int)L, tab, (int)(2 * nside), nblk, nullptr, tab, 1, 0, 0,
                                    Low{0, 0, 1}, sp, ld, smap, st);
    return launch_syn<2, false>(name, cf, (int)nside, (int)L, tab, (int)(2 * nside), nblk, nullptr, tab, 1, 0, 0,
                                Low{0, 0, 1}, sp, ld, smap, st);
}

}  // namespace gm

using namespace gm;

namespace {
int check_2(const char* name, int64_t nside, int64_t lmax, int64_t jsplit, int64_t mpol) {
    if (nside < 1 || (nside & (nside - 1)) || nside > 8192) return fail(GM_E_ARG, "%s: bad nside", name);
    if (lmax < 2 || lmax > 24 * nside) return fail(GM_E_ARG, "%s: bad lmax %lld", name, (long long)lmax);
    if (jsplit < 1 || jsplit > 2 * nside) return fail(GM_E_ARG, "%s: jsplit outside [1, 2 nside]", name);
    if (mpol < 0 || mpol > lmax + 1) return fail(GM_E_ARG, "%s: mpol outside [0, lmax + 1]", name);
    return GM_OK;
}
constexpr int kSlots = 4;
}  // namespace

extern "C" int64_t gm_lat2_chunks(int64_t nside, int64_t jsplit) {
    if (nside < 1 || jsplit < 1 || jsplit > 2 * nside) return -1;
    const int CH = pair_shape(nside, 2, true, false).CH;
    return (jsplit + CH - 1) / CH;
}

extern "C" int64_t gm_lat2_slots(int64_t nside, int64_t jsplit) {
    const int64_t n = gm_lat2_chunks(nside, jsplit);
    return nside <= 4096 || n <= kSlots ? n : kSlots;
}

extern "C" int64_t gm_lat2_polar_size(int64_t nside, int64_t lmax, int64_t jsplit, int64_t mpol) {
    if (check_2("gm_lat2_polar_size", nside, lmax, jsplit, mpol)) return -1;
    const int CHP = 64 * pair_shape(nside, 2, true, false).NW * kRP;
    const Low low = low_orders(nside, jsplit, mpol, CHP);
    return 4 * (polar_blocks(nside, jsplit, CHP) * table_base(mpol, lmax + 1) + low.nb * table_base(low.n, lmax + 1));
}

extern "C" int gm_lat2_ana(const double* spec, int64_t ld, int64_t nside, int64_t lmax, int64_t jsplit, int64_t mpol,
                           const double* alpha, const double* smant, const int32_t* sexp, const int32_t* nact,
                           const double* alpha2, const double* gamma2, const double* smant2, const int32_t* sexp2,
                           const int32_t* nact2, double* part, double* ppart, int64_t chunk0, void* stream) {
    const char* name = "gm_lat2_ana";
    if (int e = check_2(name, nside, lmax, jsplit, mpol)) return e;
    if (!spec || !alpha || !smant || !sexp || !nact || !part) return fail(GM_E_ARG, "%s: null pointer", name);
    if (mpol > 0 && (!alpha2 || !gamma2 || !smant2 || !sexp2 || !nact2 || !ppart))
        return fail(GM_E_ARG, "%s: null pointer", name);
    const int64_t Lm = lmax + 1;
    if (ld < 2 * Lm - 1) return fail(GM_E_SHAPE, "%s: ld < 2 lmax + 1", name);
    const int slots = (int)gm_lat2_slots(nside, jsplit), chunks = (int)gm_lat2_chunks(nside, jsplit);
    if (chunk0 < 0 || chunk0 >= chunks || chunk0 % slots) return fail(GM_E_ARG, "%s: bad chunk0", name);
    const int nblk = (int)(chunks - chunk0 < slots ? chunks - chunk0 : slots);
    const Tables tab{alpha, nullptr, smant, sexp, nact, (int)Lm + 2};
    const Tables pol{alpha2, gamma2, smant2, sexp2, nact2, (int)Lm};
    const Shape s = pair_shape(nside, 2, true, false);
    const int CH = s.CH, CHP = 64 * s.NW * kRP, nbp = polar_blocks(nside, jsplit, CHP);
    const Low low = low_orders(nside, jsplit, mpol, CHP);
    const int npol = chunk0 == 0 ? low.n * low.nb + ((int)mpol - low.n) * nbp : 0;
    const int jbeg = (int)chunk0 * CH, jend = jbeg + nblk * CH < jsplit ? jbeg + nblk * CH : (int)jsplit;
    return launch_ana<2, true>(name, reinterpret_cast<const double2*>(spec), ld, 0, (int)nside, (int)Lm, tab, jbeg, jend,
                               nblk, part, pol, (int)(2 * jsplit - 1), nbp, npol, low, ppart,
                               table_base(mpol, Lm), (hipStream_t)stream);
}

extern "C" int gm_lat2_finish(const double* part, const double* ppart, int64_t nside, int64_t lmax, int64_t jsplit,
                              int64_t mpol, const int32_t* nact, const double* P, const int32_t* nact2, const double* P2,
                              double* alm_e, double* alm_b, int mode, int64_t chunk0, void* stream) {
    const char* name = "gm_lat2_finish";
    if (int e = check_2(name, nside, lmax, jsplit, mpol)) return e;
    if (mode < 0 || mode > 2 || chunk0 < 0) return fail(GM_E_ARG, "%s: bad mode / chunk0", name);
    if (!part || !nact || !P || !alm_e || !alm_b || (mpol > 0 && (!ppart || !nact2 || !P2)))
        return fail(GM_E_ARG, "%s: null pointer", name);
    const int Lm = (int)lmax + 1;
    const Shape s = pair_shape(nside, 2, true, false);
    const int T = 64 * s.NW, CHP = T * kRP;
    const int64_t end = (chunk0 + gm_lat2_slots(nside, jsplit)) * s.CH;
    hipLaunchKernelGGL(k_finish_2, dim3((Lm + kFin - 1) / kFin, Lm), dim3(kFin), 0, (hipStream_t)stream, part, ppart, T, s.R,
                       (int)chunk0 * s.CH, (int)(end < jsplit ? end : jsplit), (int)jsplit, nact, P,
                       polar_blocks(nside, jsplit, CHP), CHP, (int)mpol, low_orders(nside, jsplit, mpol, CHP), nact2, P2, Lm,
                       table_base(mpol, Lm),
                       reinterpret_cast<double2*>(alm_e), reinterpret_cast<double2*>(alm_b), mode);
    return check_launch(name);
}

extern "C" int gm_lat2_prep(const double* alm_e, const double* alm_b, const double* P, const double* P2, int64_t lmax,
                            int64_t mpol, double* coef, double* pcoef, void* stream) {
    const char* name = "gm_lat2_prep";
    if (int e = check_2(name, 8192, lmax, 1, mpol)) return e;
    if (!alm_e || !alm_b || !P || !coef || (mpol > 0 && (!P2 || !pcoef))) return fail(GM_E_ARG, "%s: null pointer", name);
    const int Lm = (int)lmax + 1;
    hipLaunchKernelGGL(k_prep_2, dim3((Lm + 2 + GM_TABLE_PAD + kFin - 1) / kFin, Lm), dim3(kFin), 0, (hipStream_t)stream,
                       reinterpret_cast<const double2*>(alm_e), reinterpret_cast<const double2*>(alm_b), P, P2, Lm,
                       (int)mpol, reinterpret_cast<double2*>(coef), reinterpret_cast<double2*>(pcoef));
    return check_launch(name);
}

extern "C" int gm_lat2_syn(const double* coef, const double* pcoef, int64_t nside, int64_t lmax, int64_t jsplit,
                           int64_t mpol, const double* alpha, const double* smant, const int32_t* sexp,
                           const int32_t* nact, const double* alpha2, const double* gamma2, const double* smant2,
                           const int32_t* sexp2, const int32_t* nact2, double* spec, int64_t ld, void* stream) {
    const char* name = "gm_lat2_syn";
    if (int e = check_2(name, nside, lmax, jsplit, mpol)) return e;
    if (!coef || !alpha || !smant || !sexp || !nact || !spec) return fail(GM_E_ARG, "%s: null pointer", name);
    if (mpol > 0 && (!pcoef || !alpha2 || !gamma2 || !smant2 || !sexp2 || !nact2))
        return fail(GM_E_ARG, "%s: null pointer", name);
    const int64_t Lm = lmax + 1;
    if (ld < 2 * Lm - 1) return fail(GM_E_SHAPE, "%s: ld < 2 lmax + 1", name);
    const Tables tab{alpha, nullptr, smant, sexp, nact, (int)Lm + 2};
    const Tables pol{alpha2, gamma2, smant2, sexp2, nact2, (int)Lm};
    const Shape s = pair_shape(nside, 2, true, true);
    const int CH = s.CH, chp = 64 * s.NW * kRP;
    const int nblk = (int)((jsplit + CH - 1) / CH), nbp = polar_blocks(nside, jsplit, chp);
    const Low low = low_orders(nside, jsplit, mpol, chp);
    const int npol = low.n * low.nb + ((int)mpol - low.n) * nbp;
    return launch_syn<2, true>(name, reinterpret_cast<const double2*>(coef), (int)nside, (int)Lm, tab, (int)jsplit, nblk,
                               reinterpret_cast<const double2*>(pcoef), pol, nbp, npol, (int)((Lm - mpol) * nbp), low,
                               reinterpret_cast<double2*>(spec), ld, 0, (hipStream_t)stream);
}
