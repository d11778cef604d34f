// The row sums of the mode-coupling matrix for one pair l1 <= l2, walked in l3 without square
// roots (host and device).
//
// f0 = (l1 l2 l3; 0 0 0) obeys Q(l3+1) f0(l3+1) = -Q(l3) f0(l3-1) with
//     Q(l3)^2 = q(l3) = (l3^2 - d^2) ((l1+l2+1)^2 - l3^2),   d = l2 - l1,
// from the closed form at l3 = d, so f0^2 at even J = l1 + l2 + l3 (l3 = d, d + 2, ...) is R / P
// with R the product of q over the odd degrees passed and P over the even ones.
//
// f2 = (l1 l2 l3; 2 -2 0) needs no recursion of its own.  The m recursion of 3j symbols
// (Schulten & Gordon 1975), (L1 + L2 - 2 m^2 - X) f_m + C(m+1) f_{m+1} + C(m) f_{m-1} = 0 with
// X = l3 (l3+1), L = l (l+1) and f_{-1} = f_1 at even J, gives there, with E = X - L1 - L2 + 1,
//     f2 = f0 (E^2 - K) / (2 N),   K = 1 + 2 L1 L2,   N^2 = L1 L2 (l1-1)(l1+2)(l2-1)(l2+2),
// and the l3 recursion Q(l3+1) f2(l3+1) = 4 (2 l3 + 1) f2(l3) - Q(l3) f2(l3-1), solved for the
// odd degree between two even ones, gives f2(l3+1)^2 = f0(l3)^2 q(l3+1) (E + E')^2 / (16 N^2),
// E' being E at l3 + 2.  (E is an exact integer; E^2 - K is one fused operation, K exact up to l ~ 8192
// and rounded beyond, which leaves f2 an error of 2^-53 f0.  The recursion of f2 in l3 was 29 FP64
// operations per two degrees for everything, this is 22.)
//
// q(l3) = k (2 l1 + 1 - k) Y with k = l3 - d, Y = (2d + k)(2d + k + 2 l1 + 1): the first factor is
// the same for every l2 of a row, Y steps by exact integer differences.  The sums sum W'_l3 f^2
// are accumulated in Horner form, G <- G q(l3) + W' R (...), and divided by P once at the end.
// P grows by at most S^4 / 4 < 2^66 per two degrees (S = l1 + l2 + 1 < 2^17); every 8 pairs of
// degrees all are rescaled by a power of two (exact), so nothing leaves the FP64 range.
#pragma once

#include <hip/hip_runtime.h>

namespace gm {

struct CoupleRun {
    double R, P;              // f0^2 = R / P at the current even degree
    double G00, G02, GE, GO;  // Horner sums (scale P): 0-0, 0-2, 2-2 even J, 2-2 odd J, without 2 N, (2 N)^2, (4 N)^2
    double Y, y1;             // Y at the next degree, its step
    double E, sx, p2;         // E at the even degree, its step, E^2 - K
    double me;                // P ratio of the last even step
    double K, n2;             // n2 = N^2 (0 where f2 is not defined, l1 < 2)

    // g[p] = Gamma(p + 1/2) / (sqrt(pi) Gamma(p + 1)), p <= l2.
    __host__ __device__ void init(const double* __restrict__ g, int l1, int l2) {
        const int d = l2 - l1;
        const double a = l1, b = l2, n = 2.0 * a + 1.0, v = 2.0 * d + 1.0;
        const double L1 = a * (a + 1.0), L2 = b * (b + 1.0);
        R = g[l1] * g[d] / ((2.0 * b + 1.0) * g[l2]);
        P = 1.0;
        G00 = G02 = GE = GO = 0.0;
        Y = v * (v + n);
        y1 = 2.0 * v + 1.0 + n;
        E = (double)d * (d + 1.0) - L1 - L2 + 1.0;
        sx = 4.0 * d + 6.0;
        K = fma(2.0 * L1, L2, 1.0);
        p2 = fma(E, E, -K);
        me = 1.0;
        n2 = l1 >= 2 ? (L1 * (L1 - 2.0)) * (L2 * (L2 - 2.0)) : 0.0;  // (l - 1)(l + 2) = l (l + 1) - 2
    }

    // Terms of an even degree.
    __host__ __device__ __forceinline__ void even_term(double we) {
        const double t = we * R, t2 = t * p2;
        G00 = fma(G00, me, t);
        G02 = fma(G02, me, t2);
        GE = fma(GE, me, t2 * p2);
    }

    // Terms of the even degree l3 = d + k (weight we) and of l3 + 1 (weight wo);
    // ko = (k + 1) (2 l1 - k).  Past the last degree (on false, zero weights) R stays.
    __host__ __device__ __forceinline__ void half_a(double we, double wo, double ko, bool on = true) {
        even_term(we);
        R *= on ? ko * Y : 1.0;
        Y += y1;
        y1 += 2.0;
        const double En = E + sx, h = E + En;
        E = En;
        sx += 8.0;
        GO = fma(GO, me, (wo * R * h) * h);
    }

    // Step to the next even degree, ke = (k + 2) (2 l1 - 1 - k); past the last degree (on false)
    // the sums keep their scale.
    __host__ __device__ __forceinline__ void half_b(double ke, bool on = true) {
        me = on ? ke * Y : 1.0;
        Y += y1;
        y1 += 2.0;
        P *= me;
        p2 = fma(E, E, -K);
    }

    // Exact power-of-two rescale bringing P into [1/2, 1).
    __host__ __device__ __forceinline__ void rescale() {
        int e;
        (void)frexp(P, &e);
        R = ldexp(R, -e);
        P = ldexp(P, -e);
        G00 = ldexp(G00, -e);
        G02 = ldexp(G02, -e);
        GE = ldexp(GE, -e);
        GO = ldexp(GO, -e);
    }

    // Row sums (a00, a02, aE, aO).  ended_even: the last degree was even, so the odd sum is one
    // even step behind.  A quotient each, by the product of exact or once rounded factors: with 1 / P
    // and 1 / N multiplied on, their rounding counts twice in the squares (rms error of the l3 = 0 and
    // 1 terms of l1 = l2 up to 2100: 1.3 and 1.5 units of 2^-53, now 1.0 and 1.1).
    __host__ __device__ void finish(bool ended_even, double s[4]) const {
        const double odd = ended_even ? GO * me : GO, p4 = 4.0 * P * n2;
        s[0] = G00 / P;
        s[1] = n2 > 0.0 ? G02 / (2.0 * P * sqrt(n2)) : G02 * 0.0;
        s[2] = n2 > 0.0 ? GE / p4 : GE * 0.0;
        s[3] = n2 > 0.0 ? odd / (4.0 * p4) : odd * 0.0;
    }
};

// The factor k (2 l1 + 1 - k) of q.
__host__ __device__ __forceinline__ double couple_kappa(int k, int l1) { return (double)k * (double)(2 * l1 + 1 - k); }

// A window that stages the factors k0 + 1 .. k0 + 64 with the weights returns them by kappa(t);
// any other has them computed.
template <class Win>
__host__ __device__ __forceinline__ auto couple_kappa_at(const Win& w, int t, int, int) -> decltype(w.kappa(t)) {
    return w.kappa(t);
}
template <class Win>
__host__ __device__ __forceinline__ double couple_kappa_at(const Win&, int, long k, int l1) {
    return couple_kappa((int)k, l1);
}

// Degrees l3 = d .. min(l1 + l2, lmax_w) of one pair, W' read from Wp; s = (a00, a02, aE, aO).
__host__ __device__ inline void couple_pair(const double* __restrict__ Wp, int lmax_w, const double* __restrict__ g,
                                            int l1, int l2, double s[4]) {
    const int d = l2 - l1;
    const int n = min(l1 + l2, lmax_w) - d + 1;  // degrees with a term
    if (n <= 0) {
        s[0] = s[1] = s[2] = s[3] = 0.0;
        return;
    }
    CoupleRun r;
    r.init(g, l1, l2);
    const int np = n >> 1;
    const bool odd = n & 1;
    const int nfull = odd ? np : np - 1;
    int l3 = d;
    for (int j = 0; j < nfull; ++j) {
        r.half_a(Wp[l3], Wp[l3 + 1], couple_kappa(2 * j + 1, l1));
        r.half_b(couple_kappa(2 * j + 2, l1));
        l3 += 2;
        if ((j & 7) == 7) r.rescale();
    }
    if (odd)
        r.even_term(Wp[l3]);
    else
        r.half_a(Wp[l3], Wp[l3 + 1], couple_kappa(2 * nfull + 1, l1));
    r.finish(odd, s);
}

// ---------------------------------------------------------------- full matrix, one l1 per wave
// Work items are (l1, chunk j): the wave takes l2 = l1 + 64 j + lane.  Items run in
// descending l1 (longest rows first): rows l1 in [L - 64 (t+1), L - 64 t - 1] have t + 1
// chunks each, so 32 t (t + 1) items precede group t and row-major order inside it follows.
__host__ __device__ inline int64_t couple_items(int L) {
    int64_t n = 0;
    for (int t = 0; 64 * t < L; ++t) n += (int64_t)min(64, L - 64 * t) * (t + 1);
    return n;
}

__host__ __device__ inline void couple_decode(int64_t item, int L, int& l1, int& j) {
    int t = (int)((sqrt(1.0 + (double)item / 8.0) - 1.0) * 0.5);
    while (32LL * (t + 1) * (t + 2) <= item) ++t;
    while (t > 0 && 32LL * t * (t + 1) > item) --t;
    const int64_t r = item - 32LL * t * (t + 1);
    l1 = L - 1 - 64 * t - (int)(r / (t + 1));
    j = (int)(r % (t + 1));
}

// One lane of a wave's item: row l1, columns l2 = l2_0 + lane (l2_0 >= l1).  All lanes run
// the degree count of lane 0 (the smallest d, so the longest row): a lane with fewer
// degrees in the window reads zeros past lmax_w (the window is zero-padded) and leaves its sums
// unscaled from there, and every lane stays inside its triangle (l3 <= l1 + l2).  Win supplies W' per lane: stage(k0) loads
// W'[d0 + k0 + t], t < 128, d0 = l2_0 - l1 (zero past lmax_w), and at(t) returns entry t;
// lane i at degree l3 = d0 + i + k reads entry i + k - k0, with k0 = 64 floor(k / 64).
// Lanes with l2 >= L run the row of l2 = L - 1; the caller stores only the lanes it owns.
template <class Win>
__host__ __device__ inline void couple_wave_lane(Win& win, int lmax_w, const double* __restrict__ g, int L, int l1,
                                                 int l2_0, int lane, double s[4]) {
    const int d0 = l2_0 - l1;
    const int n = min(l1 + l2_0, lmax_w) - d0 + 1;  // lane 0's degrees (all lanes run these)
    const int l2 = min(l2_0 + lane, L - 1);
    if (n <= 0) {
        s[0] = s[1] = s[2] = s[3] = 0.0;
        return;
    }
    CoupleRun r;
    r.init(g, l1, l2);
    const int np = n >> 1;
    const bool odd = n & 1;
    const int nfull = odd ? np : np - 1;
    win.stage(0);
    int p = 0;  // pair index: degrees d + 2p, d + 2p + 1
    auto kappa = [&](int q, int u) { return couple_kappa_at(win, 2 * (q & 31) + u - 1, 2 * q + u, l1); };
    auto pair = [&](int q, int last) {  // last: pairs after which the lane has ended
        const int o = lane + 2 * (q & 31);
        r.half_a(win.at(o), win.at(o + 1), kappa(q, 1), q <= last);
        r.half_b(kappa(q, 2), q < last);
    };
    // full pairs of this lane, and of the lane with the fewest (all equal unless the window ends)
    const int nl = min(l1 + l2, lmax_w) - (l2 - l1) + 1, mine = nl > 0 ? (nl - 1) >> 1 : 0;
    const int n63 = min(l1 + l2_0 + 63, lmax_w) - (d0 + 63) + 1;
    const int all = min(n63 > 0 ? (n63 - 1) >> 1 : 0, nfull);
    for (; p + 8 <= all; p += 8) {
        if (p && (p & 31) == 0) win.stage(2 * p);
#pragma unroll
        for (int u = 0; u < 8; ++u) pair(p + u, p + 8);
        r.rescale();
    }
    for (; p + 8 <= nfull; p += 8) {
        if (p && (p & 31) == 0) win.stage(2 * p);
#pragma unroll
        for (int u = 0; u < 8; ++u) pair(p + u, mine);
        r.rescale();
    }
    for (; p < nfull; ++p) {
        if (p && (p & 31) == 0) win.stage(2 * p);
        pair(p, mine);
    }
    if (p && (p & 31) == 0) win.stage(2 * p);
    const int o = lane + 2 * (p & 31);
    if (odd)
        r.even_term(win.at(o));
    else
        r.half_a(win.at(o), win.at(o + 1), kappa(p, 1), p <= mine);
    r.finish(odd, s);
}

}  // namespace gm
