// Ring FFTs of pairs of real rings (ringpair.hip), called by the entry points in ringfft.hip.
#pragma once

#include "common.h"

namespace gm {

struct RingArgs {
    const double* a;  // maps (spin 2: Q)
    const double* b;  // spin 2: U
    int64_t mstride;
    int nmaps, nside, L;
    double2* spec;
    int64_t ld, smap;
    hipStream_t stream;
};

// Cap rings q <= kRingPairQ of both hemispheres, and the belt where 4 nside is a power of two from
// 256 to 8192 points.
constexpr int kRingPairQ = 2048;
inline bool ring_pair_belt(int64_t nside) { return nside >= 64 && nside <= 2048; }
int ring_pairs_fwd(const RingArgs& r, bool spin2);
int ring_pairs_inv(const RingArgs& r, bool spin2);

// Raises a kernel's dynamic LDS limit once per kernel and device.
int ring_set_lds(const void* fn, size_t bytes);

}  // namespace gm
