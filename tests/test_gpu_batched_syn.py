"""Batched synthesis where FP32 and polar FP64 ring pairs share a launch (Nside <= 1024, up to two
maps and a field, four maps or two fields) and where they do not (eight maps), against the FP64
transforms.  Tolerance: FP32 operands and sums of at most 3 Nside terms outside sin^2 = 1/16, 16 times
2^-24 per rounding, 2^-20 sqrt(3 Nside) of the largest value."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k0,k2", [(1, 1), (2, 1), (0, 1), (0, 2), (2, 0), (4, 0), (8, 0)])
@pytest.mark.parametrize("nside,lmax", [(1, 2), (4, 11), (32, 64), (128, 300)])
def test_batched_synthesis_small(nside, lmax, k0, k2):
    from gmaster_amd import batched, sht

    print(f"batched synthesis nside={nside} lmax={lmax} k0={k0} k2={k2}", flush=True)
    L = lmax + 1
    ne = L * (L + 1) // 2
    g = torch.Generator("cuda").manual_seed(10 * nside + k0)
    a = torch.randn((k0 + 2 * k2, ne), dtype=torch.complex128, device="cuda", generator=g)
    a[:, :L] = a[:, :L].real.to(torch.complex128)  # m = 0
    ell = torch.cat([torch.arange(m, L) for m in range(L)]).cuda()
    a[k0:, ell < 2] = 0
    a0 = a[:k0].contiguous() if k0 else None
    a2 = a[k0:].reshape(k2, 2, ne).contiguous() if k2 else None
    m0, m2 = batched.alm2map(a0, a2, nside, lmax)
    tol = 2.0 ** -20 * np.sqrt(3.0 * nside + 3)
    for k in range(k0):
        ref = sht.alm2map_s0(a0[k:k + 1], nside, lmax)[0]
        assert float((m0[k] - ref).abs().max()) <= tol * float(ref.abs().max()), k
    for f in range(k2):
        ref = sht.alm2map_spin(a2[f], nside, lmax, 2)
        assert float((m2[f] - ref).abs().max()) <= tol * float(ref.abs().max()), f
