"""The ring-pair FFTs where they end: at Nside 4096 the largest cap they take (q = 2048, whose
convolution fills its 4096 points), the next ring (2049) and the largest cap (4095) that single-ring
transforms take, and the belt of 16384 pixels, which they leave too; and the belt's ends at Nside 32
and 64.  Against numpy's FFT, tolerance 1e-12 of the ring's largest value: three FFTs of at most
2^12 points carry 3 * 12 eps of the ring's rms, the single rings' direct passes over a prime p
p eps (4095 = 3 3 5 7 13, 2049 = 3 683)."""

import numpy as np
import pytest
import torch

from oracle.geometry import Rings

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _phase(m, R, r):
    return np.exp(-1j * np.pi * ((m * R.phi0_num[r]) % (2 * R.phi0_den[r])) / R.phi0_den[r])


def _close(got, ref, what):
    e = float(np.max(np.abs(got - ref)) / np.max(np.abs(ref)))
    assert e < TOL, (what, e)


@pytest.mark.parametrize("nside,caps", [(4096, (1, 2047, 2048, 2049, 4095)), (64, (63,)), (32, (31,))])
def test_ring_pair_limits(nside, caps):
    from gmaster_amd import _lib

    lmax = 500
    print(f"ring pair limits nside={nside}", flush=True)
    R = Rings(nside)
    L, W, npix, nring = lmax + 1, 2 * lmax + 1, 12 * nside * nside, 4 * nside - 1
    north = list(caps) + [nside, nside + 1, 2 * nside]
    sample = sorted({q - 1 for q in north} | {nring - q for q in north})
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(nside)
    m, mc = np.arange(L), np.arange(-lmax, L)

    maps = torch.randn((2, npix), dtype=torch.float64, device="cuda", generator=g)
    at = {r: slice(int(R.offset[r]), int(R.offset[r]) + int(R.nphi[r])) for r in sample}
    spec = torch.full((nring, L), 9.0, dtype=torch.complex128, device="cuda")
    _lib.call("gm_ring_pair_fwd_s0", _lib.ptr(maps), 1, npix, nside, lmax, _lib.ptr(spec), L, nring * L, st)
    src = torch.randn((nring, L), dtype=torch.complex128, device="cuda", generator=g)
    src[:, 0].imag = 0.0
    back = torch.full_like(maps, 9.0)
    _lib.call("gm_ring_pair_inv_s0", _lib.ptr(src), 1, L, nring * L, nside, lmax, _lib.ptr(back), npix, st)
    spec2 = torch.full((nring, W), 9.0, dtype=torch.complex128, device="cuda")
    _lib.call("gm_ring_pair_fwd_s", _lib.ptr(maps[0]), _lib.ptr(maps[1]), nside, lmax, _lib.ptr(spec2), W, st)
    src2 = torch.randn((nring, W), dtype=torch.complex128, device="cuda", generator=g)
    out = torch.full_like(maps, 9.0)
    _lib.call("gm_ring_pair_inv_s", _lib.ptr(src2), W, nside, lmax, _lib.ptr(out[0]), _lib.ptr(out[1]), st)
    for t in (spec, spec2, back[0], out):  # every ring is somebody's
        v = torch.view_as_real(t) if t.is_complex() else t
        assert not (v == 9.0).any()
    assert (back[1] == 9.0).all()
    for r in sample:
        n = int(R.nphi[r])
        z = maps[:, at[r]].cpu().numpy()
        _close(spec[r].cpu().numpy(), R.weight * np.fft.fft(z[0])[m % n] * _phase(m, R, r), ("fwd_s0", r))
        _close(spec2[r].cpu().numpy(), R.weight * np.fft.fft(z[0] + 1j * z[1])[mc % n] * _phase(mc, R, r), ("fwd_s", r))
        F = src[r].cpu().numpy() * np.conj(_phase(m, R, r))
        Y = np.zeros(n, dtype=np.complex128)
        np.add.at(Y, m % n, F)
        np.add.at(Y, (-m[1:]) % n, np.conj(F[1:]))
        _close(back[0, at[r]].cpu().numpy(), (n * np.fft.ifft(Y)).real, ("inv_s0", r))
        Y = np.zeros(n, dtype=np.complex128)
        np.add.at(Y, mc % n, src2[r].cpu().numpy() * np.conj(_phase(mc, R, r)))
        x = out[:, at[r]].cpu().numpy()
        _close(x[0] + 1j * x[1], n * np.fft.ifft(Y), ("inv_s", r))
