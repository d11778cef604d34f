"""Rounding error of the ring-pair FFTs against scipy's long-double FFT: no more than that of the
single-ring transforms of the same rings.

Bound: a transform's rms error is the sum in quadrature of its passes' roundings and of its twiddles';
both kinds of transform run 3 to 6 passes of a rounded butterfly and a twiddle of a few roundings, so
they agree to a quarter (twiddles as powers of one rounded base carry up to 15 times its
rounding: 1.5 to 1.9 times the belt's error)."""

import numpy as np
import pytest
import scipy.fft
import torch

from oracle.geometry import Rings

pytestmark = pytest.mark.gpu
LD = np.longdouble


def _phase(m, R, r):
    a = 4 * np.arctan(LD(1)) * ((m * int(R.phi0_num[r])) % (2 * int(R.phi0_den[r]))).astype(LD) / LD(int(R.phi0_den[r]))
    return np.cos(a) - 1j * np.sin(a)


@pytest.mark.parametrize("nside", [64, 256, 1024, 2048])
def test_ring_pairs_round_no_more_than_single_rings(nside):
    from gmaster_amd import _lib

    lmax = 2 * nside
    print(f"ring pair error nside={nside}", flush=True)
    R = Rings(nside)
    L, W, npix, nring = lmax + 1, 2 * lmax + 1, 12 * nside * nside, 4 * nside - 1
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(nside)
    maps = torch.randn((2, npix), dtype=torch.float64, device="cuda", generator=g)
    src = torch.randn((nring, L), dtype=torch.complex128, device="cuda", generator=g)
    src[:, 0].imag = 0.0
    src2 = torch.randn((nring, W), dtype=torch.complex128, device="cuda", generator=g)
    out = {}
    for kind in ("fft", "pair"):
        s = torch.empty((nring, L), dtype=torch.complex128, device="cuda")
        s2 = torch.empty((nring, W), dtype=torch.complex128, device="cuda")
        b, b2 = torch.empty(npix, dtype=torch.float64, device="cuda"), torch.empty_like(maps)
        _lib.call(f"gm_ring_{kind}_fwd_s0", _lib.ptr(maps), 1, npix, nside, lmax, _lib.ptr(s), L, nring * L, st)
        _lib.call(f"gm_ring_{kind}_fwd_s", _lib.ptr(maps[0]), _lib.ptr(maps[1]), nside, lmax, _lib.ptr(s2), W, st)
        _lib.call(f"gm_ring_{kind}_inv_s0", _lib.ptr(src), 1, L, nring * L, nside, lmax, _lib.ptr(b), npix, st)
        _lib.call(f"gm_ring_{kind}_inv_s", _lib.ptr(src2), W, nside, lmax, _lib.ptr(b2[0]), _lib.ptr(b2[1]), st)
        b2 = b2.cpu().numpy()
        out[kind] = (s.cpu().numpy(), s2.cpu().numpy(), b.cpu().numpy(), b2[0] + 1j * b2[1])
    hm, hs, hs2 = maps.cpu().numpy(), src.cpu().numpy(), src2.cpu().numpy()
    m, mc = np.arange(L), np.arange(-lmax, L)
    weight = 16 * np.arctan(LD(1)) / npix
    rng = np.random.default_rng(nside)
    belt = np.concatenate([[nside, nside + 1, 2 * nside], rng.integers(nside, 2 * nside, 12)])
    for what, rings in (("belt", belt), ("caps", rng.integers(1, nside, 15))):
        err = {k: np.zeros(4) for k in out}
        for q in rings:
            for r in {int(q) - 1, nring - int(q)}:
                n, at = int(R.nphi[r]), slice(int(R.offset[r]), int(R.offset[r]) + int(R.nphi[r]))
                z = hm[:, at].astype(LD)
                Y, Y2 = np.zeros(n, dtype=np.clongdouble), np.zeros(n, dtype=np.clongdouble)
                F = hs[r] * np.conj(_phase(m, R, r))
                np.add.at(Y, m % n, F)
                np.add.at(Y, (-m[1:]) % n, np.conj(F[1:]))
                np.add.at(Y2, mc % n, hs2[r] * np.conj(_phase(mc, R, r)))
                exact = (weight * scipy.fft.fft(z[0].astype(np.clongdouble))[m % n] * _phase(m, R, r),
                         weight * scipy.fft.fft(z[0] + 1j * z[1])[mc % n] * _phase(mc, R, r),
                         (n * scipy.fft.ifft(Y)).real, n * scipy.fft.ifft(Y2))
                for k, o in out.items():
                    for i, (x, e) in enumerate(zip((o[0][r], o[1][r], o[2][at], o[3][at]), exact)):
                        err[k][i] += float(np.mean(np.abs(x - e) ** 2) / np.mean(np.abs(e) ** 2))
        ratio = np.sqrt(err["pair"] / err["fft"])
        print(f"  {what}: fwd_s0 fwd_s inv_s0 inv_s", np.round(ratio, 2), flush=True)
        assert ratio.max() < 1.25, (what, ratio)
