"""The ring FFTs of ring pairs at the edges of their size classes, against numpy's FFT: caps on
both sides of q = 128, 256, 512 and 1024, the smallest rings, the belt's smallest (256 points)
and largest (8192) power of two and its absence (Nside 32), three maps in padded rows, lmax
from far below to above 3 Nside.

Tolerance 1e-12 of the ring's largest value: three FFTs of at most 2^12 points in a Bluestein
convolution carry ~3 * 12 eps of the ring's rms (1e-14 of the largest), and the inverse adds up to
2 lmax / 4 aliases in a word of the smallest ring (2^12 eps = 5e-13)."""

import numpy as np
import pytest
import torch

from oracle.geometry import Rings

pytestmark = pytest.mark.gpu
TOL = 1e-12
EDGES = (1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047)


def _phase(m, R, r):
    return np.exp(-1j * np.pi * ((m * R.phi0_num[r]) % (2 * R.phi0_den[r])) / R.phi0_den[r])


def _close(got, ref, what):
    e = float(np.max(np.abs(got - ref)) / max(np.max(np.abs(ref)), 1e-300))
    assert e < TOL, (what, e)


def Y0_imag(F):
    """Im F[0] (zero for a real map) enters the packed half-length inverse, which every ring
    shorter or longer than the pairs' sizes takes, as minus itself at Nyquist; the pairs keep that."""
    return F[0].imag


@pytest.mark.parametrize("nside,lmax", [(1, 2), (32, 101), (64, 7), (128, 400), (512, 1535), (2048, 4100)])
def test_ring_pairs_at_class_edges(nside, lmax):
    from gmaster_amd import _lib

    print(f"ring pairs nside={nside} lmax={lmax}", flush=True)
    R = Rings(nside)
    L, W, npix, nring = lmax + 1, 2 * lmax + 1, 12 * nside * nside, 4 * nside - 1
    K, ld, ldc, ms = (3 if nside <= 512 else 1), L + 3, W + 5, npix + 7
    north = sorted({q for q in EDGES if q < nside} | {nside, nside + 1 if nside > 1 else 1, 2 * nside})
    sample = sorted({q - 1 for q in north} | {nring - q for q in north})
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(nside)
    m, mc = np.arange(L), np.arange(-lmax, L)

    maps = torch.randn((K, ms), dtype=torch.float64, device="cuda", generator=g)
    spec = torch.full((K, nring, ld), 9.0, dtype=torch.complex128, device="cuda")
    _lib.call("gm_ring_pair_fwd_s0", _lib.ptr(maps), K, ms, nside, lmax, _lib.ptr(spec), ld, spec.stride(0), st)
    src = torch.randn((K, nring, ld), dtype=torch.complex128, device="cuda", generator=g)
    back = torch.full_like(maps, 9.0)
    _lib.call("gm_ring_pair_inv_s0", _lib.ptr(src), K, ld, src.stride(0), nside, lmax, _lib.ptr(back), ms, st)
    hm, hs, hb, hf = maps.cpu().numpy(), spec[:, sample].cpu().numpy(), back.cpu().numpy(), src[:, sample].cpu().numpy()
    assert (hs[:, :, L:] == 9.0).all() and (hb[:, npix:] == 9.0).all()  # padding untouched
    for k in range(K):
        for i, r in enumerate(sample):
            n, o = int(R.nphi[r]), int(R.offset[r])
            _close(hs[k, i, :L], R.weight * np.fft.fft(hm[k, o:o + n])[m % n] * _phase(m, R, r), ("fwd_s0", k, r))
            F = hf[k, i, :L] * np.conj(_phase(m, R, r))
            Y = np.zeros(n, dtype=np.complex128)
            np.add.at(Y, m % n, F)
            np.add.at(Y, (-m[1:]) % n, np.conj(F[1:]))
            Y[n // 2] -= Y0_imag(F)
            _close(hb[k, o:o + n], (n * np.fft.ifft(Y)).real, ("inv_s0", k, r))

    qu = torch.randn((2, npix), dtype=torch.float64, device="cuda", generator=g)
    spec = torch.full((nring, ldc), 9.0, dtype=torch.complex128, device="cuda")
    _lib.call("gm_ring_pair_fwd_s", _lib.ptr(qu[0]), _lib.ptr(qu[1]), nside, lmax, _lib.ptr(spec), ldc, st)
    src = torch.randn((nring, ldc), dtype=torch.complex128, device="cuda", generator=g)
    out = torch.empty_like(qu)
    _lib.call("gm_ring_pair_inv_s", _lib.ptr(src), ldc, nside, lmax, _lib.ptr(out[0]), _lib.ptr(out[1]), st)
    hz, ho = (t[0].cpu().numpy() + 1j * t[1].cpu().numpy() for t in (qu, out))
    hs, hf = spec[sample].cpu().numpy(), src[sample].cpu().numpy()
    assert (hs[:, W:] == 9.0).all()
    for i, r in enumerate(sample):
        n, o = int(R.nphi[r]), int(R.offset[r])
        _close(hs[i, :W], R.weight * np.fft.fft(hz[o:o + n])[mc % n] * _phase(mc, R, r), ("fwd_s", r))
        Y = np.zeros(n, dtype=np.complex128)
        np.add.at(Y, mc % n, hf[i, :W] * np.conj(_phase(mc, R, r)))
        _close(ho[o:o + n], n * np.fft.ifft(Y), ("inv_s", r))
