"""The FP64 transforms that run on ring pairs, at the launch shapes and pass counts of large
geometries, against the C oracle on a sample of orders: spin 2 on spin-0 rows (its low orders, both
sides of the orders that reach the polar rings, the highest) up to Nside 4096, and the analyses of
both spins at Nside 8192, where the passes' finishes store, add or subtract and only the first one
sees the polar sums.

Tolerances are those of the same geometries' tests of the kernels on single rings: 1e-10 of an
order's largest alm, 1e-9 of its largest ring value (the recurrence's own conditioning, measured
4.4e-10 at Nside 4096)."""

import os
import subprocess

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def cb():
    subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle", "c")], check=True)
    from oracle.c import cpu_baseline

    return cpu_baseline


@pytest.fixture(autouse=True)
def _free_plans():
    yield
    from gmaster_amd import sht

    sht.clear_plans()
    torch.cuda.empty_cache()


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _start(lmax, m):
    return m * (2 * lmax + 1 - m) // 2


def _orders(p):
    """Orders 0 and 7 (the last low one), 8, both sides of mpol, the middle and the last."""
    L = p.lmax + 1
    return np.unique(np.array([0, 7, 8, p.mpol - 1, min(p.mpol, L - 1), L // 2, L - 1]))


def _noise_spectrum(nring, width, nside, seed):
    """Ring spectra as those of a white map: of variance ~ pixels of the ring."""
    g = torch.Generator("cuda").manual_seed(seed)
    out = torch.empty((nring, width), dtype=torch.complex128, device="cuda")
    torch.view_as_real(out).normal_(0.0, 1.0 / nside, generator=g)
    i = torch.arange(1, 4 * nside, device="cuda")
    q = torch.minimum(torch.minimum(i, 4 * nside - i), torch.full_like(i, nside))
    return out.mul_(torch.sqrt(q / nside)[:, None])


def _eb(cb, nside, lmax, spec, orders):
    """E, B of the sampled orders, (2, orders, L)."""
    L = lmax + 1
    ell = np.arange(L)
    dcol = spec[:, torch.as_tensor(L - 1 + orders, device="cuda")].T.cpu().numpy()
    mcol = spec[:, torch.as_tensor(L - 1 - orders, device="cuda")].T.cpu().numpy()
    out = cb.lat_ana_s_cols(nside, lmax, 2, dcol, mcol, orders)
    eb = np.zeros((2, len(orders), L), dtype=np.complex128)
    for n, m in enumerate(orders):
        plus = out[n, :, 0] + 1j * out[n, :, 1]
        minus = (-1.0) ** m * np.conj((-1.0) ** ell * (out[n, :, 2] + 1j * out[n, :, 3])) if m else np.conj(plus)
        eb[0, n], eb[1, n] = -(plus + minus) / 2, 0.5j * (plus - minus)
        eb[:, n, :max(2, m)] = 0
    return eb


def _check_eb(alm, ref, lmax, orders, sign=1.0, base=None):
    for n, m in enumerate(orders):
        at = torch.arange(_start(lmax, m) + m, _start(lmax, m) + lmax + 1, device="cuda")
        for c in range(2):
            got = alm[c, at].cpu().numpy()
            if base is not None:
                got = got - base[c, at].cpu().numpy()
            e = _rel(sign * got, ref[c, n, m:])
            assert e < 1e-10, (c, m, e)


@pytest.mark.parametrize("nside,lmax", [(256, 767), (1024, 3071), (2048, 4097), (4096, 12287)])
def test_spin2_analysis(cb, nside, lmax):
    from gmaster_amd import sht

    print(f"spin-2 analysis on pairs nside={nside} lmax={lmax}", flush=True)
    L, nring = lmax + 1, 4 * nside - 1
    p = sht.plan2(nside, lmax, "cuda")
    assert p.nchunks == p.nslots
    spec = _noise_spectrum(nring, 2 * L - 1, nside, nside)
    alm = torch.empty((2, L * (L + 1) // 2), dtype=torch.complex128, device="cuda")
    sht._analysis_2(p, spec, alm[0], alm[1], 0)
    orders = _orders(p)
    _check_eb(alm, _eb(cb, nside, lmax, spec, orders), lmax, orders)


@pytest.mark.parametrize("nside,lmax", [(512, 1535), (1024, 3071), (4096, 12287)])
def test_spin2_synthesis(cb, nside, lmax):
    from gmaster_amd import sht

    print(f"spin-2 synthesis on pairs nside={nside} lmax={lmax}", flush=True)
    L, nring = lmax + 1, 4 * nside - 1
    g = torch.Generator("cuda").manual_seed(nside + 9)
    eb = torch.randn((2, L * (L + 1) // 2), dtype=torch.complex128, device="cuda", generator=g)
    eb[:, :L] = eb[:, :L].real.to(torch.complex128)
    p = sht.plan2(nside, lmax, "cuda")
    spec = torch.empty((nring, 2 * L - 1), dtype=torch.complex128, device="cuda")
    sht._synthesis_2(p, eb[0], eb[1], spec)
    orders = _orders(p)
    no = len(orders)
    got = spec[:, torch.as_tensor(np.concatenate([L - 1 + orders, L - 1 - orders]), device="cuda")].cpu().numpy()
    del spec
    E, B = np.zeros((2, no, L), dtype=np.complex128)
    for n, m in enumerate(orders):
        at = slice(_start(lmax, m) + m, _start(lmax, m) + L)
        E[n, m:], B[n, m:] = eb[0, at].cpu().numpy(), eb[1, at].cpu().numpy()
        E[n, :max(m, 2)] = B[n, :max(m, 2)] = 0
    ell = np.arange(L)
    cd = -(E + 1j * B)
    cm = -((-1.0) ** orders)[:, None] * (-1.0) ** ell * (np.conj(E) + 1j * np.conj(B))
    out = cb.lat_syn_s(nside, lmax, 2, cd, cm, orders, extended=True)
    for n, m in enumerate(orders):
        scale = np.max(np.abs(out[n]))
        e = float(np.max(np.abs(got[:, n] - (out[n, :, 0] + 1j * out[n, :, 1])))) / scale
        assert e < 1e-9, ("direct", m, e)
        if m:
            e = float(np.max(np.abs(got[:, no + n] - (out[n, :, 2] + 1j * out[n, :, 3])))) / scale
            assert e < 1e-9, ("mirror", m, e)


def test_spin2_analysis_passes_nside8192(cb):
    from gmaster_amd import sht

    nside, lmax = 8192, 9000
    print(f"spin-2 analysis passes nside={nside} lmax={lmax}", flush=True)
    L, nring = lmax + 1, 4 * nside - 1
    # every ring: the oracle has no polar skip, whose tail is 4e-10 of an alm at this lmax
    p = sht.plan2(nside, lmax, "cuda", polar_skip=False)
    assert p.nchunks > p.nslots
    spec = _noise_spectrum(nring, 2 * L - 1, nside, 3)
    orders = _orders(p)
    ref = _eb(cb, nside, lmax, spec, orders)
    alm = torch.empty((2, L * (L + 1) // 2), dtype=torch.complex128, device="cuda")
    sht._analysis_2(p, spec, alm[0], alm[1], 0)
    _check_eb(alm, ref, lmax, orders)
    g = torch.Generator("cuda").manual_seed(4)
    base = torch.randn(alm.shape, dtype=torch.complex128, device="cuda", generator=g) * alm.abs().max() * 0.1
    alm = base.clone()
    sht._analysis_2(p, spec, alm[0], alm[1], 1)  # alm -= analysis, pass by pass
    _check_eb(alm, ref, lmax, orders, -1.0, base)


def test_spin0_analysis_passes_nside8192(cb):
    from gmaster_amd import sht

    nside, lmax = 8192, 9000
    print(f"spin-0 analysis passes nside={nside} lmax={lmax}", flush=True)
    L, nring = lmax + 1, 4 * nside - 1
    p = sht.plan(nside, lmax, 0, "cuda", polar_skip=False)
    assert len(sht._passes(p, 0, False, 2, p.nchunks, 0)) > 1
    spec = torch.stack([_noise_spectrum(nring, L, nside, k) for k in (5, 6)])
    alm = torch.empty((2, L * (L + 1) // 2), dtype=torch.complex128, device="cuda")
    sht._analysis_s0(p, spec, alm, 0)
    again = alm.clone()
    sht._analysis_s0(p, spec, again, 1)
    assert float(again.abs().max()) == 0.0 or float(again.abs().max() / alm.abs().max()) < 1e-14
    orders = np.array([0, 8, 4097, L // 2, L - 1])
    for k in range(2):
        dcol = spec[k][:, torch.as_tensor(orders, device="cuda")].T.cpu().numpy()
        out = cb.lat_ana_s_cols(nside, lmax, 0, dcol, np.zeros_like(dcol), orders)
        for n, m in enumerate(orders):
            at = torch.arange(_start(lmax, m) + m, _start(lmax, m) + L, device="cuda")
            e = _rel(alm[k, at].cpu().numpy(), out[n, m:, 0] + 1j * out[n, m:, 1])
            assert e < 1e-10, (k, m, e)
