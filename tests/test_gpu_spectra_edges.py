"""gm_coupled_cell and gm_bin_block at the edges of their unrolled steps: lmax on both sides of
8, 32 and 256 orders for one and two components, and bins of 1 to 9 degrees.  Tolerance: n + 4
roundings of the largest term for a sum of n terms."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.mark.parametrize("lmax", [0, 1, 6, 7, 8, 31, 32, 33, 255, 256, 300])
def test_coupled_cell_edges(lmax):
    from gmaster_amd import _lib

    L = lmax + 1
    ne = L * (L + 1) // 2
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(lmax)
    a = torch.randn((2, ne + 3), dtype=torch.complex128, device="cuda", generator=g)
    b = torch.randn((2, ne + 3), dtype=torch.complex128, device="cuda", generator=g)
    ha, hb = a.cpu().numpy(), b.cpu().numpy()
    for n1 in (1, 2):
        for n2 in (1, 2):
            cl = torch.empty((n1 * n2, L), dtype=torch.float64, device="cuda")
            work = torch.empty(_lib.query("gm_cl_work_size", lmax, n1 * n2), dtype=torch.float64, device="cuda")
            _lib.call("gm_coupled_cell", _lib.ptr(a), n1, _lib.ptr(b), n2, ne + 3, lmax, _lib.ptr(cl), _lib.ptr(work), st)
            got = cl.cpu().numpy()
            for l in range(L):
                m = np.arange(l + 1)
                at = m * (2 * L - 1 - m) // 2 + l
                t = np.where(m > 0, 2.0, 1.0)[None, None] * (ha[:n1, None, at] * np.conj(hb[None, :n2, at])).real
                ref = t.sum(-1).reshape(-1) / (2 * l + 1)
                assert np.abs(got[:, l] - ref).max() <= (l + 5) * 2 * EPS * np.abs(t).max(), (n1, n2, l)


@pytest.mark.parametrize("nlb", [1, 3, 4, 5, 8, 9])
def test_bin_block_edges(nlb):
    from gmaster_amd import _lib

    L = 61
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(nlb)
    M = torch.randn((L, L), dtype=torch.float64, device="cuda", generator=g)
    start = list(range(0, L - 1, nlb)) + [L - 1]
    ells = torch.arange(1, L, dtype=torch.int32, device="cuda")  # the last bin is short
    bs = torch.tensor(start, dtype=torch.int32, device="cuda")
    wo, ti = (torch.rand(L - 1, dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    nb = len(start) - 1
    out = torch.empty((nb, nb), dtype=torch.float64, device="cuda")
    _lib.call("gm_bin_block", _lib.ptr(M), L - 1, _lib.ptr(ells), _lib.ptr(bs), nb, _lib.ptr(wo), _lib.ptr(ti), _lib.ptr(out), st)
    t = wo[:, None] * M[1:, 1:] * ti[None, :]
    sel = torch.zeros((nb, L - 1), dtype=torch.float64, device="cuda")
    for i in range(nb):
        sel[i, start[i]:start[i + 1]] = 1.0
    ref = sel @ t @ sel.T
    assert float((out - ref).abs().max()) <= (nlb * nlb + 4) * 2 * EPS * float(t.abs().max())


@pytest.mark.parametrize("ncls,nslots", [(1, 1), (4, 8), (7, 11)])
def test_bin_blocks_fill_their_slots(ncls, nslots):
    """gm_bin_blocks against gm_bin_block block by block: every slot, its sign, and nothing else."""
    import ctypes

    from gmaster_amd import _lib

    L, nlb = 70, 3
    st = _lib.stream_ptr("cuda")
    g = torch.Generator("cuda").manual_seed(ncls)
    nblk = min(9, nslots)
    Ms = [torch.randn((L, L), dtype=torch.float64, device="cuda", generator=g) for _ in range(nblk)]
    start = list(range(0, L - 1, nlb)) + [L - 1]
    ells = torch.arange(1, L, dtype=torch.int32, device="cuda")
    bs = torch.tensor(start, dtype=torch.int32, device="cuda")
    wo, ti = (torch.rand(L - 1, dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    nb = len(start) - 1
    at = [(k // ncls, (3 * k) % ncls) if ncls > 1 else (0, 0) for k in range(nslots)]
    assert len(set(at)) == nslots
    slots = [(k % nblk, c1, c2, -1 if k % 3 == 2 else 1) for k, (c1, c2) in enumerate(at)]
    ref = torch.full((nb, ncls, nb, ncls), 5.0, dtype=torch.float64, device="cuda")
    out = ref.clone()
    one = torch.empty((nb, nb), dtype=torch.float64, device="cuda")
    for k, c1, c2, sign in slots:
        _lib.call("gm_bin_block", _lib.ptr(Ms[k]), L - 1, _lib.ptr(ells), _lib.ptr(bs), nb, _lib.ptr(wo), _lib.ptr(ti),
                  _lib.ptr(one), st)
        ref[:, c1, :, c2] = sign * one
    ptrs = (ctypes.c_void_p * nblk)(*[m.data_ptr() for m in Ms])
    flat = (ctypes.c_int32 * (4 * nslots))(*[v for s in slots for v in s])
    _lib.call("gm_bin_blocks", ctypes.cast(ptrs, ctypes.c_void_p), nblk, L - 1, _lib.ptr(ells), _lib.ptr(bs), nb,
              _lib.ptr(wo), _lib.ptr(ti), ncls, ctypes.cast(flat, ctypes.c_void_p), nslots, _lib.ptr(out), st)
    assert torch.equal(out, ref)
