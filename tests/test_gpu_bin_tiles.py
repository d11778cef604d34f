"""gm_bin_block beyond one tile: more than 256 columns and more than 64 or 256 bins (both bin counts
of a workgroup, one and two rows of bins), bins across the 256-column boundary, a last partial group of bins, uneven bands with
gaps.  Tolerance: n + 4 roundings of the largest term for a sum of n terms."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


def _bands(kind, lmax):
    """Multipoles (ascending, some left out) and band starts."""
    if kind == "uneven":  # bands of 1 .. 300 degrees
        rng = np.random.default_rng(5)
        ells = np.flatnonzero(rng.random(lmax + 1) < 0.95)
        sizes = []
        while sum(sizes) < len(ells):
            sizes.append(int(rng.choice([1, 2, 7, 40, 255, 257, 300])))
        start = np.minimum(np.concatenate([[0], np.cumsum(sizes)]), len(ells))
    else:
        ells = np.arange(2, lmax + 1)
        start = np.concatenate([np.arange(0, len(ells), kind), [len(ells)]])
    return ells, start


@pytest.mark.parametrize("kind,lmax", [(1, 600), (1, 257), (1, 768), (2, 900), (2, 2100), (3, 1000), (3, 2200), (7, 999), (100, 700), (300, 900),
                                       ("uneven", 1000)])
def test_bin_block_tiles(kind, lmax):
    from gmaster_amd import _lib

    print(f"bin tiles {kind} lmax {lmax}", flush=True)
    ells, start = _bands(kind, lmax)
    L, nb = lmax + 1, len(start) - 1
    g = torch.Generator("cuda").manual_seed(lmax)
    M = torch.randn((L, L), dtype=torch.float64, device="cuda", generator=g)
    wo, ti = (torch.rand(len(ells), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    de = torch.as_tensor(ells, dtype=torch.int32, device="cuda")
    ds = torch.as_tensor(start, dtype=torch.int32, device="cuda")
    out = torch.full((nb + 1, nb), 7.0, dtype=torch.float64, device="cuda")
    _lib.call("gm_bin_block", _lib.ptr(M), lmax, _lib.ptr(de), _lib.ptr(ds), nb, _lib.ptr(wo), _lib.ptr(ti),
              _lib.ptr(out), _lib.stream_ptr("cuda"))
    t = wo.cpu().numpy()[:, None] * M.cpu().numpy()[np.ix_(ells, ells)] * ti.cpu().numpy()[None, :]
    keep = np.diff(start) > 0  # reduceat would repeat an element for an empty band
    ref = np.zeros((nb, nb))
    ref[np.ix_(keep, keep)] = np.add.reduceat(np.add.reduceat(t, start[:-1][keep], 0), start[:-1][keep], 1)
    got = out.cpu().numpy()
    assert (got[nb] == 7.0).all()
    n = int(np.max(np.diff(start)))
    assert np.max(np.abs(got[:nb] - ref)) <= (n * n + 4) * 2 * EPS * np.max(np.abs(t))
