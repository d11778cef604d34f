"""FP64 ring-pair kernels: spin-0 maps (one, two) and spin-2 fields against the numpy oracle at
sizes on the edges of the launch shapes (a workgroup's ring pairs, 8-degree reductions, 32-degree
stages, no polar rings at Nside 2), and whole alms and maps of the spin-2 path against the
spin-2 recurrence on every ring at larger Nside, where every shape of the dispatch runs.

Tolerance: both paths evaluate the same sums in FP64 over rows whose recurrence error grows like
l^2 2^-53 near the poles (1e-12 at lmax 767); the bound is 2e-11 of the largest value."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(torch.max(torch.abs(a - b)) / torch.max(torch.abs(b)))


@pytest.mark.parametrize("nside,lmax", [(2, 2), (2, 5), (4, 8), (8, 23), (16, 31), (16, 33), (32, 64)])
@pytest.mark.parametrize("spin", [0, 2])
def test_pairs_match_oracle(nside, lmax, spin):
    from gmaster_amd import sht
    from oracle import sht as osht
    print(f"pairs: nside {nside} lmax {lmax} spin {spin}", flush=True)
    rng = np.random.default_rng(nside * 100 + lmax + spin)
    n = 1 if spin == 0 else 2
    maps = rng.normal(size=(n, 12 * nside * nside))
    ref = osht.map2alm(maps, spin, nside, lmax, 1)
    got = sht.map2alm(torch.as_tensor(maps, device="cuda"), spin, lmax, n_iter=1)
    assert np.max(np.abs(got.cpu().numpy() - ref)) < 2e-11 * np.max(np.abs(ref))
    back = sht.alm2map(torch.as_tensor(ref, device="cuda"), spin, nside, lmax).cpu().numpy()
    rback = osht.alm2map(ref, spin, nside, lmax)
    assert np.max(np.abs(back - rback)) < 2e-11 * np.max(np.abs(rback))
    if spin == 0:  # two maps through one recurrence
        pair = rng.normal(size=(2, 12 * nside * nside))
        two = sht.map2alm_s0(torch.as_tensor(pair, device="cuda"), lmax).cpu().numpy()
        for k in range(2):
            r = osht.map2alm(pair[k:k + 1], 0, nside, lmax, 0)[0]
            assert np.max(np.abs(two[k] - r)) < 2e-11 * np.max(np.abs(r))


@pytest.mark.parametrize("nside,lmax", [(64, 191), (128, 300), (256, 767), (512, 1535), (512, 1001), (1024, 2047)])
@pytest.mark.parametrize("polar_skip", [True, False])
def test_spin2_on_spin0_rows_matches_the_spin2_recurrence(nside, lmax, polar_skip):
    from gmaster_amd import sht
    if not polar_skip and nside > 256:
        pytest.skip("full rings: small sizes only")
    print(f"spin-2 rows: nside {nside} lmax {lmax} skip {polar_skip}", flush=True)
    g = torch.Generator("cuda").manual_seed(nside + lmax)
    dev = torch.device("cuda", torch.cuda.current_device())
    L, nring = lmax + 1, 4 * nside - 1
    spec = torch.view_as_complex(torch.randn((nring, 2 * L - 1, 2), dtype=torch.float64, device=dev, generator=g))
    p2, p = sht.plan2(nside, lmax, dev, polar_skip), sht.plan(nside, lmax, 2, dev, polar_skip)
    ne = L * (L + 1) // 2
    a, b = (torch.empty((2, ne), dtype=torch.complex128, device=dev) for _ in range(2))
    sht._analysis_2(p2, spec, a[0], a[1], 0)
    sht._analysis_s(p, spec, b[0], b[1], 0)
    # the polar rings the two activity rules differ on add below the skip's own bound
    assert _rel(a, b) < 2e-11
    for mode, want in ((1, 0.0), (2, 1.0)):  # subtract, then add back
        sht._analysis_2(p2, spec, a[0], a[1], mode)
        assert abs(float(a.abs().max() / b.abs().max()) - want) < 1e-10
    s, t = torch.empty_like(spec), torch.empty_like(spec)
    sht._synthesis_2(p2, b[0], b[1], s)
    sht._synthesis_s(p, b[0], b[1], t)
    assert _rel(s, t) < 2e-11
