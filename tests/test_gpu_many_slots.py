"""Workspaces with one block per channel pair: a joint TEB workspace (7 channels, 49 pairs) after
``update_coupling_matrix`` with a full matrix, and read back from its file, against a dense
binning and solve.  Tolerances: a binned element is a sum of n = nlb^2 products of three factors,
(n + 4) 2^-53 of the largest; the bandpowers' solve adds its condition number (below 10)."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.mark.parametrize("nlb", [1, 5])
def test_teb_workspace_with_a_full_matrix(tmp_path, nlb):
    import gmaster_amd as nmt

    nside, lmax, ncls = 8, 20, 7
    L = lmax + 1
    rng = np.random.default_rng(nlb)
    mask = rng.uniform(0.5, 1.0, 12 * nside * nside)
    f0 = nmt.NmtField(mask, rng.normal(size=(1, 12 * nside * nside)), lmax=lmax, lmax_mask=lmax, n_iter=0)
    f2 = nmt.NmtField(mask, rng.normal(size=(2, 12 * nside * nside)), lmax=lmax, lmax_mask=lmax, n_iter=0)
    b = nmt.NmtBin.from_lmax_linear(lmax, nlb)
    w = nmt.NmtWorkspace.from_fields(f0, f2, b, is_teb=True)
    n = L * ncls
    new = np.eye(n) + rng.uniform(-1, 1, size=(n, n)) / n
    w.update_coupling_matrix(new)
    nb = b.get_n_bands()
    W = b.binning_matrix(torch.device("cuda")).cpu().numpy()  # (bands, L)
    sel = (W > 0).astype(np.float64)
    m4 = new.reshape(L, ncls, L, ncls)
    want = np.einsum("il,lcmd,jm->icjd", W, m4, sel).reshape(nb * ncls, nb * ncls)
    got = w.mcm_binned.cpu().numpy()
    assert np.max(np.abs(got - want)) <= (nlb * nlb + 4) * 2 * EPS * np.max(np.abs(new)) * nlb
    cl = rng.uniform(size=(ncls, L))
    ref = np.linalg.solve(want, (cl @ W.T).T.reshape(-1)).reshape(nb, ncls).T
    bp = w.decouple_cell(cl).cpu().numpy()
    assert np.max(np.abs(bp - ref)) < 10 * nb * ncls * EPS * np.max(np.abs(ref))
    fn = str(tmp_path / "w.fits")
    w.write_to(fn)
    again = nmt.NmtWorkspace.from_file(fn)
    assert torch.equal(again.mcm_binned, w.mcm_binned)
    assert np.array_equal(again.decouple_cell(cl).cpu().numpy(), bp)
