"""gm_lu_factor / gm_lu_solve at the edges of their 64-row blocks and of the one- and four-column
solves: sizes one below, at and above 64, 128 and 192, 1 to 5 right-hand sides, and pivots far
outside the unit range (row scales 2^-1010 .. 2^1010 of a diagonally dominant matrix, the plain
quotients).  Residuals of L U and of the solve in units of eps n max|a| max|x|: each entry of a
residual is a sum of n products of FP64-rounded terms (4 covers the factors' own rounding)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.mark.parametrize("scale", [0, 1010, -1010])
@pytest.mark.parametrize("n", [1, 17, 63, 64, 65, 127, 128, 129, 193])
def test_lu_blocks(n, scale):
    from gmaster_amd import _lib

    print(f"lu edges n={n} scale={scale}", flush=True)
    st = _lib.stream_ptr("cuda")
    g = torch.Generator().manual_seed(n)
    a = torch.eye(n, dtype=torch.float64) * 2 + torch.randn((n, n), generator=g, dtype=torch.float64) / (8 * n)
    a = (a * 2.0 ** scale).cuda()
    lu, flag = a.clone(), torch.ones(1, dtype=torch.int32, device="cuda")
    _lib.call("gm_lu_factor", _lib.ptr(lu), n, _lib.ptr(flag), st)
    assert int(flag) == 0
    tol = 4 * EPS * (n + 4)
    L = torch.tril(lu, -1) + torch.eye(n, dtype=torch.float64, device="cuda")
    U = torch.triu(lu) * 2.0 ** -scale
    assert float((L @ U - a * 2.0 ** -scale).abs().max()) <= tol * 2.5
    lut = lu.T.contiguous()
    for k in (1, 2, 3, 4, 5):
        b = torch.randn((n, k), generator=g, dtype=torch.float64).cuda()
        x = b.clone()
        _lib.call("gm_lu_solve", _lib.ptr(lu), _lib.ptr(lut), n, _lib.ptr(x), k, st)
        y = x * 2.0 ** scale
        assert float(((a * 2.0 ** -scale) @ y - b).abs().max()) <= tol * 2.5 * max(float(y.abs().max()), 1e-300), k
