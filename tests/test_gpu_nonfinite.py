"""Maps with a pixel that is not finite: a spin-2 analysis has no alm below l = 2, whatever the ring
sums are, and every other alm of an order sees the pixel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("pixel", [0, 500, 24000])  # cap, cap edge, belt
def test_spin2_analysis_of_a_pixel_that_is_not_finite(value, pixel):
    from gmaster_amd import sht

    nside, lmax = 64, 70
    print(f"not finite: {value} at pixel {pixel}", flush=True)
    maps = torch.randn((2, 12 * nside * nside), dtype=torch.float64, device="cuda",
                       generator=torch.Generator("cuda").manual_seed(pixel))
    maps[0, pixel] = value
    L = lmax + 1
    low = torch.tensor([0, 1, L], device="cuda")  # (l, m) = (0, 0), (1, 0), (1, 1)
    for n_iter in (0, 1):
        alm = torch.view_as_real(sht.map2alm_spin(maps, lmax, 2, n_iter=n_iter))
        assert float(alm[:, low].abs().max()) == 0.0
        alm[:, low] = float("nan")
        assert not torch.isfinite(alm[:, :, 0]).any()
