"""Rows of the mode-coupling recursion that the mask window cuts short inside a wave (host build,
the helpers of test_coupling_host.py)."""

import numpy as np
import pytest

from test_coupling_host import _run, _window, host_bin  # noqa: F401  (fixture)


@pytest.mark.parametrize("lmax,lw", [(700, 1100), (700, 720)])
def test_lanes_that_end_before_their_wave(host_bin, tmp_path, lmax, lw):
    """Long rows cut by the window: lanes end up to 63 degrees before their wave does and must
    give their pair's sums bit for bit (their factors stay finite meanwhile)."""
    pair, wave = _run(host_bin, tmp_path, _window("white", lw + 1, 3), lmax)
    iu = np.triu_indices(lmax + 1)
    assert np.isfinite(pair).all()
    assert np.array_equal(wave[iu], pair[iu])
