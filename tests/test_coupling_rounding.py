"""Rounding of the coupling sums' first terms (host build, the helpers of test_coupling_host.py):
with the window at l3 = 0 or 1 alone and l1 = l2 = l the sums are (l l 0; m -m 0)^2 = 1 / (2l + 1) and
(l l 1; 2 -2 0)^2 = 4 / (l (l+1) (2l+1)).  Near the diagonal these terms of a mask's window are
most of the sum.  Bound: the rms relative error that two recursions (one for each of f0 and f2)
have over l = 2 .. 600, 1.16 units of 2^-53 for the even sums and 1.24 for the odd one, and 3%."""

import numpy as np
import pytest

from test_coupling_host import _run, host_bin  # noqa: F401  (fixture)


@pytest.mark.parametrize("l3", [0, 1])
def test_first_terms(host_bin, tmp_path, l3):
    lmax = 600
    window = np.zeros(l3 + 1)
    window[l3] = 4 * np.pi / (2 * l3 + 1)
    _run(host_bin, tmp_path, window, lmax)
    pair = np.fromfile(tmp_path / "p").reshape(lmax + 1, lmax + 1, 4)  # the sums themselves
    l = np.arange(2, lmax + 1).astype(np.longdouble)
    w = np.longdouble(window[l3] * (2 * l3 + 1) / (4 * np.pi))
    if l3 == 0:
        cases = [(0, 1 / (2 * l + 1), 1.16), (1, 1 / (2 * l + 1), 1.16), (2, 1 / (2 * l + 1), 1.16)]
    else:
        cases = [(3, 4 / (l * (l + 1) * (2 * l + 1)), 1.24)]
    for k, exact, bound in cases:
        got = pair[np.arange(2, lmax + 1), np.arange(2, lmax + 1), k]
        rms = float(np.sqrt(np.mean((got / (w * exact) - 1) ** 2))) * 2.0 ** 53
        print(f"sum {k}: {rms:.2f}")
        assert rms < 1.03 * bound, (k, rms)
