"""Partial slots of the FP64 spin-0 analyses (host query): the ring pairs of a pass in workgroups of
128 (Nside 64) to 2048 pairs, never more than the chunks that the pass counts."""

import pytest

from gmaster_amd import _lib


@pytest.mark.parametrize("nside,slots", [(1, 1), (64, 1), (128, 1), (256, 1), (512, 2), (1024, 1), (2048, 2), (4096, 4),
                                         (8192, 3)])
def test_spin0_slots(nside, slots):
    assert _lib.query("gm_lat_slots_s0", nside) == slots
    assert slots <= _lib.query("gm_lat_nchunks", nside, 0)
