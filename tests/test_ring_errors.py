"""Refused ring FFT calls name the entry that was called (host checks, nothing is launched)."""

import pytest

from gmaster_amd import _lib


@pytest.mark.parametrize("kind", ["fft", "pair"])
@pytest.mark.parametrize("entry,args", [
    ("fwd_s0", (None, 1, 48, 2, 5, None, 6, 42, None)),
    ("fwd_s", (None, None, 2, 5, None, 11, None)),
    ("inv_s0", (None, 1, 6, 42, 2, 5, None, 48, None)),
    ("inv_s", (None, 11, 2, 5, None, None, None)),
])
def test_null_pointers_are_named(kind, entry, args):
    name = f"gm_ring_{kind}_{entry}"
    with pytest.raises(_lib.GmError) as e:
        _lib.call(name, *args)
    assert f"{name}: null pointer" in str(e.value)
