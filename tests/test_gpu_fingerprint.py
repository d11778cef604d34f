"""gm_fingerprint against its definition (sums of position-keyed splitmix64 hashes) on the host, at
sizes around its workgroup, its unroll, its largest grid and with odd bytes at the end."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


@pytest.mark.parametrize("nbytes", [0, 1, 8, 13, 8 * 1023, 8 * 1024, 8 * 1025 + 7, 8 * 262144, 8 * 262145, 8 * 1100000 + 3])
def test_fingerprint_matches_host(nbytes):
    from gmaster_amd import _lib

    data = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    n = nbytes // 8
    with np.errstate(over="ignore"):
        w = data[:8 * n].view(np.uint64)
        key = _mix(np.arange(n, dtype=np.uint64) + np.uint64(0x9E3779B97F4A7C15))
        h = _mix(w ^ key)
        if nbytes % 8:
            t = np.uint64(int.from_bytes(data[8 * n:].tobytes(), "little"))
            k = _mix(np.array([n], dtype=np.uint64) + np.uint64(0x9E3779B97F4A7C15))
            h = np.concatenate([h, _mix(t ^ k ^ np.uint64(0xFF51AFD7ED558CCD))])
        ref = [int(h.sum(dtype=np.uint64)), int(_mix(h ^ np.uint64(0x632BE59BD9B4E019)).sum(dtype=np.uint64))]
    dev = torch.as_tensor(np.concatenate([data, np.zeros(8, np.uint8)])).cuda()
    out = torch.empty(2, dtype=torch.int64, device="cuda")
    _lib.call("gm_fingerprint", _lib.ptr(dev), nbytes, _lib.ptr(out), _lib.stream_ptr("cuda"))
    assert [int(v) % 2 ** 64 for v in out.cpu()] == ref
