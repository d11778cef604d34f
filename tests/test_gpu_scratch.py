"""Scratch memory of the FP64 analyses: what their kernels write and no more."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside,maps", [(64, 1), (512, 2), (1024, 1), (1024, 2), (2048, 2)])
def test_spin0_partial_sums(nside, maps):
    """At Nside 1024 one workgroup takes an order's 2048 ring pairs, at 2048 two."""
    from gmaster_amd import _lib, sht

    lmax = 300
    print(f"scratch: nside {nside} maps {maps}", flush=True)
    p = sht.plan(nside, lmax, 0, "cuda")
    g = torch.Generator("cuda").manual_seed(nside)
    spec = torch.randn((maps, 4 * nside - 1, lmax + 1), dtype=torch.complex128, device="cuda", generator=g)
    alm = torch.empty((maps, (lmax + 1) * (lmax + 2) // 2), dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_stats()["requested_bytes.all.current"]
    sht._analysis_s0(p, spec, alm, 0)
    used = torch.cuda.memory_stats()["requested_bytes.all.peak"] - base
    slots = {64: 1, 512: 2, 1024: 1, 2048: 2}[nside]
    assert used <= slots * int(_lib.query("gm_table_size", lmax)) * 16 * maps


@pytest.mark.parametrize("nside,lmax", [(256, 767), (512, 1535)])
def test_spin2_tables(nside, lmax):
    """The spin-2 tables that a geometry keeps beside the spin-0 ones: the orders of the polar rings
    alone, equal to the head of the full tables."""
    from gmaster_amd import _lib, sht

    sht.clear_plans()
    dev = torch.device("cuda", torch.cuda.current_device())
    base = torch.cuda.memory_stats()["requested_bytes.all.current"]
    p = sht.plan2(nside, lmax, dev)
    kept = torch.cuda.memory_stats()["requested_bytes.all.current"] - base
    assert p.mpol < (lmax + 1) // 3
    tables = 2 * int(_lib.query("gm_table_size", lmax + 2)) + 3 * p.ptsize
    assert kept <= 8 * tables + 64 * (lmax + 3)  # and a few numbers per order
    full = sht.plan(nside, lmax, 2, dev)
    for name in ("alpha", "gamma", "P"):
        assert torch.equal(getattr(p.pol, name), getattr(full, name)[:p.ptsize])
