"""Rigid scans on a device without memory to spare."""
import numpy as np
import pytest

from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu


def test_scan_without_room_for_its_split_form():
    """A scan of 12,288 tiles whose split form would take 450 MiB, on a device with less than 300
    MiB left: it runs in the whole form, and gives the energies that the split form gives once
    there is memory (both add the atoms' energies in the same order)."""
    import torch
    lig, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    lid = ctx.add_ligand(lig)
    rots, trans = synth.so3_rotations(1536), synth.lattice((0.0, 0.0, 0.0), 8, 0.5)
    out = torch.empty(len(rots) * len(trans), dtype=torch.float64, device="cuda:0")
    ctx.scan(lid, ff.SHIFTED, rots[:1], trans[:1], out=out[:1])   # everything but the split's memory
    ctx.tune(scan_split=0)
    ctx.scan(lid, ff.SHIFTED, rots, trans, out=out)
    want = out.clone()
    ctx.tune(scan_split=12288)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    held = torch.empty(free - (200 << 20), dtype=torch.uint8, device="cuda:0")
    out.zero_()
    ctx.scan(lid, ff.SHIFTED, rots, trans, out=out)
    assert torch.equal(out, want)
    del held
    torch.cuda.empty_cache()
    out.zero_()
    ctx.scan(lid, ff.SHIFTED, rots, trans, out=out)
    assert torch.equal(out, want)
