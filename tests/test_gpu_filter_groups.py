"""The workgroups of the scan filters."""
import numpy as np
import pytest

from mmo_amd import _lib, ff, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrot,ntrans", [(2100, 65), (70_000, 63), (1100, 300), (3, 9000)])
def test_filters_of_large_and_small_scans(nrot, ntrans):
    """Scans whose workgroups take 32, 16, 8 and 4 tiles, with fewer than 64 translations and with
    more: the poses skipped before and after scoring are those of scans of a few rotations."""
    import torch
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    lid = ctx.add_ligand(synth.make_ligand(np.random.default_rng(5), 12, 8, 0))
    rng = np.random.default_rng(nrot)
    rots, trans = synth.random_rotations(rng, nrot), rng.uniform(-6, 6, (ntrans, 3))
    x = np.stack([rec["xs"], rec["ys"], rec["zs"]], 1)
    origin = x.min(axis=0) - 2.0
    ctx.set_vdw_mask(0.375, tuple(int(v) for v in np.ceil((x.max(axis=0) + 2.0 - origin) / 0.375) + 1), origin)
    flags = _lib.SCAN_ATOM_CLASH
    after = torch.zeros(nrot * ntrans, dtype=torch.float64, device="cuda:0")
    ctx.scan_filter(lid, rots, trans, after, flags=flags)
    before, kept = ctx.scan_filtered(lid, ff.SHIFTED, rots, trans, flags=flags)
    skipped = torch.isposinf(after)
    assert kept == int((~skipped).sum()) and 0 < kept < nrot * ntrans
    assert torch.all(torch.isposinf(before)[skipped])
    step = max(1, nrot // 40)
    for r in range(0, nrot, step):
        few = rots[r:r + 2]
        part = torch.zeros(len(few) * ntrans, dtype=torch.float64, device="cuda:0")
        ctx.scan_filter(lid, few, trans, part, flags=flags)
        assert torch.equal(torch.isposinf(part), skipped[r * ntrans:(r + len(few)) * ntrans])
        e, k = ctx.scan_filtered(lid, ff.SHIFTED, few, trans, flags=flags)
        assert torch.equal(e, before[r * ntrans:(r + len(few)) * ntrans])
