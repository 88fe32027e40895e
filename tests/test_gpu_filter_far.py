"""Scan filters on positions far outside the mask."""
import numpy as np
import pytest

from mmo_amd import _lib, ff, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntrans", [40, 80])
def test_positions_beyond_the_range_of_an_int(ntrans):
    """Translations whose voxel numbers pass the range of a 32-bit integer (either sign, up to
    1e308 and not finite) clash with nothing, whichever axis they lie on; those in the pocket clash
    as alone."""
    import torch
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    lid = ctx.add_ligand(synth.make_ligand(np.random.default_rng(5), 12, 8, 0))
    rng = np.random.default_rng(ntrans)
    x = np.stack([rec["xs"], rec["ys"], rec["zs"]], 1)
    origin = x.min(axis=0) - 2.0
    ctx.set_vdw_mask(0.375, tuple(int(v) for v in np.ceil((x.max(axis=0) + 2.0 - origin) / 0.375) + 1), origin)
    rots, trans = synth.random_rotations(rng, 3), rng.uniform(-6, 6, (ntrans, 3))
    alone = torch.zeros(3 * ntrans, dtype=torch.float64, device="cuda:0")
    ctx.scan_filter(lid, rots, trans, alone, flags=_lib.SCAN_ATOM_CLASH)
    far = [s * v for v in (1e9, 2.0 ** 31 * 0.375, 1.7e9, 1e12, 1e300, 1e308) for s in (1.0, -1.0)] + \
        [np.inf, -np.inf, np.nan]
    at = rng.permutation(ntrans)[:len(far)]
    for k, (t, v) in enumerate(zip(at, far)):
        trans[t, k % 3] = v
    e = torch.zeros(3 * ntrans, dtype=torch.float64, device="cuda:0")
    ctx.scan_filter(lid, rots, trans, e, flags=_lib.SCAN_ATOM_CLASH)
    skipped, want = (torch.isposinf(v).cpu().numpy().reshape(3, ntrans) for v in (e, alone))
    want[:, at] = False
    assert np.array_equal(skipped, want) and want.any()
