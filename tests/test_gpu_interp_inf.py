"""Interpolated scans through grids with infinite nodes."""
import numpy as np
import pytest

from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 4, 6), (1, 1, 23)])
def test_infinite_nodes(dims):
    """Poses inside the grid whose atoms lie among +inf nodes are +inf in both scan kernels and
    in the filtered scan, as in the batch (NaN is the mark of an atom outside the grid); all
    other poses agree with the batch to 1e-12 of the sum of their terms (75 terms of 8 products:
    600 roundings of 2^-53 each)."""
    import torch
    lig, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    rng = np.random.default_rng(4)
    n, step = 40, 0.6
    grids = rng.normal(0.0, 3.0, (2, n, n, n)).astype(np.float32)
    grids[:, 30:, :, :] = np.inf                    # z: whole layers
    grids[:, :, :, 31:] = np.inf                    # x: half a cell's nodes
    origin = np.full(3, -0.5 * step * (n - 1))
    ctx.set_grids(grids, step, origin)
    lid = ctx.add_ligand(lig, types=rng.integers(0, 2, len(lig["xs"])))
    ax = [np.sort(rng.uniform(-9.0, 9.0, d)) for d in dims]
    g = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    trans = np.stack([g[2].ravel(), g[1].ravel(), g[0].ravel()], 1)
    rots = synth.random_rotations(rng, 40)
    x = np.stack([lig["xs"], lig["ys"], lig["zs"]], 1)
    posed = np.concatenate([x @ r.T + t for r in rots for t in trans])
    b = ctx.batch(np.full(len(rots) * len(trans), lid))
    want = b.score(posed, ff.F_INTER_INTERP)[0][:, 0]
    kinds = [np.isnan(want), np.isposinf(want), np.isfinite(want)]
    assert all(k.sum() > 10 for k in kinds)
    fin = kinds[2]
    for how in (0, 2):
        ctx.tune(scan_lattice=how)
        got = ctx.scan(lid, ff.INTERP, rots, trans).cpu().numpy()
        assert np.array_equal(np.isnan(got), kinds[0]) and np.array_equal(np.isposinf(got), kinds[1])
        np.testing.assert_allclose(got[fin], want[fin], rtol=0, atol=1e-12 * 75 * 15.0)
    ctx.tune(scan_lattice=1)
    flt, _ = ctx.scan_filtered(lid, ff.INTERP, rots, trans, flags=0)
    assert torch.equal(flt.nan_to_num(7.0, 8.0), torch.tensor(got, device=flt.device).nan_to_num(7.0, 8.0))
