"""The z tiles of the interpolated lattice scan."""
import numpy as np
import pytest

from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [11, 12, 13, 21, 24, 25, 37])
@pytest.mark.parametrize("spread", [4.0, 40.0])
def test_z_tiles(nz, spread):
    """z axes of one tile, of several equal ones and of tiles that differ by one, within the grid
    and far beyond it (wavefronts whose poses are all outside): the general kernel's energies bit
    for bit."""
    lig, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    probe_a, probe_q, types = synth.grid_types([lig], 10)
    origin, gdims, gstep = synth.grid_spec((0.0, 0.0, 0.0), 64, 0.375)
    ctx.compute_grids(probe_a, probe_q, gstep, gdims, origin, copy_out=False)
    lid = ctx.add_ligand(lig, types=types[0])
    rng = np.random.default_rng(nz)
    ax = [np.sort(rng.uniform(-1, 1, n)) * w for n, w in ((9, spread), (8, spread), (nz, min(spread, 0.6 * nz)))]
    g = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    trans = np.stack([g[2].ravel(), g[1].ravel(), g[0].ravel()], 1)
    rots = synth.random_rotations(rng, 5)
    got = []
    for how in (0, 2):
        ctx.tune(scan_lattice=how)
        got.append(ctx.scan(lid, ff.INTERP, rots, trans).cpu().numpy())
    assert np.array_equal(got[0], got[1], equal_nan=True)
    assert np.any(np.isfinite(got[0])) or spread > 4.0


@pytest.mark.parametrize("nz, nrot, spacing", [(13, 4000, 0.5), (13, 5121, 0.5), (13, 20479, 0.5), (13, 20480, 0.5), (20, 20500, 0.375),
                                               (20, 20500, 0.9), (37, 10240, 0.3)])
def test_long_z_tiles(nz, nrot, spacing):
    """Many wavefronts: z axes in longer tiles where their layers are close, on both sides of each
    limit of that rule: the general kernel's energies bit for bit."""
    rng = np.random.default_rng(nz)
    lig = synth.make_ligand(rng, 7, 4, 1)
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    probe_a, probe_q, types = synth.grid_types([lig], 10)
    origin, gdims, gstep = synth.grid_spec((0.0, 0.0, 0.0), 64, 0.375)
    ctx.compute_grids(probe_a, probe_q, gstep, gdims, origin, copy_out=False)
    lid = ctx.add_ligand(lig, types=types[0])
    trans = np.array([(x, y, z) for z in (np.arange(nz) - (nz - 1) / 2) * spacing
                      for y in (-0.7, 0.4) for x in (-1.1, 0.0, 0.3)])
    rots = synth.random_rotations(rng, nrot)
    got = []
    for how in (0, 2):
        ctx.tune(scan_lattice=how)
        got.append(ctx.scan(lid, ff.INTERP, rots, trans).cpu().numpy())
    assert np.array_equal(got[0], got[1], equal_nan=True)
    assert np.any(np.isfinite(got[0]))
