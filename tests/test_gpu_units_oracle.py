"""Batches by units of four ligand atoms against the oracle: the parts of the energy and the
gradient, each by itself."""
import numpy as np
import pytest

import oracle
from mmo_amd import ff, synth

from parity import assert_energy, assert_grad, inter_abs_sum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atoms", [1, 3, 4, 5, 75, 131])
@pytest.mark.parametrize("n", [1, 2400])
def test_parts_and_gradient(atoms, n):
    """Electrostatic and van der Waals parts and dE/dx of sampled poses, for ligands whose last unit is
    full or not, with one and with two units a wavefront (131 atoms: 79,200 units)."""
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    rng = np.random.default_rng(atoms + n)
    big = max(synth.library(24), key=lambda l: len(l["xs"]))
    m = min(atoms, len(big["xs"]))
    lig = {k: big[k][:m].copy() for k in ("xs", "ys", "zs", "q", "anum")}
    lig.update(dists=np.asarray(big["dists"])[:m, :m].copy(), rb_left=np.zeros(0, np.int32),
               rb_right=np.zeros(0, np.int32), rg_off=np.zeros(1, np.int32), rg_atoms=np.zeros(0, np.int32))
    rows = np.stack([lig["xs"], lig["ys"], lig["zs"]], 1)
    b = ctx.batch(np.full(n, ctx.add_ligand(lig)))
    x = np.concatenate([rows @ r.T + rng.uniform(-4, 4, 3) for r in synth.random_rotations(rng, n)])
    parts, _ = b.score(x, ff.F_INTER_SHIFTED | ff.F_COMPONENTS)
    e, g = b.score(x, ff.F_INTER_SHIFTED | ff.F_GRAD)
    both, g2 = b.score(x, ff.F_INTER_SHIFTED | ff.F_GRAD | ff.F_COMPONENTS)
    assert np.array_equal(both, parts) and np.array_equal(g2, g)
    for p in rng.choice(n, min(n, 5), replace=False):
        xp = x[p * m:(p + 1) * m]
        posed = dict(lig, xs=xp[:, 0].copy(), ys=xp[:, 1].copy(), zs=xp[:, 2].copy())
        s = inter_abs_sum(rec, xp, lig, True)
        want = oracle.ene_inter(rec, posed, shifted=True, components=True)
        assert_energy(parts[p, [0, 2, 3]], want, [s, s, s], what="parts, %d atoms" % m)
        ref, gref = oracle.grad_inter(rec, posed, shifted=True)
        assert_energy(e[p, 0], ref, s, what="gradient's energy, %d atoms" % m)
        assert_grad(g[p * m:(p + 1) * m], gref, what="gradient, %d atoms" % m)
