"""One pose against large receptors."""
import numpy as np
import pytest

import oracle
from mmo_amd import ff, synth

from parity import assert_energy, assert_grad, inter_abs_sum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrec", [32768, 32769, 98305])
@pytest.mark.parametrize("atoms", [30, 131])
def test_plain_forms_at_slice_lengths(nrec, atoms):
    """Receptors on either side of the sizes at which the slices of one pose grow from 64 atoms to
    128 and 256, the last slice with one atom: energy, parts and gradient, both modes."""
    base = synth.config4_receptor()
    rng = np.random.default_rng(nrec + atoms)
    x = np.concatenate([np.stack([base["xs"], base["ys"], base["zs"]], 1) + 62.0 * np.array(s)
                        for s in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1))])
    pick = np.sort(rng.permutation(len(x))[:nrec])
    x = x[pick]
    rec = {"xs": x[:, 0].copy(), "ys": x[:, 1].copy(), "zs": x[:, 2].copy(),
           "q": np.tile(base["q"], 7)[pick], "anum": np.tile(base["anum"], 7)[pick].astype(np.int32)}
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    big = max(synth.library(24), key=lambda l: len(l["xs"]))
    keep = np.arange(min(atoms, len(big["xs"])))
    lig = {k: big[k][keep].copy() for k in ("xs", "ys", "zs", "q", "anum")}
    p = np.stack([lig["xs"], lig["ys"], lig["zs"]], 1) + 31.0 + rng.uniform(-3, 3, 3)
    lig.update(xs=p[:, 0].copy(), ys=p[:, 1].copy(), zs=p[:, 2].copy())
    for mode, shifted in ((ff.SHIFTED, True), (ff.GLOBAL, False)):
        s = inter_abs_sum(rec, p, lig, shifted)
        got = ctx.ene_inter(lig, mode, components=True)
        assert_energy(got, oracle.ene_inter(rec, lig, shifted=shifted, components=True), [s, s, s], what="plain")
        e, g = ctx.ene_inter_grad(lig, mode)
        want, gwant = oracle.grad_inter(rec, lig, shifted=shifted)
        assert_energy(e, want, s, what="plain gradient's energy")
        assert_grad(g, gwant, what="plain gradient")
