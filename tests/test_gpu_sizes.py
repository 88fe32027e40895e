"""GPU paths chosen by size: at the edges of each rule, the paths on its two sides agree with
each other and with the FP64 oracle."""
import numpy as np
import pytest

import oracle
from mmo_amd import ff, synth

from parity import assert_energy, inter_abs_sum

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sys0():
    lig, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    return ctx, lig, rec


def _rows(m):
    return np.stack([m["xs"], m["ys"], m["zs"]], 1)


@pytest.mark.parametrize("nrot,ntrans,scan_cull", [(1, 1, 5), (3, 63, 5), (2, 64, 6), (5, 65, 5),
                                                   (2, 343, 6)])
def test_split_scan_equals_whole_scan(sys0, nrot, ntrans, scan_cull):
    """The row-list scan with one ligand atom per wavefront (few tiles) gives the energies of
    the one-wavefront-per-tile form bit for bit (both add the atoms' energies in atom order),
    on partly filled tiles too, and the oracle's to 1e-5."""
    ctx, lig, rec = sys0
    lid = ctx.add_ligand(lig)
    rng = np.random.default_rng(nrot * 1000 + ntrans)
    rots, trans = synth.random_rotations(rng, nrot), rng.uniform(-4, 4, (ntrans, 3))
    got = []
    for split in (0, 1 << 20):
        ctx.tune(scan_split=split, scan_cull=scan_cull)
        got.append(ctx.scan(lid, ff.SHIFTED, rots, trans).cpu().numpy())
    ctx.tune(scan_split=12288, scan_cull=5)
    assert np.array_equal(got[0], got[1])
    pick = rng.choice(nrot * ntrans, min(16, nrot * ntrans), replace=False)
    pr, pt = (pick // ntrans).astype(np.int32), (pick % ntrans).astype(np.int32)
    want = oracle.scan_shifted(rec, lig, rots, pr, trans, pt, nthreads=4)
    sums = []
    for a, b in zip(pr, pt):
        x = _rows(lig) @ rots[a].T + trans[b]
        sums.append(inter_abs_sum(rec, x, lig, True))
    assert_energy(got[1][pick], want, sums, what="split scan")
