"""Which launches pool their sweeps, and what the others do not allocate."""
import numpy as np
import pytest

from mmo_amd import ff, mc, synth
from mmo_amd.minimize import Minimizer

pytestmark = pytest.mark.gpu


def _chains(ctx, ids, n, mode=ff.SHIFTED):
    rng = np.random.default_rng(n)
    return mc.MonteCarlo(ctx, ids[np.arange(n) % len(ids)], synth.random_rotations(rng, n),
                         rng.uniform(-1, 1, (n, 3)), mode, 4, flags=mc.TWEAK_RBONDS | mc.INTRA_UFF)


@pytest.fixture(scope="module")
def small():
    ctx = ff.Context(0)
    ctx.set_receptor(synth.config0()[1])
    return ctx, np.array([ctx.add_ligand(l) for l in synth.library(6)])


@pytest.mark.parametrize("chains", [1, 256, 257, 3072, 3073])
def test_chains_pool_up_to_twelve_per_cu(small, chains):
    """The pooled form runs where the rule says so: compared with the other form elsewhere, the
    launches there are really of it."""
    ctx, ids = small
    cus = 256
    slots = -(-chains // cus)
    m = _chains(ctx, ids, chains)
    m.run(1)
    m.state()
    assert ctx.tuning("mc_pooled_slots") == (slots if slots <= 12 else 0)
    ctx.tune(mc_pool=0)
    m = _chains(ctx, ids, chains)
    m.run(1)
    m.state()
    ctx.tune(mc_pool=12)
    assert ctx.tuning("mc_pooled_slots") == 0


@pytest.mark.parametrize("poses,slots", [(1, 1), (257, 2), (800, 4), (1536, 6), (1537, 4), (2048, 4), (2049, 0)])
def test_minimiser_pools_up_to_eight_per_cu(small, poses, slots):
    """The same of the minimiser: up to six poses a CU all at once, up to eight half of them."""
    import torch
    ctx, ids = small
    b = ctx.batch(ids[np.arange(poses) % len(ids)])
    d = torch.zeros(int(b.dof_off[-1]), dtype=torch.float64, device="cuda:0")
    Minimizer(b, flags=ff.F_INTER_SHIFTED | ff.F_INTRA).run(d, 1)
    torch.cuda.synchronize()
    assert ctx.tuning("min_pooled_slots") == slots


@pytest.mark.parametrize("rec,mode,room", [("small", "shifted", True), ("large", "shifted", False),
                                           ("small", "sweep 0", False)])
def test_sums_of_pooled_sweeps_only_where_they_run(rec, mode, room):
    """3,000 chains hold the pooled sweeps' 3 KiB per four atoms only where these can run: not on
    a receptor too large for LDS, not with the sub-block sweep."""
    import torch
    ctx = ff.Context(0)
    ctx.set_receptor(synth.config0()[1] if rec == "small" else synth.config4_receptor())
    if mode == "sweep 0":
        ctx.tune(mc_sweep=0)
    ids = np.array([ctx.add_ligand(l) for l in synth.library(6)])
    _chains(ctx, ids, 8)   # the registry's own lists
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    m = _chains(ctx, ids, 3000)
    used = free - torch.cuda.mem_get_info()[0]
    atoms = max(ctx.ligand_natoms(int(i)) for i in ids)
    sums = 12 * 256 * -(-atoms // 4) * 3072
    assert (used >= sums) if room else (used < sums // 4), (used, sums)
    m.run(1)
    m.state()
    assert (ctx.tuning("mc_pooled_slots") > 0) == room
