"""DOF gradients of batches whose ligands take different adjoint kernels."""
import numpy as np
import pytest

from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu


def _facing(n, rng):
    """A zigzag of n atoms with two torsions whose groups face each other."""
    i = np.arange(n)
    x = np.stack([1.25 * (i - (n - 1) / 2), 0.8 * (i % 2) + 0.3 * (i % 5), 0.5 * (i % 3)], 1)
    x -= x.mean(0)
    a, b = n // 3, 2 * n // 3
    groups = [i[a + 2:], i[:b]]
    return {"xs": x[:, 0].copy(), "ys": x[:, 1].copy(), "zs": x[:, 2].copy(),
            "q": rng.uniform(-0.4, 0.4, n), "anum": np.full(n, 6, np.int32),
            "dists": np.abs(i[:, None] - i[None, :]).astype(np.int32),
            "rb_left": np.array([a, b + 1], np.int32), "rb_right": np.array([a + 1, b], np.int32),
            "rg_off": np.cumsum([0] + [len(g) for g in groups]).astype(np.int32),
            "rg_atoms": np.concatenate(groups).astype(np.int32)}


@pytest.mark.parametrize("mix", ["free", "facing", "both", "one facing of many", "one free of many"])
@pytest.mark.parametrize("intra", [True, False])
def test_a_pose_does_not_depend_on_its_batch(mix, intra):
    """Energies and DOF gradients of a pose are bit for bit those it has in a batch of its ligand
    alone, whichever ligands share the batch (those whose torsions need a serial pass and those
    that do not)."""
    import torch
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    rng = np.random.default_rng(1)
    free = synth.library(4)
    facing = [_facing(20, rng), _facing(45, rng)]
    ligs = free + facing
    ids = np.array([ctx.add_ligand(l) for l in ligs])
    n = 90
    pick = {"free": np.arange(n) % 4, "facing": 4 + np.arange(n) % 2, "both": np.arange(n) * 7 % 6,
            "one facing of many": np.where(np.arange(n) == 40, 4, np.arange(n) % 4),
            "one free of many": np.where(np.arange(n) == 0, 1, 4 + np.arange(n) % 2)}[mix]
    dofs = [np.concatenate([rng.uniform(-2, 2, 3), rng.uniform(-3, 3, 3),
                            rng.uniform(-0.3, 0.3, len(ligs[k]["rb_left"]))]) for k in pick]
    flags = ff.F_INTER_SHIFTED | ff.F_GRAD | (ff.F_INTRA if intra else 0)

    def run(which):
        b = ctx.batch(ids[pick[which]])
        d = torch.tensor(np.concatenate([dofs[p] for p in which]), device="cuda:0")
        e = torch.full((len(which), 4), -7.0, dtype=torch.float64, device="cuda:0")
        g = torch.full_like(d, -7.0)
        b.score_dofs_dev(d, e, gdof=g, flags=flags)
        torch.cuda.synchronize()
        return e.cpu().numpy(), np.split(g.cpu().numpy(), np.cumsum([len(dofs[p]) for p in which])[:-1])
    e, g = run(np.arange(n))
    for k in np.unique(pick):
        mine = np.flatnonzero(pick == k)
        e1, g1 = run(mine)
        assert np.array_equal(e1, e[mine])
        assert all(np.array_equal(a, g[p]) for a, p in zip(g1, mine))
