"""The rule that a ligand's torsions need no serial pass, over words of its atom sets."""
import numpy as np
import pytest

import oracle
from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 63, 64, 65, 127, 129, 192])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_random_groups_across_words(n, seed):
    """Groups of random kinds (far sides, near sides, a few atoms near the words' edges): whichever adjoint the rule picks, the DOF gradient is the oracle's Jacobian applied to
    the coordinate gradient, to 1e-9 of the sum of its terms (a few hundred FP64 terms, coordinates
    equal to 1e-13 A, pairs beyond 0.5 A)."""
    import torch
    rng = np.random.default_rng(100 * n + seed)
    i = np.arange(n)
    x = np.stack([1.25 * (i - (n - 1) / 2), 0.8 * (i % 2) + 0.3 * (i % 5), 0.5 * (i % 3)], 1)
    x -= x.mean(0)
    left, right, groups = [], [], []
    for b in np.sort(rng.choice(n - 1, min(7, n - 2), replace=False)):
        kind = rng.integers(0, 4)
        if kind == 1:
            left.append(b + 1), right.append(b), groups.append(i[:b])
        else:
            left.append(b), right.append(b + 1)
            far = i[b + 2:]
            if kind == 2:
                rest = np.setdiff1d(i, [b, b + 1])
                near = rest[np.argsort(np.minimum(rest % 64, 63 - rest % 64), kind="stable")]
                far = np.sort(near[:rng.integers(1, min(6, len(rest)) + 1)])
            groups.append(far)
    off = np.cumsum([0] + [len(g) for g in groups]).astype(np.int32)
    lig = {"xs": x[:, 0].copy(), "ys": x[:, 1].copy(), "zs": x[:, 2].copy(), "q": rng.uniform(-.4, .4, n),
           "anum": np.full(n, 6, np.int32), "dists": np.abs(i[:, None] - i[None, :]).astype(np.int32),
           "rb_left": np.array(left, np.int32), "rb_right": np.array(right, np.int32), "rg_off": off,
           "rg_atoms": np.concatenate(groups).astype(np.int32)}
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    b = ctx.batch(np.array([ctx.add_ligand(lig)]))
    d = np.concatenate([rng.uniform(-3, 3, 6), rng.uniform(-0.3, 0.3, len(left))])
    xo = torch.empty((n, 3), dtype=torch.float64, device="cuda:0")
    g = torch.empty(len(d), dtype=torch.float64, device="cuda:0")
    e = torch.empty((1, 4), dtype=torch.float64, device="cuda:0")
    b.score_dofs_dev(torch.tensor(d, device="cuda:0"), e, xyz_out=xo, gdof=g,
                     flags=ff.F_INTER_SHIFTED | ff.F_GRAD)
    torch.cuda.synchronize()
    _, h = b.score(xo.cpu().numpy(), ff.F_INTER_SHIFTED | ff.F_GRAD)
    J = oracle.apply_config_jvp(x, lig["rb_left"], lig["rb_right"], off, lig["rg_atoms"], d)[2]
    scale = np.abs(J).sum(axis=(1, 2)) * np.abs(h).max()
    np.testing.assert_array_less(np.abs(g.cpu().numpy() - (J * h).sum(axis=(1, 2))), 1e-9 * scale + 1e-12)
