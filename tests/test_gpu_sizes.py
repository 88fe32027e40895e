"""GPU paths chosen by size: at the edges of each rule, the paths on its two sides agree with
each other and with the FP64 oracle."""
import numpy as np
import pytest

import oracle
from mmo_amd import ff, synth

from parity import assert_energy, assert_grad, inter_abs_sum

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


def _topk_input(kind, n, rng):
    if kind == "ties":          # 7 values: far more equal keys than the candidate list holds
        return rng.integers(-3, 4, n).astype(np.float64)
    if kind == "inf":           # a filtered scan: a few finite energies
        e = np.full(n, np.inf)
        e[rng.choice(n, 50, replace=False)] = rng.normal(-20, 30, 50)
        return e
    if kind == "close":         # keys that share their first 40 bits
        return -1.0 - rng.integers(0, 1 << 20, n) * 2.0 ** -52
    e = rng.normal(0, 1, n) * 10.0 ** rng.uniform(-300, 300, n)
    e[rng.choice(n, 5, replace=False)] = [np.nan, -np.inf, 0.0, -0.0, 5e-324]
    return e


@pytest.mark.parametrize("kind", ["ties", "inf", "close", "wide"])
@pytest.mark.parametrize("n,k", [(4096, 2048), (4097, 2048), (4097, 1), (300_001, 100), (300_001, 2048)])
def test_topk_edges(sys0, kind, n, k):
    """The top-k at the sizes where its path changes (the candidate list holds 4,096), on
    ties beyond the list, +inf but for a few, keys that differ in their last bits only and
    the whole range of doubles: exactly the (energy, index) order, on an input that is not
    16-byte aligned."""
    import torch
    ctx, _, _ = sys0
    rng = np.random.default_rng(n + k)
    e = _topk_input(kind, n, rng)
    d = torch.empty(n + 1, dtype=torch.float64, device="cuda:0")[1:]
    d.copy_(torch.tensor(e))
    v, i = ctx.topk(d, k)
    bits = e.view(np.int64)
    key = np.where(bits < 0, ~bits.view(np.uint64), bits.view(np.uint64) | np.uint64(1 << 63))
    key[np.isnan(e)] = np.uint64(0xFFFFFFFFFFFFFFFF)
    want = np.lexsort((np.arange(n), key))[:k]
    assert np.array_equal(i.cpu().numpy(), want)
    assert np.array_equal(v.cpu().numpy(), e[want], equal_nan=True)


@pytest.mark.parametrize("nrot,ntrans", [(1, 1), (40, 3), (70, 63), (3, 64), (2, 2049), (1, 4500)])
def test_scan_filters_on_few_and_many_translations(sys0, nrot, ntrans):
    """The clash filters with fewer than 64 translations (slots of several rotations in a
    wavefront) and with more (one rotation per workgroup, 2,048 slots each), before and after
    scoring: the poses that the mask's corners give, and atoms or translations that are not finite
    never clash."""
    import torch
    from mmo_amd import _lib
    ctx, lig, rec = sys0
    small = synth.make_ligand(np.random.default_rng(5), 12, 8, 0)
    lid = ctx.add_ligand(small)
    rng = np.random.default_rng(nrot + ntrans)
    rots, trans = synth.random_rotations(rng, nrot), rng.uniform(-6, 6, (ntrans, 3))
    if ntrans > 3:
        trans[2, 1] = np.nan
    rxyz, step = _rows(rec), 0.375
    origin = rxyz.min(axis=0) - 2.0
    dims = tuple(int(v) for v in np.ceil((rxyz.max(axis=0) + 2.0 - origin) / step) + 1)
    ctx.set_vdw_mask(step, dims, origin)
    flags = _lib.SCAN_ATOM_CLASH
    before, kept = ctx.scan_filtered(lid, ff.SHIFTED, rots, trans, flags=flags)
    after = torch.zeros(nrot * ntrans, dtype=torch.float64, device="cuda:0")
    ctx.scan_filter(lid, rots, trans, after, flags=flags)
    skipped = np.isinf(after.cpu().numpy())
    words = ctx.vdw_mask()
    bit = lambda v: (words[v >> 5] >> (v & 31)) & 1   # noqa: E731
    c = _rows(small)
    want = np.zeros((nrot, ntrans), dtype=bool)
    for r in range(nrot):
        f = ((c @ rots[r].T)[None] + trans[:, None] - origin) * (1.0 / step)
        inside = np.all((f > -1.0) & (f < np.array(dims) - 1), axis=2)
        i = np.where(inside[..., None], np.nan_to_num(f), 0.0).astype(np.int64)
        for q in range(8):
            v = (i[..., 0] + (q & 1)) + dims[0] * ((i[..., 1] + ((q >> 1) & 1)) + dims[1] * (i[..., 2] + (q >> 2)))
            want[r] |= np.any(inside & (bit(v) != 0), axis=1)
    assert np.array_equal(skipped, want.ravel())
    e = before.cpu().numpy()
    assert kept == int((~skipped).sum()) and np.array_equal(np.isposinf(e) & skipped, skipped)
    full = ctx.scan(lid, ff.SHIFTED, rots, trans).cpu().numpy()
    assert np.array_equal(e[~skipped], full[~skipped], equal_nan=True)


def _lattice(nx, ny, nz, step, order, rng):
    """nx x ny x nz translations with unequal steps, listed with `order` from slow to fast."""
    ax = [np.sort(rng.uniform(-0.5, 0.5, n)) * step * n for n in (nx, ny, nz)]
    g = np.meshgrid(*[ax[k] for k in order], indexing="ij")
    return np.stack([g[order.index(k)].ravel() for k in range(3)], 1)


@pytest.mark.parametrize("dims,step,order", [
    ((1, 1, 1), 0.5, (2, 1, 0)), ((64, 1, 1), 0.3, (2, 1, 0)), ((5, 13, 21), 0.4, (2, 1, 0)),
    ((13, 5, 40), 0.2, (0, 1, 2)), ((7, 9, 20), 0.5, (1, 2, 0)), ((3, 4, 8), 3.0, (2, 0, 1)),
    ((2, 2, 60), 0.9, (2, 1, 0))])
def test_lattice_scan_equals_general_scan(sys0, dims, step, order):
    """The interpolated scan of a translation lattice (unequal steps, any axis fastest, columns
    that fill a wavefront or not, more and fewer z than one wavefront takes, poses that leave
    the grid) gives the general kernel's energies bit for bit."""
    ctx, lig, rec = sys0
    probe_a, probe_q, types = synth.grid_types([lig], 10)
    origin, gdims, gstep = synth.grid_spec((0.0, 0.0, 0.0), 64, 0.375)
    ctx.compute_grids(probe_a, probe_q, gstep, gdims, origin, copy_out=False)
    lid = ctx.add_ligand(lig, types=types[0])
    rng = np.random.default_rng(sum(dims))
    rots, trans = synth.random_rotations(rng, 3), _lattice(*dims, step, order, rng)
    got = []
    for how in (0, 2):
        ctx.tune(scan_lattice=how)
        got.append(ctx.scan(lid, ff.INTERP, rots, trans).cpu().numpy())
    ctx.tune(scan_lattice=1)
    assert np.array_equal(got[0], got[1], equal_nan=True)


@pytest.mark.parametrize("atoms", [1, 4, 5, 75, 131])
@pytest.mark.parametrize("n", [1, 2400])
def test_pose_units(sys0, atoms, n):
    """Batches by units of four ligand atoms: ligands whose last unit is full or not, one
    pose and enough (131 atoms: 79,200 units) for two units a wavefront.  Energies, their
    parts and gradients of sampled poses against the oracle, and each pose alone gives the
    bits it has in the batch, also through DOF vectors."""
    import torch
    ctx, _, rec = sys0
    rng = np.random.default_rng(atoms)
    lig = synth.config0()[0] if atoms == 75 else None
    if lig is None:
        big = max(synth.library(24), key=lambda l: len(l["xs"]))
        keep = np.arange(min(atoms, len(big["xs"])))
        lig = {k: big[k][keep] for k in ("xs", "ys", "zs", "q", "anum")}
        lig.update(dists=np.asarray(big["dists"])[np.ix_(keep, keep)], rb_left=np.zeros(0, np.int32),
                   rb_right=np.zeros(0, np.int32), rg_off=np.zeros(1, np.int32),
                   rg_atoms=np.zeros(0, np.int32))
    lid = ctx.add_ligand(lig)
    b = ctx.batch(np.full(n, lid))
    x = np.concatenate([_rows(lig) @ r.T + rng.uniform(-4, 4, 3) for r in synth.random_rotations(rng, n)])
    flags = ff.F_INTER_SHIFTED | ff.F_INTRA
    e, g = b.score(x, flags | ff.F_GRAD)
    ec, _ = b.score(x, flags | ff.F_COMPONENTS)
    np.testing.assert_allclose(ec[:, 2] + ec[:, 3], ec[:, 0], rtol=1e-12, atol=1e-9)
    one = ctx.batch(np.array([lid]))
    m = len(lig["xs"])
    for p in rng.choice(n, min(n, 6), replace=False):
        xp = x[p * m:(p + 1) * m]
        e1, g1 = one.score(xp, flags | ff.F_GRAD)
        assert np.array_equal(e1[0], e[p]) and np.array_equal(g1, g[p * m:(p + 1) * m])
        posed = dict(lig, xs=xp[:, 0].copy(), ys=xp[:, 1].copy(), zs=xp[:, 2].copy())
        s = inter_abs_sum(rec, xp, lig, True)
        want = oracle.ene_inter(rec, posed, shifted=True)
        assert_energy(e[p, 0], want, s, what="units %d" % atoms)
        assert_energy(ec[p, 0], want, s, what="units %d, parts" % atoms)
    d = torch.tensor(np.concatenate([np.concatenate([rng.uniform(-3, 3, 6), np.zeros(len(lig["rb_left"]))])
                                     for _ in range(n)]), device="cuda:0")
    ed = torch.full((n, 4), 7.0, dtype=torch.float64, device="cuda:0")
    gd = torch.empty_like(d)
    b.score_dofs_dev(d, ed, gdof=gd, flags=ff.F_INTER_SHIFTED | ff.F_GRAD)
    nd = len(d) // n
    e1, g1 = torch.full((1, 4), 7.0, dtype=torch.float64, device="cuda:0"), torch.empty(nd, dtype=torch.float64, device="cuda:0")
    one.score_dofs_dev(d[-nd:].clone(), e1, gdof=g1, flags=ff.F_INTER_SHIFTED | ff.F_GRAD)
    torch.cuda.synchronize()
    assert torch.equal(e1[0], ed[-1]) and torch.equal(g1, gd[-nd:])
    assert torch.all(ed[:, 1:] == 0)   # no E_intra asked for, no parts with the gradient


def _chain(n, nrb, kind, rng):
    """A zigzag of n atoms with nrb torsions: groups that are the far side of each bond
    ("nested"), both sides in turn ("facing"), two arms turned outwards ("arms"), or any
    atoms at all ("any")."""
    i = np.arange(n)
    x = np.stack([1.25 * (i - (n - 1) / 2), 0.8 * (i % 2) + 0.3 * (i % 5), 0.5 * (i % 3)], 1)
    left, right, groups = [], [], []
    for k in np.sort(rng.choice(n - 1, min(nrb, n - 1), replace=False)) if n > 2 else []:
        far, near = i[k + 2:], i[:k]
        back = {"nested": False, "facing": len(left) % 2 == 1, "arms": k < n // 2, "any": False}[kind]
        left.append(k + 1 if back else k)
        right.append(k if back else k + 1)
        groups.append(near if back else far)
        if kind == "any":
            rest = np.setdiff1d(i, [k, k + 1])
            groups[-1] = np.sort(rng.choice(rest, rng.integers(0, len(rest) + 1), replace=False))
    if kind == "arms":   # outermost last within either arm: parents before children
        order = np.argsort([-r if l > r else r for l, r in zip(left, right)], kind="stable")
        left, right, groups = ([v[o] for o in order] for v in (left, right, groups))
    off = np.concatenate([[0], np.cumsum([len(g) for g in groups])]).astype(np.int32)
    c = x - x.mean(0)
    return {"xs": c[:, 0].copy(), "ys": c[:, 1].copy(), "zs": c[:, 2].copy(),
            "q": rng.uniform(-0.4, 0.4, n), "anum": rng.choice([6, 7, 8, 1], n).astype(np.int32),
            "dists": np.abs(i[:, None] - i[None, :]).astype(np.int32),
            "rb_left": np.array(left, np.int32), "rb_right": np.array(right, np.int32), "rg_off": off,
            "rg_atoms": np.concatenate([np.zeros(0, int)] + groups).astype(np.int32)}


@pytest.mark.parametrize("kind", ["nested", "arms", "facing", "any"])
@pytest.mark.parametrize("n", [1, 2, 5, 64, 65, 128, 131, 257, 1024, 1025])
def test_dof_gradient_of_all_torsion_forms(sys0, n, kind):
    """The DOF gradient, with and without E_intra, for torsions whose derivatives can and
    cannot be taken in the final conformer, at the edges of the pair ring (odd and even atom
    counts, one and several atoms a thread, words of 64 pairs, the largest ligand): against
    the oracle's FP64 Jacobian applied to the coordinate gradient.
    Tolerance: coordinates agree to 1e-13 A of each other, forces of pairs beyond 0.5 A
    therefore to 14 x 1e-13 / 0.5 = 3e-12 of themselves; a few hundred partners: 1e-9."""
    import torch
    ctx, _, _ = sys0
    rng = np.random.default_rng(n)
    dev = torch.device("cuda:0")
    for nrb in (0, 3, 9) if n <= 257 else (3,):
        lig = _chain(n, nrb, kind, rng)
        lid = ctx.add_ligand(lig)
        b = ctx.batch(np.full(3, lid))
        nrb = len(lig["rb_left"])
        d = np.concatenate([rng.uniform(-3, 3, (3, 3)), rng.uniform(-3, 3, (3, 3)),
                            rng.uniform(-0.3, 0.3, (3, nrb))], 1)
        for flags in (ff.F_INTER_SHIFTED | ff.F_INTRA, ff.F_INTER_SHIFTED):
            e = torch.empty((3, 4), dtype=torch.float64, device=dev)
            x = torch.empty((b.natoms, 3), dtype=torch.float64, device=dev)
            g = torch.empty(d.size, dtype=torch.float64, device=dev)
            b.score_dofs_dev(torch.tensor(d.ravel(), device=dev), e, xyz_out=x, gdof=g,
                             flags=flags | ff.F_GRAD)
            torch.cuda.synchronize()
            x, g, e = x.cpu().numpy(), g.cpu().numpy().reshape(3, -1), e.cpu().numpy()
            _, gx = b.score(x, ff.F_INTER_SHIFTED | ff.F_GRAD)
            for p in range(3):
                xp, h = x[p * n:(p + 1) * n], gx[p * n:(p + 1) * n].copy()
                posed = dict(lig, xs=xp[:, 0].copy(), ys=xp[:, 1].copy(), zs=xp[:, 2].copy())
                if flags & ff.F_INTRA:
                    want, gi = oracle.grad_intra(posed)
                    h += gi
                    assert e[p, 1] == pytest.approx(want, rel=1e-9, abs=1e-9)
                J = oracle.apply_config_jvp(_rows(lig), lig["rb_left"], lig["rb_right"], lig["rg_off"],
                                            lig["rg_atoms"], d[p])[2]
                scale = np.abs(J).sum(axis=(1, 2)) * np.abs(h).max()
                np.testing.assert_array_less(np.abs(g[p] - (J * h).sum(axis=(1, 2))), 1e-9 * scale + 1e-12)


@pytest.mark.parametrize("npose,iters", [(1, 1), (7, 30), (257, 12), (800, 5), (1793, 4), (2049, 2)])
@pytest.mark.parametrize("intra", [False, True])
def test_pooled_minimiser(sys0, npose, iters, intra):
    """The minimiser whose workgroups pool their poses' sweeps (one to seven poses a CU, one or
    several a workgroup, the rest from the queue) gives the one-wavefront form's points,
    energies and decisions bit for bit: ligands of 1, 4, 5, 64, 65 atoms and the library's, poses
    in contact, out of reach and too long; above its range the other form runs."""
    import torch
    from mmo_amd.minimize import Minimizer
    ctx, lig, _ = sys0
    rng = np.random.default_rng(npose)
    ligs = [lig] + synth.library(5) + [_chain(n, 3, "facing", rng) for n in (1, 4, 5, 64, 65)]
    ids = np.array([ctx.add_ligand(l) for l in ligs])
    pick = rng.integers(0, len(ligs), npose)
    b = ctx.batch(ids[pick])
    start = np.concatenate([np.concatenate([rng.uniform(-12, 12, 3), rng.uniform(-3, 3, 3),
                                            rng.uniform(-0.4, 0.4, len(ligs[k]["rb_left"]))]) for k in pick])
    start[::7] *= 4.0   # among them poses beyond the cutoff
    got = []
    for pooled in (0, 8):
        ctx.tune(min_pooled=pooled)
        mz = Minimizer(b, flags=ff.F_INTER_SHIFTED | (ff.F_INTRA if intra else 0), max_step=0.3)
        for _ in range(2):   # the second run starts from nothing of the first
            d = torch.tensor(start, device="cuda:0")
            e = mz.run(d, iters)
            torch.cuda.synchronize()
        got.append((e.cpu().numpy(), d.cpu().numpy(), mz.info()))
    ctx.tune(min_pooled=8)
    assert np.array_equal(got[0][0], got[1][0], equal_nan=True)
    assert np.array_equal(got[0][1], got[1][1], equal_nan=True)
    for k in got[0][2]:
        assert np.array_equal(got[0][2][k], got[1][2][k], equal_nan=True), k


@pytest.mark.parametrize("mode", ["grid", "direct"])
@pytest.mark.parametrize("chains,frames", [(1, 9), (40, 130)])
def test_chains_keep_round_energies(sys0, mode, chains, frames):
    """Chains that keep the E_intra of every round of 64 pairs and evaluate those a torsion
    changes follow the chains that evaluate all pairs: ligands without torsions, with no pairs,
    with less than a round, with one and with several mask words, groups of any atoms; in one
    run and in pieces, also through a graph.  Kept rounds hold pairs whose atoms turned
    together since: distances equal to rounding, 12 x 2^-52 of a pair's energy; the energies
    of these chains in contact agree to 1e-10 relative, the decisions are the same."""
    from mmo_amd import mc
    ctx, lig, _ = sys0
    rng = np.random.default_rng(chains)
    ligs = [lig] + synth.library(6) + [_chain(n, r, k, rng) for n, r, k in (
        (1, 0, "nested"), (5, 2, "nested"), (40, 0, "nested"), (64, 6, "facing"),
        (91, 9, "any"), (100, 12, "nested"))]
    probe_a, probe_q, types = synth.grid_types(ligs, 10)
    origin, gdims, gstep = synth.grid_spec((0.0, 0.0, 0.0), 64, 0.375)
    ctx.compute_grids(probe_a, probe_q, gstep, gdims, origin, copy_out=False)
    ids = np.array([ctx.add_ligand(l, types=t) for l, t in zip(ligs, types)])
    pick = np.arange(chains) % len(ligs)
    rot, pos = synth.random_rotations(rng, chains), rng.uniform(-1, 1, (chains, 3))

    def make():
        return mc.MonteCarlo(ctx, ids[pick], rot, pos, ff.INTERP if mode == "grid" else ff.SHIFTED,
                             frames, flags=mc.TWEAK_RBONDS | mc.INTRA_UFF | mc.HARD_ROI,
                             roi_center=(0.0, 0.0, 0.0), roi_r=8.0, seed=7)

    def run(how):
        m = make()
        if how == "pieces":
            m.run(1)
            m.run_graph(1, 3)
            m.run(frames - 4)
        else:
            m.run(frames)
        return m.state()
    ctx.tune(mc_keep_pairs=0)
    want = run("whole")
    ctx.tune(mc_keep_pairs=1)
    whole, pieces = run("whole"), run("pieces")
    for k in want:
        a, b, c = (np.asarray(s[k]) for s in (want, whole, pieces))
        assert np.array_equal(b, c, equal_nan=a.dtype.kind == "f"), k
        if a.dtype.kind == "f":
            np.testing.assert_allclose(b, a, rtol=1e-10, atol=1e-10, err_msg=k)
        else:
            assert np.array_equal(a, b), k


@pytest.mark.parametrize("n", [1, 64, 65, 128, 131])
@pytest.mark.parametrize("nrec", [1, 63, 64, 65, 577])
def test_plain_forms_at_slice_edges(n, nrec):
    """One pose against slices of 64 receptor atoms (one, a full one, one and a remainder, ten)
    with one, two and four ligand atoms a lane: energy, its parts and gradient in both modes."""
    _, rec = synth.config0()
    rng = np.random.default_rng(n + nrec)
    big = max(synth.library(24), key=lambda l: len(l["xs"]))
    keep = np.arange(min(n, len(big["xs"])))
    lig = {k: big[k][keep].copy() for k in ("xs", "ys", "zs", "q", "anum")}
    at = np.argsort(np.hypot(rec["xs"], rec["ys"]) + np.abs(rec["zs"]))[:nrec]
    part = {k: np.asarray(rec[k])[at].copy() for k in ("xs", "ys", "zs", "q", "anum")}
    ctx = ff.Context(0)
    ctx.set_receptor(part)
    x = _rows(lig) + rng.uniform(-1, 1, 3)
    lig.update(xs=x[:, 0].copy(), ys=x[:, 1].copy(), zs=x[:, 2].copy())
    for mode, shifted in ((ff.SHIFTED, True), (ff.GLOBAL, False)):
        s = inter_abs_sum(part, x, lig, shifted)
        e, el, vd = ctx.ene_inter(lig, mode, components=True)
        want, wel, wvd = oracle.ene_inter(part, lig, shifted=shifted, components=True)
        assert_energy([e, el, vd], [want, wel, wvd], [s, s, s], what="plain %d x %d" % (n, nrec))
        eg, g = ctx.ene_inter_grad(lig, mode)
        ref, gref = oracle.grad_inter(part, lig, shifted=shifted)
        assert_energy(eg, ref, s, what="plain gradient's energy")
        assert_grad(g, gref, what="plain gradient %d x %d" % (n, nrec))


@pytest.mark.parametrize("npose", [1, 16, 257])
def test_dof_totals(sys0, npose):
    """Totals and gradients of poses within and beyond a length limit, with radii equal to it,
    infinite and NaN, are what the same torch operations give."""
    import torch
    ctx, lig, _ = sys0
    rng = np.random.default_rng(npose)
    ligs = [lig, _chain(5, 0, "nested", rng), _chain(40, 7, "nested", rng)]
    b = ctx.batch(np.array([ctx.add_ligand(l) for l in ligs])[np.arange(npose) % 3])
    dev = torch.device("cuda:0")
    e = torch.tensor(rng.normal(size=(npose, 4)), device=dev)
    rad = torch.tensor(rng.choice([3.0, 12.0, np.nextafter(12.0, 13.0), np.inf, np.nan, 40.0], npose), device=dev)
    g = torch.tensor(rng.normal(size=int(b.dof_off[-1])), device=dev)
    e[0, 0] = float("nan")
    pose = torch.repeat_interleave(torch.arange(npose), torch.tensor(np.diff(b.dof_off).astype(np.int64))).to(dev)
    beyond = rad > 12.0
    want = torch.where(beyond, torch.full_like(rad, float("inf")), e[:, 0] + e[:, 1])
    gwant = g.masked_fill(beyond[pose], 0.0)
    total = torch.empty_like(rad)
    b.dof_totals_dev(e, rad, 12.0, total)
    assert torch.equal(total.nan_to_num(7.0, 8.0), want.nan_to_num(7.0, 8.0))
    total.zero_()
    b.dof_totals_dev(e, rad, 12.0, total, g)
    assert torch.equal(total.nan_to_num(7.0, 8.0), want.nan_to_num(7.0, 8.0)) and torch.equal(g, gwant)


@pytest.mark.parametrize("dims,ntypes", [((61, 45, 83), 12), ((128, 128, 64), 3), ((700, 701, 2), 3),
                                         ((9, 7, 45000), 1)])
def test_large_grids_reach_the_host_whole(sys0, dims, ntypes):
    """Grids of 10 MiB and more, computed in one, two or four slabs and taken by several threads
    in pieces, are bit for bit the grids of one type at a time (below that size: one launch, one
    copy): slabs of unequal and of single bricks, pieces that end a type early, a region of
    interest."""
    ctx, _, _ = sys0
    rng = np.random.default_rng(ntypes)
    anum, q = rng.choice([1, 6, 7, 8], ntypes).astype(np.int32), rng.uniform(-0.5, 0.5, ntypes)
    step = 0.5 if dims[2] < 1000 else 0.001
    origin = -0.5 * step * np.asarray(dims, dtype=float)
    kw = dict(roi_center=(0.0, 0.0, 0.0), roi_r=11.0)
    whole = ctx.compute_grids(anum, q, step, dims, origin, **kw)
    assert whole.nbytes >= 10 << 20
    cut = dims[2] if ntypes > 1 else dims[2] // 3 // 4 * 4   # a multiple of the brick
    for t in range(ntypes):
        one = ctx.compute_grids(anum[t:t + 1], q[t:t + 1], step, (dims[0], dims[1], cut), origin, **kw)
        assert one.nbytes < 10 << 20
        assert np.array_equal(one[0], whole[t][:cut]) and np.any(one != 0)


@pytest.mark.parametrize("chains,frames", [(1, 7), (257, 40), (1100, 6), (3072, 4)])
def test_pooled_chains(sys0, chains, frames):
    """Direct chains whose workgroups pool their sweeps (one to twelve chains a CU) have the
    states of chains that each sweep alone, bit for bit, in one run, in pieces, through a graph
    and one launch per ligand: ligands of 1, 4, 5, 64, 65 atoms and the library's, chains that
    leave the region, chains that end too long."""
    from mmo_amd import mc
    ctx, lig, _ = sys0
    rng = np.random.default_rng(chains)
    long = _chain(18, 6, "nested", rng)
    ligs = [lig] + synth.library(4) + [_chain(n, min(n - 1, 2) if n > 4 else 0, "nested", rng)
                                       for n in (1, 4, 5, 64, 65)] + [long]
    ids = np.array([ctx.add_ligand(l) for l in ligs])
    pick = rng.integers(0, len(ligs), chains)
    rot, pos = synth.random_rotations(rng, chains), rng.uniform(-6, 6, (chains, 3))
    got = []
    for pool, how in ((0, "run"), (12, "run"), (12, "pieces"), (12, "ligand")):
        ctx.tune(mc_pool=pool)
        m = mc.MonteCarlo(ctx, ids[pick], rot, pos, ff.SHIFTED, frames,
                          flags=mc.TWEAK_RBONDS | mc.INTRA_UFF | mc.HARD_ROI,
                          roi_center=(0.0, 0.0, 0.0), roi_r=7.0, seed=11)
        if how == "run":
            m.run(frames)
        elif how == "ligand":
            m.run_per_ligand(frames)
        else:
            m.run(1)
            m.run_graph(1, 2)
            m.run(frames - 3)
        got.append((m.state(), m.coords()))
    ctx.tune(mc_pool=12)
    for st, xyz in got[1:]:
        for k, v in got[0][0].items():
            a, b = np.asarray(v), np.asarray(st[k])
            assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), k
        assert all(np.array_equal(x, y) for x, y in zip(got[0][1][1], xyz[1]))
