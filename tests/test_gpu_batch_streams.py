"""Calls on one batch that overlap: on several streams, in captured graphs, and a first call
that is captured."""
import numpy as np
import pytest

from mmo_amd import ff, synth

pytestmark = pytest.mark.gpu
FLAGS = ff.F_INTER_SHIFTED | ff.F_INTRA


@pytest.fixture(scope="module")
def setup():
    _, rec = synth.config0()
    ctx = ff.Context(0)
    ctx.set_receptor(rec)
    ligs = synth.library(8)
    ids = np.array([ctx.add_ligand(l) for l in ligs])
    return ctx, ligs, ids


def _batch(setup, npose):
    ctx, ligs, ids = setup
    pick = np.arange(npose) % len(ligs)
    return ctx.batch(ids[pick]), [ligs[k] for k in pick]


def _poses(ligs, seed):
    import torch
    rng = np.random.default_rng(seed)
    x = [np.stack([l["xs"], l["ys"], l["zs"]], 1) @ r.T + rng.uniform(-3, 3, 3)
         for l, r in zip(ligs, synth.random_rotations(rng, len(ligs)))]
    return torch.tensor(np.concatenate(x), device="cuda:0")


def _buffers(b, grad):
    import torch
    e = torch.full((b.npose, 4), -7.0, dtype=torch.float64, device="cuda:0")
    return e, torch.full((b.natoms, 3), -7.0, dtype=torch.float64, device="cuda:0") if grad else None


@pytest.mark.parametrize("streams", [2, 7])
@pytest.mark.parametrize("grad", [False, True])
def test_one_batch_on_several_streams(setup, streams, grad):
    """Interleaved calls on one batch, each stream with its own poses and outputs (more streams
    than a batch keeps buffers for, too), give what the calls give alone, bit for bit."""
    import torch
    b, ligs = _batch(setup, 600)
    x = [_poses(ligs, k) for k in range(streams)]
    flags = FLAGS | (ff.F_GRAD if grad else ff.F_COMPONENTS)
    want = []
    for k in range(streams):
        e, g = _buffers(b, grad)
        b.score_dev(x[k], e, g, flags=flags)
        torch.cuda.synchronize()
        want.append((e, g))
    ss = [torch.cuda.Stream() for _ in range(streams)]
    got = [[_buffers(b, grad) for _ in range(12)] for _ in range(streams)]
    torch.cuda.synchronize()
    for call in range(12):
        for k in range(streams):
            e, g = got[k][call]
            b.score_dev(x[k], e, g, flags=flags, stream=ss[k])
    torch.cuda.synchronize()
    for k in range(streams):
        for e, g in got[k]:
            assert torch.equal(e, want[k][0]) and (not grad or torch.equal(g, want[k][1]))


def test_dof_energies_on_two_streams(setup):
    """Energies of DOF vectors with coordinate buffers of their own, on two streams."""
    import torch
    b, ligs = _batch(setup, 300)
    rng = np.random.default_rng(3)
    ss = [torch.cuda.Stream() for _ in range(2)]
    d = [torch.tensor(np.concatenate([np.concatenate([
        rng.uniform(-2, 2, 3), rng.uniform(-3, 3, 3), rng.uniform(-.3, .3, len(l["rb_left"]))])
        for l in ligs]), device="cuda:0") for _ in ss]
    x = [torch.empty(b.natoms, 3, dtype=torch.float64, device="cuda:0") for _ in ss]
    want = []
    for k in range(2):
        e, _ = _buffers(b, False)
        b.score_dofs_dev(d[k], e, xyz_out=x[k], flags=FLAGS)
        torch.cuda.synchronize()
        want.append(e)
    got = [[_buffers(b, False)[0] for _ in range(12)] for _ in ss]
    torch.cuda.synchronize()
    for call in range(12):
        for k in range(2):
            b.score_dofs_dev(d[k], got[k][call], xyz_out=x[k], flags=FLAGS, stream=ss[k])
    torch.cuda.synchronize()
    assert all(torch.equal(e, want[k]) for k in range(2) for e in got[k])


def test_captured_calls(setup):
    """A batch whose first call is captured, then captured again into a second graph: both
    graphs replay at once on two streams, with eager calls between, and follow their inputs."""
    import torch
    ctx = setup[0]
    warm, ligs = _batch(setup, 400)
    e, _ = _buffers(warm, False)
    warm.score_dev(_poses(ligs, 0), e, flags=FLAGS)   # the registry is on the device
    torch.cuda.synchronize()
    b, ligs = _batch(setup, 400)
    ins = [_poses(ligs, 10 + k) for k in range(2)]
    outs = [_buffers(b, True) for _ in range(2)]
    graphs = []
    for k in range(2):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            b.score_dev(ins[k], outs[k][0], outs[k][1], flags=FLAGS | ff.F_GRAD)
        graphs.append(graph)
    ss = [torch.cuda.Stream() for _ in range(2)]
    for round_ in range(4):
        new = [_poses(ligs, 20 + 2 * round_ + k) for k in range(2)]
        want = []
        for k in range(2):
            ins[k].copy_(new[k])
            we, wg = _buffers(b, True)
            b.score_dev(new[k], we, wg, flags=FLAGS | ff.F_GRAD)
            want.append((we, wg))
        torch.cuda.synchronize()
        for _ in range(3):
            for k in range(2):
                with torch.cuda.stream(ss[k]):
                    graphs[k].replay()
            e, g = _buffers(b, True)
            b.score_dev(new[0], e, g, flags=FLAGS | ff.F_GRAD)
        torch.cuda.synchronize()
        assert torch.equal(e, want[0][0])
        for k in range(2):
            assert torch.equal(outs[k][0], want[k][0]) and torch.equal(outs[k][1], want[k][1])
    assert ctx is b.ctx


def test_captured_first_call_of_the_sub_block_kernel(setup):
    """A batch made with pose_sweep = 0 has its slot order: its first call can be captured."""
    import torch
    ctx = setup[0]
    ctx.tune(pose_sweep=0)
    try:
        b, ligs = _batch(setup, 300)
        x = _poses(ligs, 1)
        (e, g), (we, wg) = _buffers(b, True), _buffers(b, True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            b.score_dev(x, e, g, flags=FLAGS | ff.F_GRAD)
        for k in range(3):
            x.copy_(_poses(ligs, 2 + k))
            b.score_dev(x, we, wg, flags=FLAGS | ff.F_GRAD)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(e, we) and torch.equal(g, wg)
    finally:
        ctx.tune(pose_sweep=1)
