"""Monte Carlo runs that a caller's graph captures."""
import numpy as np
import pytest

from mmo_amd import ff, mc, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("new_table", [False, True])
def test_captured_run_then_eager_run(new_table):
    """A run that is only captured leaves the chains (and the pair energies they keep) as they
    were: an eager run after it, then the graph, give the states of three eager runs, for chains
    just made and for chains whose parameter table has been set again."""
    import torch
    _, rec = synth.config0()
    ligs = synth.library(6)

    def chains(ctx, ids):
        rng = np.random.default_rng(2)
        return mc.MonteCarlo(ctx, ids, synth.random_rotations(rng, len(ids)),
                             rng.uniform(-1, 1, (len(ids), 3)), ff.SHIFTED, 60,
                             flags=mc.TWEAK_RBONDS | mc.INTRA_UFF | mc.HARD_ROI,
                             roi_center=(0.0, 0.0, 0.0), roi_r=8.0, seed=5)
    states = []
    for captured in (False, True):
        ctx = ff.Context(0)
        ctx.set_receptor(rec)
        ids = np.array([ctx.add_ligand(l) for l in ligs])
        m = chains(ctx, ids)
        if new_table:
            ctx.set_uff_table({a: (x, d) for a, x, d in TABLE})
            ctx.set_receptor(rec)
            other = chains(ctx, ids)   # brings the registry to the device again
            other.run(1)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        if captured:
            with torch.cuda.graph(graph):
                m.run(20, stream=torch.cuda.current_stream())
        m.run(20)
        torch.cuda.synchronize()
        for _ in range(2):
            if captured:
                graph.replay()
            else:
                m.run(20)
            torch.cuda.synchronize()
        states.append((m.state(), m.coords()))
    for k, v in states[0][0].items():
        a, b = np.asarray(v), np.asarray(states[1][0][k])
        if a.dtype.kind != "f" or not new_table:
            assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), k
        else:   # the graph sums all pairs anew: distances equal to rounding, as elsewhere 1e-10
            np.testing.assert_allclose(b, a, rtol=1e-10, atol=1e-10, err_msg=k)
    assert all(np.allclose(x, y, rtol=0, atol=1e-9) for x, y in zip(states[0][1][1], states[1][1][1]))


TABLE = [(0, 0.0, 0.0), (1, 2.886, 0.044), (6, 3.851, 0.105), (7, 3.660, 0.069), (8, 3.500, 0.060),
         (9, 3.364, 0.050), (12, 3.021, 0.111), (15, 4.147, 0.305), (16, 4.035, 0.274),
         (17, 3.947, 0.227), (35, 4.189, 0.251), (53, 4.500, 0.339)]
