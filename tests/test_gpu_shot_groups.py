"""A forward batch too large for the Infinity Cache advances its shots group by
group through all steps; each shot's seismograms and final state equal its own
single-shot run, whichever entry point drives the loop."""
import numpy as np
import pytest
import torch

from tests.gpu_helpers import grid_of
from tests.problems import tiny

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fuse", [True, False])
def test_grouped_batch_equals_single_shots(gpu_lib, fuse):
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    nt, S = 14, 13        # a 92^3 shot takes 33 MB with its CPML slabs: 13 make groups of 7 and 6
    p = tiny(n=(92, 92, 92), nt=nt, W=4, seed=5, nrec=6)
    grid = grid_of(p)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    med = f(p.lam), f(p.mu), f(p.rho)
    rng = np.random.default_rng(7)
    src = rng.integers(30, 60, (S, 3))
    m6 = rng.uniform(-1, 1, (S, 6))
    nts = rng.integers(nt // 2, nt + 1, S)
    rec = src[:, None, :] + rng.integers(-4, 5, (S, 6, 3))
    wav = np.repeat(np.asarray(p.wavelet, np.float32)[None], S, 0) + 1.0
    batch = lambda i: ShotBatch(grid, src[i], m6[i], wav[i], nts[i], rec[i], p.cp, fuse_receivers=fuse)
    prop = Propagator(grid, *med, batch(np.arange(S)))
    g, st = prop.forward()
    states = prop.record(strategy="store")
    gg, gst = Propagator(grid, *med, batch(np.arange(S)), graphs=True).forward(graph_chunk=5)
    assert torch.equal(gg, g) and torch.equal(gst.fields, st.fields)
    assert torch.equal(states["gathers"], g)
    for s in range(S):
        one = Propagator(grid, *med, batch(np.array([s])))
        g1, st1 = one.forward()
        assert float(g1.abs().max()) > 0
        assert torch.equal(g1[0], g[s])
        assert torch.equal(st1.fields[:, 0], st.fields[:, s]) and torch.equal(st1.psi_y[0], st.psi_y[s])
        assert torch.equal(st.fields[:3, s], states["states"][int(nts[s])].v[:, s])
