"""The reverse sweep images two steps at a time; the gradient must not notice
where the pairs are cut: by the tape's segments (odd and even starts and lengths,
one step alone), by each shot's own record length, or by the receiver mode."""
import numpy as np
import pytest
import torch

from oracle import elastic_fp64 as O
from tests.gpu_helpers import grid_of
from tests.problems import rel_l2, tiny

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,nts,W", [((35, 19, 17), (25, 24, 1), 4),      # odd and even ends, a one-step record
                                         ((70, 11, 12), (24, 23, 22), 3)])    # rows of more than a wave
def test_gradient_does_not_depend_on_how_pairs_are_cut(gpu_lib, shape, nts, W):
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    nt, S = max(nts), len(nts)
    p = tiny(n=shape, nt=nt, W=W, seed=17, nrec=8)
    grid = grid_of(p)
    rng = np.random.default_rng(2)
    src = np.stack([rng.integers(5, n - 5, S) for n in shape], 1)
    rec = np.clip(src[:, None, :] + rng.integers(-3, 4, (S, 8, 3)), 2, np.array(shape) - 3)
    m6 = rng.uniform(-1, 1, (S, 6))
    wav = p.wavelet + 1.0                       # acting from the first step on
    obs = 1e-8 * rng.standard_normal((S, 3, nt, 8)).astype(np.float32)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    ref = {"lam": 0.0, "mu": 0.0, "rho": 0.0}
    for s in range(S):
        hist, n = [], nts[s]
        g, _ = O.forward(p.medium(), p.cpml(), p.c, tuple(src[s]), m6[s], wav[:n], rec[s], n, history=hist)
        r, _ = O.misfit(g, obs[s, :, :n])
        a = O.exact_adjoint(p.medium(), p.cpml(), p.c, tuple(src[s]), wav[:n], rec[s], n, r, hist)
        for k in ref:
            ref[k] = ref[k] + a[k]
    out = {}
    for fuse in (True, False):
        batch = ShotBatch(grid, src, m6, [wav] * S, nts, rec, p.cp, fuse_receivers=fuse)
        prop = Propagator(grid, f(p.lam), f(p.mu), f(p.rho), batch)
        for K in (None, 1, 2, 3, 4, 7):
            kw = dict(strategy="store") if K is None else dict(strategy="checkpoint", K=K)
            out[fuse, K] = prop.gradient(f(obs), **kw)[2:5]
        out[fuse, "hybrid"] = prop.gradient(f(obs), strategy="hybrid", m=9, K=5)[2:5]
    # float32 against the float64 oracle: 25 steps of 1-ulp roundings stay below 1e-5
    for k, got in zip(("lam", "mu", "rho"), out[True, None]):
        assert rel_l2(got.double().cpu().numpy(), ref[k]) < 1e-5, k
    for key, grads in out.items():
        assert all(torch.equal(a, b) for a, b in zip(grads, out[True, None])), key
