"""A forward batch whose line-aligned walk would pass 2^32 work-items while its interior
cells do not: 641 shots of 32x460x460 (one shot exceeds the Infinity Cache, so all shots
share a launch).  It runs, and a shot of it equals its own single-shot run bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_batch_beyond_the_aligned_walk(gpu_lib):
    from elastic_fm_vp_vs_rho_amd.propagator import Grid, Propagator, ShotBatch
    nx, ny, nz, S, nt = 32, 460, 460, 641, 3
    aligned = -(-((nz - 4) * nx + 27) // 128) * 128 * (ny - 4) * S
    interior = -(-((nz - 4) * (nx - 4)) // 128) * 128 * (ny - 4) * S
    assert interior < 1 << 32 < aligned
    if torch.cuda.mem_get_info()[0] < 175 * 10 ** 9:
        pytest.skip("needs 175 GB of free GPU memory")
    grid = Grid(nx, ny, nz, 10.0, 1e-3, (0,) * 6)
    cp = {k: np.zeros(n, np.float32) for k, n in
          (("ax", nx), ("bx", nx), ("ay", ny), ("by", ny), ("az", nz), ("bz", nz))}
    rng = np.random.default_rng(1)
    rho = torch.full(grid.shape, 2200.0, device="cuda")
    mu = torch.full(grid.shape, 2200.0 * 1300.0 ** 2, device="cuda")
    src = np.stack([rng.integers(2, n - 2, S) for n in (nx, ny, nz)], 1)
    src[-1] = (nx - 3, ny - 3, nz - 3)                      # the last interior cell of the last shot
    rec = src[:, None, :] + np.array([[0, 0, 0], [-1, 0, 0]])
    rec[..., 0] = np.maximum(rec[..., 0], 0)
    m6, wav = rng.uniform(0.5, 1, (S, 6)), np.ones((S, nt), np.float32)
    batch = lambda i: ShotBatch(grid, src[i], m6[i], wav[i], np.full(len(i), nt), rec[i], cp, device="cuda")
    prop = Propagator(grid, mu, mu, rho, batch(np.arange(S)))
    g, st = prop.forward()
    for s in (0, S // 2, S - 1):
        g1, st1 = Propagator(grid, mu, mu, rho, batch(np.array([s]))).forward()
        assert float(g1.abs().max()) > 0
        assert torch.equal(g1[0], g[s])
        assert torch.equal(st1.fields[:, 0], st.fields[:, s])
