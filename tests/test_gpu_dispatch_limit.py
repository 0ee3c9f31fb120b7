"""A forward batch whose line-aligned walk would pass 2^32 work-items while its interior
cells do not: 641 shots of 32x460x460 (one shot exceeds the Infinity Cache, so all shots
share a launch).  It runs, and a shot of it equals its own single-shot run bit for bit.

And a reverse loop whose adjoint sweep fills a dispatch to 8 blocks of the limit, so that
the blocks for its receivers no longer fit."""
import ctypes

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


def test_reverse_loop_at_the_dispatch_limit(gpu_lib):
    """(256, 1, 1, 8) blocks on rows of 10 cells: 127 shots of 132104 blocks are 2^24 - 8.  The
    images equal those of the default tile to the roundings a kernel's other instance may
    make: 8·2^-24 a term over 2 iterations."""
    from elastic_fm_vp_vs_rho_amd import _capi, autotune
    from elastic_fm_vp_vs_rho_amd.propagator import Grid, Propagator, ShotBatch, _ptr, _stream
    nx, ny, nz, S, nt, W, nrec = 10, 2700, 49, 127, 3, 1, 20
    blocks = nz * (ny - 4) * S
    assert blocks * 256 < 1 << 32 <= (blocks + -(-S * nrec // 256)) * 256
    grid = Grid(nx, ny, nz, 10.0, 1e-3, (0,) * 6)
    cp = {k: np.zeros(n, np.float32) for k, n in
          (("ax", nx), ("bx", nx), ("ay", ny), ("by", ny), ("az", nz), ("bz", nz))}
    rng = np.random.default_rng(2)
    src = np.stack([rng.integers(3, n - 3, S) for n in (nx, ny, nz)], 1)
    along = np.arange(nrec) * 130 + 60
    rec = np.stack([np.broadcast_to(np.stack([np.full(nrec, nx // 2), along, np.full(nrec, 5)], 1), (S, nrec, 3))])[0]
    batch = ShotBatch(grid, src, rng.uniform(0.5, 1, (S, 6)), np.ones((S, nt), np.float32), np.full(S, nt), rec, cp,
                      device="cuda")
    rho = torch.full(grid.shape, 2200.0, device="cuda")
    mu = torch.full(grid.shape, 2200.0 * 1300.0 ** 2, device="cuda")
    prop = Propagator(grid, mu, mu, rho, batch)
    d, m, sh, by = prop.dims(), prop.medium(), batch.struct(), ctypes.byref
    gen = torch.Generator(device="cuda").manual_seed(3)
    res = torch.randn((S, 3, nt, nrec), device="cuda", generator=gen)
    per = gpu_lib.efm_border_floats(by(d), W)
    assert per > 0
    from tests.test_gpu_reverse_pairs import _faces
    vols = rng.standard_normal((nt * 3,) + grid.shape).astype(np.float32)
    step = torch.as_tensor(np.concatenate([_faces(v, W) for v in vols]), device="cuda")
    assert step.numel() == nt * per
    borders = step.expand(S, -1).contiguous()
    images = []
    was = [autotune.get_tile(k) for k in range(2)]
    try:
        for tile in ((256, 1, 1, 8), autotune.DEFAULT_TILE):
            for k in range(2):
                autotune.set_tile(k, tile)
            fwd, adj = prop.new_wavefield(), prop.new_wavefield()
            for w in (fwd, adj):
                for k in range(9):
                    w.fields[k].normal_(generator=gen.manual_seed(10 + k))
            vpres = torch.zeros(S * 3 * grid.N, device="cuda")
            g3 = [torch.zeros((S,) + grid.shape, device="cuda") for _ in range(3)]
            _capi.check(gpu_lib.efm_backward_remake_ref(
                by(d), by(m), by(sh), by(fwd.struct()), _ptr(vpres), _ptr(borders), W, by(adj.struct()), _ptr(res),
                1e-3, 10.0, 10.0, 10.0, *[_ptr(t) for t in g3], _stream()), "remake")
            torch.cuda.synchronize()
            images.append([t[[0, S // 2, S - 1]].cpu() for t in g3])
            del fwd, adj, vpres, g3
    finally:
        for k in range(2):
            autotune.set_tile(k, was[k])
    for a, b in zip(*images):
        assert float(b.abs().max()) > 0
        assert float((a - b).abs().max()) <= 2 * 8 * 2.0 ** -24 * float(b.abs().max())
