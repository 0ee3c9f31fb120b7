"""Receivers sampled and injected by the waves that hold their cells, against the kernels
that take one thread per receiver: lists below, at and above a wave's 64 lanes (part-empty
waves take shorter shares), unused entries, a whole row of receivers, cells in the guard
rows (never sampled by the sweep), each block mapping."""

import ctypes

import numpy as np
import pytest
import torch

from elastic_fm_vp_vs_rho_amd import _capi
from tests.gpu_helpers import grid_of
from tests.problems import tiny

pytestmark = pytest.mark.gpu
TILES = [(128, 1, 1, 16), (128, 1, 2, 16), (64, 4, 2, 8), (64, 2, 1, 0)]


@pytest.fixture(autouse=True)
def _restore_tiles():
    lib, was = _capi.lib(), []
    for k in range(4):
        v = [ctypes.c_int() for _ in range(4)]
        _capi.check(lib.efm_get_tile(k, *[ctypes.byref(x) for x in v]), "efm_get_tile")
        was.append([x.value for x in v])
    yield
    for k, t in enumerate(was):
        _capi.check(lib.efm_set_tile(k, *t), "efm_set_tile")


@pytest.mark.parametrize("nrec,tile", [(1, 0), (50, 0), (63, 1), (64, 2), (65, 3), (200, 0), (200, 2)])
def test_wave_receivers_equal_a_thread_per_receiver(gpu_lib, nrec, tile):
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    for k in range(4):
        _capi.check(_capi.lib().efm_set_tile(k, *TILES[tile]), "efm_set_tile")
    n, nts, S = (73, 21, 20), (30, 17), 2
    p = tiny(n=n, nt=nts[0], W=4, seed=5, nrec=1)
    rng = np.random.default_rng(nrec)
    cells = np.stack(np.meshgrid(np.arange(2, 71), np.arange(2, 19), np.arange(2, 18), indexing="ij"), -1).reshape(-1, 3)
    rec = np.stack([cells[rng.permutation(len(cells))[:nrec]] for _ in range(S)])    # a cell at most once
    src = np.array([(20, 10, 9), (40, 8, 8)])
    if nrec > 60:
        rec[:, :40] = [(x, 10, 9) for x in range(10, 50)]
        rec[:, 40:] = np.where((rec[:, 40:, 1:] == (10, 9)).all(-1, keepdims=True), -1, rec[:, 40:])
        rec[0, 45] = -1
        if nrec == 200:
            rec[1, 46] = (30, 10, 1)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    obs = f(1e-8 * rng.standard_normal((S, 3, nts[0], nrec)))
    out = []
    for fused in (True, False):
        batch = ShotBatch(grid_of(p), src, np.ones((S, 6)), [p.wavelet] * S, nts, rec, p.cp,
                          fuse_receivers=fused)
        prop = Propagator(grid_of(p), f(p.lam), f(p.mu), f(p.rho), batch)
        g, _ = prop.forward()
        guard = torch.as_tensor((rec[..., 2] == 1)[:, None, None, :], device="cuda")
        out.append((torch.where(guard, torch.zeros((), device="cuda"), g),
                    *(prop.gradient(obs, strategy="store")[2:5] if nrec < 200 else ())))
    assert nrec == 1 or float(out[0][0].abs().max()) > 0     # the lone cell lies beyond the wave
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_injection_adds_a_long_list_in_order(gpu_lib):
    """Every receiver's residual reaches its cell, several on one cell included: the
    gradient with each of 160 receivers listed against the sum of their residuals on 80
    cells (float32 sums of at most three terms: a few roundings, 1e-6 of the gradient)."""
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    from tests.problems import rel_l2
    p = tiny(n=(73, 21, 20), nt=24, W=4, seed=5, nrec=1)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    one = np.array([(x, y, 9) for y in (8, 12) for x in range(12, 52)])
    grads = []
    for rec, q in ((np.concatenate([one, one]), 160), (one, 80)):
        batch = ShotBatch(grid_of(p), [(20, 10, 9)], np.ones((1, 6)), [p.wavelet], [24], [rec], p.cp)
        prop = Propagator(grid_of(p), f(p.lam), f(p.mu), f(p.rho), batch)
        rng = np.random.default_rng(3)
        r = 1e-8 * rng.standard_normal((1, 3, 24, 160)).astype(np.float32)
        if q == 80:
            r = r[..., :80] + r[..., 80:]
        grads.append(prop.backprop(prop.record(None, "store", None), f(r))[:3])
    for a, b in zip(*grads):
        assert rel_l2(a.double().cpu().numpy(), b.double().cpu().numpy()) < 1e-6


@pytest.mark.parametrize("tile", [0, 1, 3])
@pytest.mark.parametrize("n", [(27, 70, 61), (13, 260, 33), (63, 33, 55)])
def test_many_cells_in_short_rows_equal_single_shots(gpu_lib, n, tile):
    """A large batch on a narrow grid walks only the interior cells of each plane; every
    shot's seismograms, wavefield and saved borders equal its own run's."""
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    for k in range(4):
        _capi.check(_capi.lib().efm_set_tile(k, *TILES[tile]), "efm_set_tile")
    nt, S, W, nrec = 12, 11, 2, 70
    assert np.prod(n) < 1 << 20 <= np.prod(n) * S
    p = tiny(n=n, nt=nt, W=W, seed=5, nrec=1)
    rng = np.random.default_rng(n[0])
    c = np.array(n) // 2
    rec = np.stack([rng.integers(2, n[0] - 2, (S, nrec)), c[1] + rng.integers(-3, 4, (S, nrec)),
                    c[2] + rng.integers(-3, 4, (S, nrec))], -1)
    rec[:, 0] = c
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    wav = np.repeat(np.asarray(p.wavelet, np.float32)[None], S, 0) + 1.0

    def run(i):
        batch = ShotBatch(grid_of(p), [c] * len(i), np.ones((len(i), 6)), wav[i], [nt] * len(i), rec[i], p.cp)
        prop = Propagator(grid_of(p), f(p.lam), f(p.mu), f(p.rho), batch)
        borders = prop.border_buffer(W)
        g, st = prop.forward(borders=borders, W=W)
        return g, st.fields, borders

    g, st, borders = run(np.arange(S))
    for s in (0, 5, S - 1):
        g1, st1, b1 = run(np.array([s]))
        assert float(g1.abs().max()) > 0
        assert n[0] > 60 or float(b1.abs().max()) > 0      # the wave stays clear of the widest grid's borders
        assert torch.equal(g1[0], g[s])
        assert torch.equal(st1[:, 0], st[:, s]) and torch.equal(b1[0], borders[s])
