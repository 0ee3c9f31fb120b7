"""The shared launches of the reference-style reverse loop against its separate ones: a
run over all iterations (adjoint and reconstruction sweeps in pairs, images one iteration
late, borders restored by the velocity sweep) against the same iterations one call each,
where the reconstruction's velocity sweep, border restore, zeroing and images are launches
of their own.  Random states, guard cells included, random border values, records that end
early, receivers in the guard rows and on one cell, CPML narrower than the guard layer,
every block mapping.  And the forward loop's border save beside the next stress sweep
against one step per call.

Both sides form the same float32 products; the compiler may fuse a multiply and an add
differently in the two kernels, and receivers that share a cell add in any order: up to
some eight roundings of 2^-24 in a cell's term of each of the 11 iterations.  Bound:
11·8·2^-24 of the largest value of each image.
"""

import ctypes

import numpy as np
import pytest
import torch

from elastic_fm_vp_vs_rho_amd import _capi, model
from elastic_fm_vp_vs_rho_amd.propagator import Grid, Propagator, ShotBatch, _ptr, _stream

pytestmark = pytest.mark.gpu
H, NT, DT = 2, 12, 1e-3
BOUND = (NT - 1) * 8 * 2.0 ** -24
by = ctypes.byref


def _prop(nx, ny, nz, W, S, nts, free_top, fuse):
    rng = np.random.default_rng(nx + 7 * ny + S)
    grid = Grid.make(nx, ny, nz, 10.0, DT, W, free_top=free_top)
    prof = model.cpml_coefficients(W, 12.0, DT, 10.0, 3500.0, nx, ny, nz, free_top=free_top)
    cpml = {k: np.stack([prof[k]] * S) for k in prof}
    src = np.stack([rng.integers(W + 2, n - W - 2, S) for n in (nx, ny, nz)], 1)
    rec = np.stack([rng.integers(H, n - H, (S, 9)) for n in (nx, ny, nz)], 2)
    rec[:, 1] = rec[:, 0]                                    # two receivers on one cell
    rec[:, 2] = (nx // 2, ny // 2, 1)                        # in the top guard rows
    rec[:, 3] = (nx // 2 + 1, ny // 2, 0)
    wav = rng.standard_normal((S, NT)).astype(np.float32)
    batch = ShotBatch(grid, src, rng.standard_normal((S, 6)), wav, np.asarray(nts), rec, cpml, device="cuda",
                      fuse_receivers=fuse)
    u = lambda lo, hi: torch.as_tensor(rng.uniform(lo, hi, grid.shape).astype(np.float32), device="cuda")
    rho = u(2000, 2400)
    vs = u(1200, 1400)
    mu = rho * vs * vs
    return Propagator(grid, mu * u(1.0, 1.3), mu, rho, batch), batch, rng


def _state(prop, rng, scale):
    w = prop.new_wavefield()
    for t in (w.fields, w.psi_x, w.psi_y, w.psi_z):
        t.copy_(torch.as_tensor(scale * rng.standard_normal(t.shape).astype(np.float32)))
    return w


def _faces(v, W):
    """Border values of a (ny, nz, nx) volume in the buffer's order."""
    ny, nz, nx = v.shape
    return np.concatenate([a.ravel() for a in (
        v[:, :, W:W + H], v[:, :, nx - W - H:nx - W], v[:, H:2 * H, :], v[:, nz - W - H:nz - W, :],
        v[W:W + H], v[ny - W - H:ny - W])])


CASES = [
    # nx, ny, nz, W, record lengths, free top, fused receivers, tiles (stress, velocity)
    (41, 23, 22, 6, (NT,), True, True, None),
    (24, 21, 26, 4, (NT, NT - 5, 3), False, True, None),
    (24, 21, 26, 4, (NT, NT - 5), True, False, ((64, 2, 1, 0), (64, 4, 2, 8))),
    (70, 20, 19, 2, (NT - 1, NT), True, True, ((128, 1, 2, 16), (64, 1, 1, 0))),
    (17, 18, 19, 1, (NT,), False, True, None),
]


def _with_tiles(tiles):
    lib = _capi.lib()
    for k, t in enumerate(tiles or ()):
        _capi.check(lib.efm_set_tile(k, *t), "efm_set_tile")


@pytest.fixture(autouse=True)
def _restore_tiles():
    lib, was = _capi.lib(), []
    for k in range(2):
        v = [ctypes.c_int() for _ in range(4)]
        _capi.check(lib.efm_get_tile(k, *[by(x) for x in v]), "efm_get_tile")
        was.append([x.value for x in v])
    yield
    _with_tiles(was)


@pytest.mark.parametrize("case", CASES)
def test_paired_launches_equal_single_iterations(case):
    nx, ny, nz, W, nts, free_top, fuse, tiles = case
    _with_tiles(tiles)
    S, L = len(nts), _capi.lib()
    images = []
    for ranges in ([(0, NT - 1)], [(i, 1) for i in range(NT - 1)], [(0, 4), (4, 0), (4, NT - 5)]):
        prop, batch, rng = _prop(nx, ny, nz, W, S, nts, free_top, fuse)
        d, m, sh = prop.dims(), prop.medium(), batch.struct()
        fwd, adj = _state(prop, rng, 1e-3), _state(prop, rng, 1e-3)
        vol = rng.standard_normal((S, NT, 3) + prop.grid.shape).astype(np.float32) * 1e-3
        borders = torch.as_tensor(np.stack([_faces(v, W) for v in vol.reshape((-1,) + prop.grid.shape)]), device="cuda")
        assert borders.numel() == S * NT * L.efm_border_floats(by(d), W)
        res = torch.as_tensor(rng.standard_normal((S, 3, NT, 9)).astype(np.float32) * 1e-3, device="cuda")
        vpres = torch.zeros(S * 3 * prop.grid.N, device="cuda")
        g3 = [torch.zeros((S,) + prop.grid.shape, device="cuda") for _ in range(3)]
        for it0, n in ranges:
            _capi.check(L.efm_backward_remake_ref_steps(
                by(d), by(m), by(sh), by(fwd.struct()), _ptr(vpres), _ptr(borders), W, by(adj.struct()), _ptr(res),
                DT, 10.0, 10.0, 10.0, *[_ptr(t) for t in g3], it0, n, _stream()), "remake")
        torch.cuda.synchronize()
        images.append([t.cpu().numpy() for t in g3])
    for other in images[1:]:
        for a, b in zip(images[0], other):
            assert np.isfinite(a).all() and np.abs(a).max() > 0
            for s in range(S):
                assert np.abs(a[s] - b[s]).max() <= BOUND * np.abs(b[s]).max()


@pytest.mark.parametrize("case", CASES)
def test_border_save_beside_the_next_sweep(case):
    nx, ny, nz, W, nts, free_top, fuse, tiles = case
    _with_tiles(tiles)
    S, L = len(nts), _capi.lib()
    got = []
    for ranges in ([(0, NT)], [(i, 1) for i in range(NT)]):
        prop, batch, rng = _prop(nx, ny, nz, W, S, nts, free_top, fuse)
        d, m, sh = prop.dims(), prop.medium(), batch.struct()
        w = _state(prop, rng, 1e-3)
        borders = torch.full((S * NT * L.efm_border_floats(by(d), W),), 7.0, device="cuda")
        gat = torch.zeros((S, 3, NT, 9), device="cuda")
        for it0, n in ranges:
            _capi.check(L.efm_forward(by(d), by(m), by(sh), by(w.struct()), _ptr(gat), _ptr(borders), W, it0, n,
                                      _stream()), "forward")
        torch.cuda.synchronize()
        got.append((borders.cpu(), gat.cpu()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert (got[0][0] != 7.0).any()


@pytest.mark.parametrize("case", CASES)
def test_ranges_leave_the_bits_of_one_run(case):
    """What a run over all iterations leaves (images, adjoint, both velocity buffers, stresses
    and memory variables of the reconstruction) is left bit for bit by any ranges."""
    nx, ny, nz, W, nts, free_top, fuse, tiles = case
    _with_tiles(tiles)
    S, L = len(nts), _capi.lib()
    left = []
    for ranges in ([(0, NT - 1)], [(i, 1) for i in range(NT - 1)], [(0, 4), (4, 0), (4, NT - 5)], [(0, 1), (1, 2), (3, NT - 4)]):
        prop, batch, rng = _prop(nx, ny, nz, W, S, nts, free_top, fuse)
        d, m, sh = prop.dims(), prop.medium(), batch.struct()
        fwd, adj = _state(prop, rng, 1e-3), _state(prop, rng, 1e-3)
        vol = rng.standard_normal((S, NT, 3) + prop.grid.shape).astype(np.float32) * 1e-3
        borders = torch.as_tensor(np.stack([_faces(v, W) for v in vol.reshape((-1,) + prop.grid.shape)]), device="cuda")
        res = torch.as_tensor(rng.standard_normal((S, 3, NT, 9)).astype(np.float32) * 1e-3, device="cuda")
        if not fuse:
            res[..., 1] = 0.0            # receivers that share a cell add in any order
        vpres = torch.zeros(S * 3 * prop.grid.N, device="cuda")
        g3 = [torch.zeros((S,) + prop.grid.shape, device="cuda") for _ in range(3)]
        for it0, n in ranges:
            _capi.check(L.efm_backward_remake_ref_steps(
                by(d), by(m), by(sh), by(fwd.struct()), _ptr(vpres), _ptr(borders), W, by(adj.struct()), _ptr(res),
                DT, 10.0, 10.0, 10.0, *[_ptr(t) for t in g3], it0, n, _stream()), "remake")
        torch.cuda.synchronize()
        parts = [vpres, *g3]
        for w in (fwd, adj):
            parts += [w.fields, w.psi_x, w.psi_y, w.psi_z]
        left.append([t.cpu() for t in parts])
    for other in left[1:]:
        for a, b in zip(left[0], other):
            assert torch.equal(a, b)
