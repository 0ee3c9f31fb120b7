"""The two walks of a compact forward sweep, whole lines or interior cells only, around the
sizes where the rule changes from one to the other: both give the bits of the row tiles, which
walk neither, in fields, CPML memory and seismograms (receivers at row ends, in the guard
rows' neighbours and sharing a cell)."""
import ctypes

import numpy as np
import pytest
import torch

from elastic_fm_vp_vs_rho_amd import _capi
from tests.gpu_helpers import grid_of
from tests.problems import tiny

pytestmark = pytest.mark.gpu


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


# 64 x ny x 64: 31 blocks a plane of whole lines, 29 of interior cells, the chip holds 3584
@pytest.mark.parametrize("n,S", [((64, 119, 64), 1), ((64, 120, 64), 1), ((64, 127, 64), 1), ((64, 128, 64), 1),
                                 ((63, 119, 64), 1), ((48, 48, 48), 5), ((41, 37, 33), 10), ((41, 37, 33), 12)])
def test_walks_agree(gpu_lib, n, S):
    from elastic_fm_vp_vs_rho_amd.propagator import Propagator, ShotBatch
    nt, nrec = 12, 70
    p = tiny(n=n, nt=nt, W=5, seed=3, nrec=1)
    rng = np.random.default_rng(S)
    src = np.stack([rng.integers(8, m - 8, S) for m in n], 1)
    rec = src[:, None, :] + rng.integers(-5, 6, (S, nrec, 3))
    rec[:, :4] = [(2, 2, 2), (n[0] - 3, n[1] - 3, n[2] - 3), (2, 5, n[2] - 3), (n[0] - 3, 5, 2)]
    rec[:, 5] = rec[:, 6]
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")
    batch = ShotBatch(grid_of(p), src, rng.uniform(-1, 1, (S, 6)), np.ones((S, nt), np.float32),
                      rng.integers(nt - 3, nt + 1, S), rec, p.cp)
    out = []
    for tile in ((128, 1, 1, 16), (64, 2, 1, 0)):
        for k in range(2):
            _capi.check(_capi.lib().efm_set_tile(k, *tile), "efm_set_tile")
        prop = Propagator(grid_of(p), f(p.lam), f(p.mu), f(p.rho), batch)
        g, st = prop.forward()
        out.append((g, st.fields, st.psi_x, st.psi_y, st.psi_z))
    assert float(out[0][0].abs().max()) > 0
    for a, b in zip(*out):
        assert torch.equal(a, b)
