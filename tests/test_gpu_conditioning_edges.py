"""Edges of the smoothing and cross-correlation kernels: lines shorter than, equal
to and longer than the kernel's support, rows around a multiple of the wave, the
fixed-radius and the general instance; trace groups around a block's receivers and
its samples per step."""
import numpy as np
import pytest
import torch
from scipy.ndimage import gaussian_filter

from elastic_fm_vp_vs_rho_amd import conditioning as C
from oracle import elastic_fp64 as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [1.0, 0.6, 2.0])          # radius 4 (its own instance), 2 and 8
@pytest.mark.parametrize("shape", [(8, 9, 10), (9, 4, 32), (3, 17, 33), (12, 5, 64), (21, 30, 65), (1, 1, 97)])
def test_gaussian_equals_scipy_on_short_and_long_lines(gpu_lib, shape, sigma):
    g = np.random.default_rng(4).standard_normal(shape).astype(np.float32)
    ref = gaussian_filter(g, sigma=sigma, mode="reflect", truncate=4.0)
    got = C.condition_gradient(torch.as_tensor(g, device="cuda"), sigma).cpu().numpy()
    # sums in double in scipy's order, one rounding per pass: at most an ulp of the scale
    assert np.abs(got - ref).max() <= 2e-7 * np.abs(ref).max()


@pytest.mark.parametrize("nrec", [1, 3, 16, 17, 40])
@pytest.mark.parametrize("nt", [1, 64, 65, 1030])
def test_xcorr_residual_for_any_trace_count_and_length(gpu_lib, nrec, nt):
    from elastic_fm_vp_vs_rho_amd import _capi
    from elastic_fm_vp_vs_rho_amd.propagator import _ptr, _stream
    rng = np.random.default_rng(nrec * 2000 + nt)
    mod, obs = (rng.standard_normal((2, 3, nt, nrec)).astype(np.float32) for _ in range(2))
    mod[0, 1, :, nrec - 1] = 0.0
    m, o = (torch.as_tensor(a, device="cuda") for a in (mod, obs))
    r, J = torch.empty_like(m), torch.zeros(1, dtype=torch.float64, device="cuda")
    _capi.check(_capi.lib().efm_xcorr_residual(_ptr(m), _ptr(o), _ptr(r), _ptr(J), 2, nt, nrec, _stream()), "xcorr")
    ref = [O.xcorr_residual(mod[s], obs[s]) for s in range(2)]
    # the residual is a difference of two terms (which cancel exactly in a trace of one
    # sample): double roundings of the terms, then one rounding to float32
    norm = lambda a: np.where((q := np.sqrt((a.astype(np.float64) ** 2).sum(2, keepdims=True))) == 0, 1.0, q)
    for s in range(2):
        term = np.abs(obs[s:s + 1].astype(np.float64)) / (norm(mod[s:s + 1]) * norm(obs[s:s + 1]))
        want = ref[s][0]
        assert (np.abs(r[s].double().cpu().numpy() - want) <= 6e-8 * np.abs(want) + 1e-14 * term[0]).all()
    assert abs(float(J) - sum(x[1] for x in ref)) <= 1e-9 * max(1.0, sum(x[1] for x in ref))


@pytest.mark.parametrize("shape,margins", [((4, 4, 4), (0,) * 6), ((5, 8, 64), (1, 1, 1, 1, 1, 1)),
                                           ((8, 9, 65), (3, 0, 0, 2, 8, 0)), ((17, 25, 131), (64, 3, 8, 8, 9, 9)),
                                           ((9, 7, 67), (0, 67, 0, 0, 0, 0)), ((24, 16, 128), (0, 0, 8, 8, 8, 0))])
def test_gaussian_tiles_and_masks(gpu_lib, shape, margins):
    """Tiles of 64 x 8 x 8 cells: volumes around one tile, ragged last tiles, tiles the mask
    covers in part, whole, and altogether."""
    g = np.random.default_rng(7).standard_normal(shape).astype(np.float32)
    ref = gaussian_filter(g, sigma=1.0, mode="reflect", truncate=4.0)
    ny, nz, nx = shape
    keep = np.zeros(shape, bool)
    xl, xh, yl, yh, zl, zh = margins
    keep[yl:ny - yh, zl:nz - zh, xl:max(xl, nx - xh)] = True
    ref[~keep] = 0
    got = C.condition_gradient(torch.as_tensor(g, device="cuda"), 1.0, 4.0, margins).cpu().numpy()
    assert (got[~keep] == 0).all()
    assert np.abs(got - ref).max() <= 2e-7 * np.abs(g).max()
