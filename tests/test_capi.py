"""The C ABI library loads, exports every symbol the headers under include/
declare, and rejects bad arguments before touching a GPU (CPU-only test)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    names = set()
    inc = os.path.join(ROOT, "include")
    for h in sorted(os.listdir(inc)):
        if h.endswith(".h"):
            with open(os.path.join(inc, h)) as f:
                src = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
            names |= set(re.findall(r"\b(efm_[a-z_0-9]+)\s*\(", src))
    return sorted(names)


@pytest.fixture(scope="module")
def L():
    from elastic_fm_vp_vs_rho_amd import _capi
    return _capi.lib()


def test_every_declared_symbol_is_exported_and_bound(L):
    from elastic_fm_vp_vs_rho_amd import _capi
    names = _declared()
    assert len(names) >= 20
    for n in names:
        assert hasattr(L, n), n
    assert set(names) == set(_capi.exported_symbols())


def test_c_host_example_is_built_and_links():
    """The C host (csrc/host_example.c) links ROCm's HIP runtime and libefm.so
    and starts without Python; run without arguments it prints its usage."""
    import subprocess
    exe = os.path.join(ROOT, "elastic_fm_vp_vs_rho_amd", "efm_host_example")
    assert os.path.exists(exe), "efm_host_example is not built (run __graft_entry__.build())"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1 and "usage" in r.stderr, (r.returncode, r.stderr)


def test_single_hip_runtime_mapped(L):
    from elastic_fm_vp_vs_rho_amd import _capi
    rts = _capi._hip_runtimes_mapped()
    assert len(rts) == 1 and "torch" in rts[0]


def test_version_and_errors(L):
    from elastic_fm_vp_vs_rho_amd import _capi
    assert L.efm_version() == 10000
    rc = L.efm_forward(None, None, None, None, None, None, 0, 0, 1, None)
    assert rc == -1
    assert "null" in _capi.last_error()
    assert L.efm_set_tile(0, 48, 3, 5, 0) == -3
    assert "tile" in _capi.last_error()
    n = L.efm_tile_variants(None, 0)
    buf = (ctypes.c_int * (4 * n))()
    assert L.efm_tile_variants(buf, n) == n
    assert all(buf[4 * i] % 64 == 0 for i in range(n))   # whole 64-lane waves along x
    assert {buf[4 * i + 3] for i in range(n)} == {0, 8, 16}   # linear, XCD-aware, compact
    assert L.efm_component_pad() == 1088
    # initializer kernels validate before launching
    assert L.efm_net_gemm(0, 1, 1, None, 0, 0, None, 0, 0, None, 1, None, None, 0, None) == -1
    assert "efm_net_gemm" in _capi.last_error()
    assert L.efm_net_im2col(None, None, 1, 1, 3, 5, 1, 0, None) == -1


def test_argument_validation_without_gpu(L):
    from elastic_fm_vp_vs_rho_amd._capi import EfmDims, EfmMedium, EfmShots, EfmState
    d = EfmDims(4, 10, 10, 1, 0, 0, 0, 0, 0, 0, 10, 0, 0.1)   # nx < 5
    m = EfmMedium(1, 1, 1)
    sh = EfmShots(*([1] * 11))
    st = EfmState(*([1] * 12))
    assert L.efm_forward(ctypes.byref(d), ctypes.byref(m), ctypes.byref(sh), ctypes.byref(st),
                         None, None, 0, 0, 1, None) == -1
    d = EfmDims(10, 10, 10, 1, 3, 3, 3, 3, 0, 3, 10, 0, 0.1)
    assert L.efm_forward(ctypes.byref(d), ctypes.byref(m), ctypes.byref(sh), ctypes.byref(st),
                         None, None, 0, 5, 6, None) == -1   # step range past ntmax


def test_size_limits_are_refused_without_gpu(L):
    """Grids whose per-shot offsets would pass 2^31, and batches whose sweep
    would pass 2^32 work-items in one dispatch, are refused by every entry point
    that takes the dimensions, before any launch."""
    from elastic_fm_vp_vs_rho_amd import _capi
    from elastic_fm_vp_vs_rho_amd._capi import EfmDims, EfmMedium, EfmShots, EfmState
    m = EfmMedium(1, 1, 1)
    sh = EfmShots(*([1] * 11))
    st = EfmState(*([1] * 12))
    big = EfmDims(2048, 1100, 1000, 1, 10, 10, 10, 10, 0, 10, 100, 0, 0.1)    # 2.25e9 cells
    many = EfmDims(512, 512, 512, 40, 10, 10, 10, 10, 0, 10, 100, 0, 0.1)     # 5.4e9 cells in all
    for d, word in ((big, "grid too large"), (many, "shot batch too large")):
        assert L.efm_forward(ctypes.byref(d), ctypes.byref(m), ctypes.byref(sh), ctypes.byref(st),
                             None, None, 0, 0, 1, None) == -1
        assert word in _capi.last_error()
        assert L.efm_derived_medium(ctypes.byref(d), ctypes.byref(m), 1, 1, None) == -1
        assert word in _capi.last_error()
        assert L.efm_gradient_combine(ctypes.byref(d), ctypes.byref(m), 1, 1, 1, 1, 1, 1, None) == -1
        assert word in _capi.last_error()
        assert L.efm_border_floats(ctypes.byref(d), 10) == -1


def test_shot_batch_validation():
    """Host-side validation of sources/receivers happens before any upload."""
    import numpy as np
    from elastic_fm_vp_vs_rho_amd.propagator import Grid, ShotBatch
    g = Grid.make(16, 16, 16, 10.0, 1e-3, 3)
    cp = {k: np.zeros(16, np.float32) for k in ("ax", "bx", "ay", "by", "az", "bz")}
    with pytest.raises(ValueError, match="interior"):
        ShotBatch(g, [(1, 8, 8)], [np.zeros(6)], [np.zeros(10)], [10], [[(5, 5, 2)]], cp, device="cpu")
    with pytest.raises(ValueError, match="receiver"):
        ShotBatch(g, [(8, 8, 8)], [np.zeros(6)], [np.zeros(10)], [10], [[(5, 16, 2)]], cp, device="cpu")


def test_shots_per_dispatch_fits_every_tile(L):
    """The batch cap that sub-batching uses keeps every compiled tile's sweep
    under 2^32 work-items, and leaves the workloads' batches whole."""
    from elastic_fm_vp_vs_rho_amd import autotune
    from elastic_fm_vp_vs_rho_amd.propagator import Grid
    for n, S_needed in (((40, 40, 40), 768), ((96, 96, 96), 256), ((256, 256, 128), 32)):
        g = Grid(n[0], n[1], n[2], 10.0, 1e-3, (10,) * 6)
        S = autotune.shots_per_dispatch(g)
        assert S >= S_needed, (n, S)
        for bx, bz, ny, mp in autotune.variants():
            if mp == 16:    # compact interior plane
                blocks = -(-(g.nx - 4) * (g.nz - 4) // (bx * bz)) * -(-(g.ny - 4) // ny) * S
            else:
                blocks = -(-g.nx // bx) * -(-g.nz // bz) * -(-(g.ny - 4) // ny) * S
            if mp:
                blocks = 8 * -(-blocks // 8)
            assert blocks * bx * bz < 1 << 32


def test_bench_traffic_table_covers_every_compiled_tile(L):
    """bench.py reports the roofline's HBM traffic from measured per-tile
    values; every tile the library compiles must have one for every sweep, or
    the bench line would carry a null traffic whichever tile the tuner picks."""
    import bench
    from elastic_fm_vp_vs_rho_amd import autotune
    keys = {",".join(str(v) for v in t) for t in autotune.variants()}
    for k in autotune.KERNELS:
        assert set(bench.MEASURED_TRAFFIC[k]) == keys, k
        assert all(v > 0 for v in bench.MEASURED_TRAFFIC[k].values())


def _structs(nrec=4):
    from elastic_fm_vp_vs_rho_amd._capi import EfmDims, EfmMedium, EfmShots, EfmState
    d = EfmDims(16, 16, 16, 1, 3, 3, 3, 3, 0, 3, 10, nrec, 0.1)
    return d, EfmMedium(1, 1, 1), EfmShots(*([1] * 12)), EfmState(*([1] * 12))


@pytest.mark.parametrize("hole", ["ax", "nt", "rec", "wavelet", "src"])
def test_null_shot_arrays_are_refused_before_launch(L, hole):
    """Every entry point that reads the shot description checks its arrays
    (a null one would reach a kernel and fault the GPU)."""
    from elastic_fm_vp_vs_rho_amd import _capi
    d, m, sh, st = _structs()
    setattr(sh, hole, None)
    by = ctypes.byref
    calls = {
        "efm_forward": lambda: L.efm_forward(by(d), by(m), by(sh), by(st), 1, None, 0, 0, 1, None),
        "efm_record": lambda: L.efm_record(by(d), by(sh), by(st), 1, 0, None),
        "efm_inject_residual": lambda: L.efm_inject_residual(by(d), by(sh), by(st), 1, 0, None),
        "efm_image_mt_ref": lambda: L.efm_image_mt_ref(by(d), by(m), by(sh), by(st), 1, 0, None),
        "efm_backward_mt_ref": lambda: L.efm_backward_mt_ref(by(d), by(m), by(sh), by(st), 1, 1, 1, None),
        "efm_backward_remake_ref": lambda: L.efm_backward_remake_ref(
            by(d), by(m), by(sh), by(st), 1, 1, 3, by(st), 1, 1.0, 1.0, 1.0, 1.0, 1, 1, 1, None),
        "efm_backward_remake_ref_steps": lambda: L.efm_backward_remake_ref_steps(
            by(d), by(m), by(sh), by(st), 1, 1, 3, by(st), 1, 1.0, 1.0, 1.0, 1.0, 1, 1, 1, 0, 1, None),
    }
    fwd = (ctypes.POINTER(type(st)) * 2)(ctypes.pointer(st), ctypes.pointer(st))
    calls["efm_adjoint"] = lambda: L.efm_adjoint(by(d), by(m), 1, 1, by(sh), fwd, by(st), by(st), 1, 1, 1,
                                                 0, 1, 1, None)
    for name, call in calls.items():
        assert call() == -1, name
        assert "null" in _capi.last_error(), (name, _capi.last_error())


@pytest.mark.parametrize("hole", ["fwd", "adj_field", "adj_psi", "adj2_psi"])
def test_efm_adjoint_checks_every_state(L, hole):
    from elastic_fm_vp_vs_rho_amd import _capi
    from elastic_fm_vp_vs_rho_amd._capi import EfmState
    d, m, sh, st = _structs()
    good = [EfmState(*([1] * 12)) for _ in range(4)]
    adj, adj2 = EfmState(*([1] * 12)), EfmState(*([0] * 9 + [1] * 3))   # adj2: ψ buffers only
    if hole == "fwd":
        good[2].tzz = None               # one forward state in the middle of the range
    elif hole == "adj_field":
        adj.vy = None
    elif hole == "adj_psi":
        adj.psi_z = None
    else:
        adj2.psi_x = None
    fwd = (ctypes.POINTER(EfmState) * 4)(*[ctypes.pointer(s) for s in good])
    by = ctypes.byref
    rc = L.efm_adjoint(by(d), by(m), 1, 1, by(sh), fwd, by(adj), by(adj2), 1, 1, 1, 5, 8, 0, None)
    assert rc == -1 and "null" in _capi.last_error(), _capi.last_error()


def test_batches_up_to_the_dispatch_limit_are_accepted(L):
    """A compact sweep of a batch just under 2^32 interior work-items walks the interior
    cells when the line-aligned walk, guard cells included, would pass the limit; just over
    it the batch is refused as before."""
    from elastic_fm_vp_vs_rho_amd import _capi
    from elastic_fm_vp_vs_rho_amd._capi import EfmDims
    for nx, ny, nz in ((32, 460, 460), (8, 40, 40), (64, 200, 200), (512, 300, 300)):
        # the default tile: 128 interior cells of a plane to a block, 8 runs of a shot's blocks
        blocks = -(-(nx - 4) * (nz - 4) // 128) * (ny - 4)
        most = ((1 << 32) - 1) // (128 * 8 * -(-blocks // 8))
        dims = lambda S: EfmDims(nx, ny, nz, S, 0, 0, 0, 0, 0, 0, 10, 0, 0.1)
        assert L.efm_border_floats(ctypes.byref(dims(most)), 2) > 0, (nx, _capi.last_error())
        assert L.efm_border_floats(ctypes.byref(dims(most + 1)), 2) == -1
        assert "shot batch too large" in _capi.last_error()


def test_implicit_convolution_limits(L):
    """A convolution that the implicit kernels' launches cannot hold (rows of a 64 x 64 tile
    grid, 2^32 work-items of 64 columns a 1024-thread block, blocks of the weight gradient)
    is not taken by them: such a network keeps the stored im2col matrix."""
    #        C, B, L, M, ks, stride, pad
    for n, shape in enumerate([(1, 1, 8, 64 * 65535 + 1, 1, 1, 0), (1, 1 << 25, 8, 1, 1, 1, 0),
                               (16384, 1, 8, 16384, 9, 1, 4)]):
        assert L.efm_net_conv1d_fits(*shape) == 0, shape
    for shape in [(1, 1, 8, 64 * 65535, 1, 1, 0), (1, (1 << 25) - 8, 8, 1, 1, 1, 0), (8192, 1, 8, 16384, 9, 1, 4),
                  (192, 64, 1024, 64, 9, 4, 4)]:
        assert L.efm_net_conv1d_fits(*shape) == 1, shape
