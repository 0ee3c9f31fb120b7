"""The implicit-convolution kernels of the initializer at the edges of their tiles and
dispatch: taps 1, 3, 8 and 9, row ends and padding wider than a load, channels and samples
that do not fill a slab, sums over (b, l) of one slab and of many, rows summed in one
block and in chains, and the shapes that keep the stored im2col matrix.

Every sum keeps the order of the stored-matrix path, so the two agree bit for bit; col2im,
which has no counterpart of the same bits, is held to a float64 sum of its at most ks
float32 terms: |error| <= ks·2^-24·sum|terms|.
"""

import ctypes

import numpy as np
import pytest
import torch

from elastic_fm_vp_vs_rho_amd import _capi
from elastic_fm_vp_vs_rho_amd.initnet import InitNet, NetSpec

pytestmark = pytest.mark.gpu

# C, B, L, M, ks, stride, pad
SHAPES = [
    (1, 1, 8, 1, 9, 1, 4),          # the smallest row, one output row, one k slab part
    (5, 3, 13, 7, 9, 4, 4),         # odd everything, Lout < 8
    (33, 2, 40, 65, 9, 4, 4),       # one past a channel slab and an M tile
    (32, 4, 64, 64, 8, 2, 3),       # whole slabs, no ninth tap
    (17, 5, 31, 64, 3, 1, 0),       # no padding, odd rows
    (16, 2, 32, 130, 1, 3, 0),      # one tap
    (6, 2, 9, 8, 9, 1, 20),         # padding past the row: whole outputs of zeros
    (16, 40, 64, 64, 9, 2, 4),      # whole slabs of the backward sum
    (24, 7, 700, 16, 9, 1, 4),      # a ragged last slab, 8 does not divide it
    (3, 9, 4000, 20, 2, 3, 1),      # rows of 36000 values: chains longer than a round
]


def _p(t):
    return t.data_ptr()


def _ok(rc):
    _capi.check(rc, "net")


def _dbl(t):
    return t.cpu().double()


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_forward_is_the_stored_matrix_product(shape):
    C, B, L, M, ks, stride, pad = shape
    lib, Lout = _capi.lib(), (L + 2 * pad - ks) // stride + 1
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(C, B, L, generator=g).bfloat16().cuda()
    W = torch.randn(M, C * ks, generator=g).bfloat16().cuda()
    bias = torch.randn(M, generator=g).cuda()
    K, N = C * ks, B * Lout
    col = torch.empty(K, N, dtype=torch.bfloat16, device="cuda")
    want, wantb = torch.empty(M, N, device="cuda"), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    wantf = torch.empty(M * Lout, B, dtype=torch.bfloat16, device="cuda")
    _ok(lib.efm_net_im2col(_p(x), _p(col), C, B, L, ks, stride, pad, None))
    _ok(lib.efm_net_gemm(M, N, K, _p(W), K, 1, _p(col), N, 1, _p(want), N, _p(bias), _p(wantb), 1, None))
    _ok(lib.efm_net_flatten(_p(wantb), _p(wantf), M, B, Lout, None))
    for flat, ref in ((0, wantb), (1, wantf)):
        y, yb = torch.empty_like(want), torch.empty_like(ref)
        _ok(lib.efm_net_conv1d(_p(x), _p(W), _p(bias), _p(y), _p(yb), C, B, L, M, ks, stride, pad, flat, None))
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(yb, ref)


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_backward_products(shape):
    C, B, L, M, ks, stride, pad = shape
    lib, Lout = _capi.lib(), (L + 2 * pad - ks) // stride + 1
    assert lib.efm_net_conv1d_fits(*shape) == 1
    g = torch.Generator().manual_seed(1 + sum(shape))
    x, W = torch.randn(C, B, L, generator=g).bfloat16().cuda(), torch.randn(M, C * ks, generator=g).bfloat16().cuda()
    dp = torch.randn(M, B * Lout, generator=g).bfloat16().cuda()
    K, N = C * ks, B * Lout
    col = torch.empty(K, N, dtype=torch.bfloat16, device="cuda")
    _ok(lib.efm_net_im2col(_p(x), _p(col), C, B, L, ks, stride, pad, None))
    wW, wcol = torch.empty(M, K, device="cuda"), torch.empty(K, N, device="cuda")
    _ok(lib.efm_net_gemm(M, K, N, _p(dp), N, 1, _p(col), 1, N, _p(wW), K, None, None, 0, None))
    _ok(lib.efm_net_gemm(K, N, M, _p(W), 1, K, _p(dp), N, 1, _p(wcol), N, None, None, 0, None))
    wide = torch.full((M, N + 72), float("nan"), dtype=torch.bfloat16, device="cuda")       # rows further apart
    wide[:, :N] = dp
    for both, d in ((True, dp), (False, dp), (True, wide)):
        dW, dcol = torch.full((M, K), 7.0, device="cuda"), torch.full((K, N), 7.0, device="cuda")
        _ok(lib.efm_net_conv1d_back(_p(d), _p(x), _p(W), _p(dW), _p(dcol) if both else None, *shape,
                                    d.stride(0), None))
        torch.cuda.synchronize()
        assert torch.equal(dW, wW)
        assert torch.equal(dcol, wcol) if both else (dcol == 7.0).all()


@pytest.mark.parametrize("shape", SHAPES)
def test_relu_and_bias_rows(shape):
    C, B, L, M, ks, stride, pad = shape
    lib, Lout = _capi.lib(), (L + 2 * pad - ks) // stride + 1
    g = torch.Generator().manual_seed(2 + sum(shape))
    y, dcol = torch.randn(C, B, L, generator=g), torch.randn(C * ks, B * Lout, generator=g)
    yd, dcold = y.cuda(), dcol.cuda()
    dy = torch.empty(C, B, L, device="cuda")
    _ok(lib.efm_net_col2im(_p(dcold), _p(dy), C, B, L, ks, stride, pad, None))
    # the transposed im2col itself against float64
    ref = torch.zeros(C, B, L + 2 * pad + ks, dtype=torch.float64)
    mag = torch.zeros_like(ref)
    d4 = dcol.double().reshape(C, ks, B, Lout)
    for k in range(ks):
        ref[:, :, k:k + stride * Lout:stride][:, :, :Lout] += d4[:, k]
        mag[:, :, k:k + stride * Lout:stride][:, :, :Lout] += d4[:, k].abs()
    ref, mag = ref[:, :, pad:pad + L], mag[:, :, pad:pad + L]
    assert ((_dbl(dy) - ref).abs() <= ks * 2.0 ** -24 * mag).all()
    dp = torch.where(yd > 0, dy, torch.zeros((), device="cuda"))
    want = torch.empty(C, device="cuda")
    _ok(lib.efm_net_bias_grad(_p(dp), _p(want), C, B * L, None))
    flat = dy.permute(0, 2, 1).reshape(C * L, B).contiguous()
    rows = lambda d, n: lambda *out: lib.efm_net_relu_bias_backward(_p(d), _p(yd), *out, C, B * L, B, n, B * L + 9, None)
    for call in (lambda *out: lib.efm_net_col2im_relu_bias(_p(dcold), _p(yd), *out, C, B, L, ks, stride, pad, B * L + 9,
                                                            None),
                 rows(dy, 0), rows(flat, L)):
        for chained in (False, True):
            dpb = torch.full((C, B * L + 9), 7.0, dtype=torch.bfloat16, device="cuda")
            db = torch.full((C,), 7.0, device="cuda")
            chains = torch.full((C, 256), float("nan"), device="cuda")
            _ok(call(_p(dpb), _p(db), _p(chains) if chained else None))
            if chained:
                assert (db == 7.0).all()
                _ok(lib.efm_net_bias_sums(ctypes.byref(_capi.EfmNetBias(_p(chains), _p(db), C)), 1, None))
            torch.cuda.synchronize()
            assert torch.equal(dpb[:, :B * L], dp.bfloat16().reshape(C, B * L)) and (dpb[:, B * L:] == 7.0).all()
            assert torch.equal(db, want)


@pytest.mark.parametrize("spec,implicit", [
    (NetSpec(cin=9, length=64, channels=8, ks=9, stride=2, pad=4, nblocks=2, hidden=16), 2),
    (NetSpec(cin=9, length=64, channels=8, ks=11, stride=2, pad=5, nblocks=2, hidden=16), 0),
    (NetSpec(cin=9, length=16, channels=8, ks=9, stride=2, pad=4, nblocks=3, hidden=16), 2),
])
def test_net_keeps_the_stored_matrix_where_it_must(spec, implicit):
    """Kernels of more than 9 taps and rows under 8 samples go through the im2col matrix;
    a step of either kind moves the loss the way its gradient says."""
    net = InitNet(spec, device="cuda", seed=2)
    b = net._buffers(5)
    assert sum(f"col{i}" not in b for i in range(spec.nblocks)) == implicit
    g = torch.Generator().manual_seed(3)
    b["x"].copy_(torch.randn(b["x"].shape, generator=g).bfloat16())
    b["t"].copy_(torch.randn(b["t"].shape, generator=g))
    net.forward_buffers(5)
    first = float(net.backward_buffers(5).item())
    for _ in range(5):
        net.adam(lr=1e-3)
        net.forward_buffers(5)
        last = float(net.backward_buffers(5).item())
    assert np.isfinite(first) and last < first


@pytest.mark.parametrize("length", [16, 13])
def test_gather_batch_rows(length):
    """Rows copied eight samples at a time and one at a time."""
    lib, C, B, nout = _capi.lib(), 5, 6, 9
    data = torch.randn(11, C, length).bfloat16().cuda()
    target = torch.randn(11, nout).cuda()
    idx = torch.tensor([10, 0, 3, 3, 7, 1], dtype=torch.int32, device="cuda")
    x = torch.empty(C, B, length, dtype=torch.bfloat16, device="cuda")
    t = torch.empty(nout, B, device="cuda")
    _ok(lib.efm_net_gather_batch(_p(data), _p(target), data.shape[0], _p(idx), B, C, length, nout, _p(x), _p(t), None))
    assert torch.equal(x, data[idx.long()].permute(1, 0, 2)) and torch.equal(t, target[idx.long()].T)


@pytest.mark.parametrize("count", [0, 1, 16, 17, 40])
def test_bias_lists(count):
    """Lists below, at and above a launch's sixteen biases."""
    lib, rng = _capi.lib(), np.random.default_rng(count)
    ins, outs, biases = [], [], (_capi.EfmNetBias * count)()
    for j in range(count):
        m = int(rng.integers(1, 70))
        ins.append(torch.as_tensor(rng.integers(-8, 9, (m, 256)).astype(np.float32)).cuda())
        outs.append(torch.empty(m, device="cuda"))
        biases[j] = _capi.EfmNetBias(_p(ins[j]), _p(outs[j]), m)
    _ok(lib.efm_net_bias_sums(biases, count, None))
    for j in range(count):
        assert torch.equal(outs[j], ins[j].sum(1))                  # whole numbers: exact


def test_longest_row():
    """A row of 2^31 - 1 values in one block: the last round of 256 passes 2^31.  Each chain is
    a whole number below 2^24, the tree over them within 8 roundings."""
    lib, N = _capi.lib(), 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < 25 * 10 ** 9:
        pytest.skip("needs 25 GB of free GPU memory")
    dy, y = torch.ones(N, device="cuda"), torch.ones(N, device="cuda")
    dpb, db = torch.zeros(N + 1, dtype=torch.bfloat16, device="cuda"), torch.zeros(1, device="cuda")
    _ok(lib.efm_net_relu_bias_backward(_p(dy), _p(y), _p(dpb), _p(db), None, 1, N, 0, 0, N, None))
    torch.cuda.synchronize()
    assert abs(float(db) - N) <= 8 * 2.0 ** -24 * N
    for at in (0, N // 2, N - 300):
        assert (dpb[at:min(at + 300, N)] == 1).all()
    assert float(dpb[N]) == 0


@pytest.mark.parametrize("spec", [
    NetSpec(cin=9, length=64, channels=8, ks=9, stride=2, pad=4, nblocks=2, hidden=16),
    NetSpec(cin=9, length=64, channels=8, ks=11, stride=2, pad=5, nblocks=2, hidden=16),
    NetSpec(cin=9, length=64, channels=8, ks=11, stride=2, pad=5, nblocks=1, hidden=16),
    NetSpec(cin=9, length=7, channels=8, ks=3, stride=1, pad=1, nblocks=2, hidden=16),
])
def test_gemm_rate_times_either_path(spec):
    """The rate of the first convolution, implicit or over the stored matrix."""
    from elastic_fm_vp_vs_rho_amd.initnet_data import gemm_rate
    net = InitNet(spec, device="cuda", seed=4)
    r = gemm_rate(net, 5, reps=3)
    ci, co, _, lo = spec.convs()[0]
    assert (r["M"], r["N"], r["K"]) == (co, 5 * lo, ci * spec.ks) and r["ms"] > 0 and r["tflops"] > 0
