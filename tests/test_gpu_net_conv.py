"""The implicit-convolution kernels of the initializer at the edges of their tiles and
dispatch: taps 1, 3, 8 and 9, row ends and padding wider than a load, channels and samples
that do not fill a slab, sums over (b, l) short, long and cut over blocks, rows cut over
blocks, and the shapes that keep the stored im2col matrix.

The forward pass is the stored-matrix path bit for bit (same sums).  Gradients are sums
of n float32 terms against float64: |error| <= min(n, 4·sqrt(n))·u·sum|terms|, n roundings
in any order (the worst case, or four standard deviations) of u = 2^-23, twice the
rounding to nearest, as the matrix instruction may truncate inside.
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
    (16, 40, 64, 64, 9, 2, 4),      # sum of 1280: cut over blocks; rows of 2560: cut
    (24, 7, 700, 16, 9, 1, 4),      # ragged last part of a cut sum, 8 does not divide it
]


def _p(t):
    return t.data_ptr()


def _ok(rc):
    _capi.check(rc, "net")


def _bound(n, mag):
    return min(n, 4 * np.sqrt(n)) * 2.0 ** -23 * mag + 1e-30


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
def test_conv_gradients(shape):
    C, B, L, M, ks, stride, pad = shape
    lib, Lout = _capi.lib(), (L + 2 * pad - ks) // stride + 1
    g = torch.Generator().manual_seed(1 + sum(shape))
    x = torch.randn(C, B, L, generator=g).bfloat16()
    dp = torch.randn(M, B * Lout, generator=g).bfloat16()
    y = torch.randn(C, B, L, generator=g)
    dcol = torch.randn(C * ks, B * Lout, generator=g)
    n = lib.efm_net_conv1d_work(C, B, L, M, ks, stride, pad)
    work = torch.full((n,), float("nan"), device="cuda")
    # weight gradient: dp · colᵀ
    xp = torch.nn.functional.pad(x.double(), (pad, pad))
    col = xp.unfold(2, ks, stride)[:, :, :Lout].permute(0, 3, 1, 2).reshape(C * ks, B * Lout)
    dW = torch.empty(M, C * ks, device="cuda")
    xd, dpd, dcold, yd = x.cuda(), dp.cuda(), dcol.cuda(), y.cuda()
    _ok(lib.efm_net_conv1d_dw(_p(dpd), _p(xd), _p(dW), C, B, L, M, ks, stride, pad, _p(work), None))
    err, mag = (_dbl(dW) - dp.double() @ col.T).abs(), dp.double().abs() @ col.abs().T
    assert (err <= _bound(B * Lout, mag)).all()
    # dy = col2im(dcol), then ReLU and the bias sum
    dy = torch.zeros(C, B, L + 2 * pad + ks, dtype=torch.float64)
    mg = torch.zeros_like(dy)
    d4 = dcol.double().reshape(C, ks, B, Lout)
    for k in range(ks):
        dy[:, :, k:k + stride * Lout:stride][:, :, :Lout] += d4[:, k]
        mg[:, :, k:k + stride * Lout:stride][:, :, :Lout] += d4[:, k].abs()
    dy, mg = dy[:, :, pad:pad + L], mg[:, :, pad:pad + L]
    dpb, db = torch.empty(C, B, L, dtype=torch.bfloat16, device="cuda"), torch.empty(C, device="cuda")
    _ok(lib.efm_net_col2im_relu_bias(_p(dcold), _p(yd), _p(dpb), _p(db), C, B, L, ks, stride, pad, _p(work), None))
    on = (y > 0).double()
    assert ((_dbl(dpb) - dy * on).abs() <= 2.0 ** -8 * (dy * on).abs() + _bound(ks, mg)).all()
    assert ((_dbl(db) - (dy * on).sum((1, 2))).abs() <= _bound(ks * B * L, (mg * on).sum((1, 2)))).all()
    # the same from a plain and a flattened dy
    dyf = dy.float()
    dyf_d = dyf.reshape(C, B * L).cuda()
    flat = dyf.permute(0, 2, 1).reshape(C * L, B).contiguous().cuda()
    for d, l in ((dyf_d, 0), (flat, L)):
        _ok(lib.efm_net_relu_bias_backward(_p(d), _p(yd), _p(dpb), _p(db), C, B * L, B, l, _p(work), None))
        assert torch.equal(dpb.cpu(), torch.where(y > 0, dyf, torch.zeros(())).bfloat16())
        ref = dyf.double() * on
        assert ((_dbl(db) - ref.sum((1, 2))).abs() <= _bound(B * L, ref.abs().sum((1, 2)))).all()


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


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_backward_in_one_launch(shape):
    """dW's parts and dcol from one launch: the separate calls' bits (the parts left unsummed
    where there are several, dcol through the general product where it cannot ride along)."""
    C, B, L, M, ks, stride, pad = shape
    lib, Lout = _capi.lib(), (L + 2 * pad - ks) // stride + 1
    g = torch.Generator().manual_seed(2 + sum(shape))
    x, W = torch.randn(C, B, L, generator=g).bfloat16().cuda(), torch.randn(M, C * ks, generator=g).bfloat16().cuda()
    dp = torch.randn(M, B * Lout, generator=g).bfloat16().cuda()
    K, N, n = C * ks, B * Lout, M * C * ks
    conv = (C, B, L, M, ks, stride, pad)
    parts = lib.efm_net_conv1d_parts(*conv)
    work = torch.zeros(max(parts * n, lib.efm_net_conv1d_work(*conv)), device="cuda")
    dW, got, dcol, want = (torch.full(s, 7.0, device="cuda") for s in ((M, K), (M, K), (K, N), (K, N)))
    _ok(lib.efm_net_conv1d_back(_p(dp), _p(x), _p(W), _p(got), _p(dcol), *conv, _p(work), None))
    if parts > 1:
        assert (got == 7.0).all()
        s = _capi.EfmNetSum(_p(work), _p(got), n, 1, n, parts)
        _ok(lib.efm_net_sum(ctypes.byref(s), 1, None))
    _ok(lib.efm_net_conv1d_dw(_p(dp), _p(x), _p(dW), *conv, _p(work), None))
    _ok(lib.efm_net_gemm(K, N, M, _p(W), 1, K, _p(dp), N, 1, _p(want), N, None, None, 0, None))
    torch.cuda.synchronize()
    assert torch.equal(got, dW) and torch.equal(dcol, want)


@pytest.mark.parametrize("count", [0, 1, 12, 13, 30])
def test_sum_lists(count):
    """Lists below, at and above a launch's twelve sums; parts side by side and one after the other."""
    lib, rng = _capi.lib(), np.random.default_rng(count)
    ins, outs, sums = [], [], (_capi.EfmNetSum * count)()
    for j in range(count):
        n, k = int(rng.integers(1, 700)), int(rng.integers(1, 9))
        ins.append(torch.as_tensor(rng.integers(-8, 9, (k, n) if j % 2 else (n, k)).astype(np.float32)).cuda())
        outs.append(torch.empty(n, device="cuda"))
        sums[j] = _capi.EfmNetSum(_p(ins[j]), _p(outs[j]), n, 1 if j % 2 else k, n if j % 2 else 1, k)
    _ok(lib.efm_net_sum(sums, count, None))
    for j in range(count):
        assert torch.equal(outs[j], ins[j].sum(0 if j % 2 else 1))          # whole numbers: exact
