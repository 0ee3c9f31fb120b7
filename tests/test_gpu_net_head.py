"""The dense head's fused kernels at the edges of their tiles and limits: examples around a
block of 16 and the 128 of the backward kernel, sums and rows that do not fill a slab, one
output and a full tile of them, and the sizes that keep the separate products.

Forward is the general product bit for bit.  Backward against float64 from the same BF16
operands: a sum of n float32 terms is within n·2^-23 of sum|terms| in any order (twice the
rounding to nearest, as the matrix instruction may truncate), dout itself within 3 roundings,
and dzpb within a BF16 rounding on top.
"""

import numpy as np
import pytest
import torch

from elastic_fm_vp_vs_rho_amd import _capi

pytestmark = pytest.mark.gpu

# B, flat, hidden, nout, what fits
SIZES = [(1, 1, 1, 1, 3), (8, 256, 128, 9, 3), (15, 33, 17, 9, 3), (17, 300, 129, 16, 3), (64, 264, 136, 9, 3),
         (128, 40, 500, 2, 3), (129, 96, 64, 9, 1), (16, 1500, 460, 17, 1), (16, 1500, 469, 9, 0)]


def _bf(a):
    return torch.as_tensor(a, dtype=torch.float32).bfloat16().cuda()


def _p(t):
    return t.data_ptr()


@pytest.mark.parametrize("B,flat,hidden,nout,fits", SIZES)
def test_head_kernels(B, flat, hidden, nout, fits):
    L, rng = _capi.lib(), np.random.default_rng(B + flat)
    assert L.efm_net_head_fits(B, flat, hidden, nout) == fits
    n = lambda *s: rng.standard_normal(s).astype(np.float32)
    f = lambda a: torch.as_tensor(a).cuda()
    X, F1, F2 = _bf(n(flat, B)), _bf(n(hidden, flat)), _bf(n(nout, hidden))
    c1, c2, tg = f(n(hidden)), f(n(nout)), f(n(nout, B))
    z, out = torch.empty(hidden, B, device="cuda"), torch.empty(nout, B, device="cuda")
    zb = torch.empty(hidden, B, dtype=torch.bfloat16, device="cuda")
    ok = lambda rc: _capi.check(rc, "net")
    args = [_p(t) for t in (X, F1, c1, F2, c2, z, zb, out)] + [B, flat, hidden, nout, None]
    if not fits:
        assert L.efm_net_head_forward(*args) != 0
        return
    ok(L.efm_net_head_forward(*args))
    rz, rout, rzb = torch.empty_like(z), torch.empty_like(out), torch.empty_like(zb)
    ok(L.efm_net_gemm(hidden, B, flat, _p(F1), flat, 1, _p(X), B, 1, _p(rz), B, _p(c1), _p(rzb), 1, None))
    ok(L.efm_net_gemm(nout, B, hidden, _p(F2), hidden, 1, _p(rzb), B, 1, _p(rout), B, _p(c2), None, 2, None))
    assert torch.equal(z, rz) and torch.equal(zb, rzb) and torch.equal(out, rout)

    dF2, dc2, dc1 = (torch.full(s, 7.0, device="cuda") for s in ((nout, hidden), (nout,), (hidden,)))
    dzpb = torch.empty_like(zb)
    loss = torch.full((1,), 5.0, dtype=torch.float64, device="cuda")
    args = [_p(t) for t in (out, tg, z, zb, F2, dF2, dc2, dc1, dzpb, loss)] + [B, hidden, nout, 1.0 / (nout * B), None]
    if fits == 1:
        assert L.efm_net_head_backward(*args) != 0
        return
    ok(L.efm_net_head_backward(*args))
    d = lambda t: t.double().cpu()
    u, r = 2.0 ** -23, out - tg
    assert abs(float(loss) - float((d(r) ** 2).mean())) <= 1e-7 * float((d(r) ** 2).mean())
    g = 2 * r * np.float32(1.0 / (nout * B))                    # float32, as the kernel forms it
    gb = d(g.bfloat16())
    assert ((d(dc2) - d(g).sum(1)).abs() <= (B + 3) * u * d(g).abs().sum(1)).all()
    assert ((d(dF2) - gb @ d(zb).T).abs() <= B * u * (gb.abs() @ d(zb).abs().T) + 1e-30).all()
    dz, mag = d(F2).T @ gb, d(F2).abs().T @ gb.abs()
    on = d((z > 0).float())
    assert ((d(dzpb) - dz * on).abs() <= 2.0 ** -8 * (dz * on).abs() + nout * u * mag * on).all()
    assert ((d(dc1) - (dz * on).sum(1)).abs() <= (nout + B) * u * (mag * on).sum(1)).all()
