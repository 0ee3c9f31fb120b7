"""Training data, training loop and the A/B test of the learned initializer.

Data: gathers of one random layered model (workloads.c5) generated by the
batched propagator (one ShotBatch of many sources, hipGraph time loop), packed
on the device into normalised BF16 network inputs (efm_net_pack_gathers).

A/B: on held-out sources the moment tensor is inverted with L-BFGS (lbfgs.py
semantics) on the exact adjoint gradient from the reference's fixed start
Mmod = (0.5, 0, 0.5, 0, 0.5, 0) (M:2777) and from the network's proposal, (a)
at the catalogue location (the reference's setting: fwi_Mij M:2217-2346 inverts
M at a known location) and (b) with the location unknown (plain: the centre of
the source range; network: its predicted location).  Every start is first
scaled by the least-squares factor (the network sees peak-normalised data and
proposes a direction only).  The misfit is quadratic in M, so each step uses
the exact line search α = -gᵀp / ‖F p‖² (one forward of the direction).
Reported: iterations until J ≤ tol · J(plain start) per setting.

    python -m elastic_fm_vp_vs_rho_amd.initnet_data --shots 12288 --heldout 8
"""
from __future__ import annotations

import argparse
import json
import sys
import time

import numpy as np
import torch

from . import _capi, autotune, lbfgs, workloads
from . import model as M
from .initnet import InitNet, NetSpec, pack_gathers
from .propagator import Grid, Propagator, ShotBatch, _ptr, _stream, lame

PLAIN_START = np.array([0.5, 0.0, 0.5, 0.0, 0.5, 0.0])


def targets_of(src, m6, lo, hi):
    """(S, 9): the normalised MT and the source position scaled to [-1, 1] over [lo, hi)."""
    pos = 2.0 * (np.asarray(src, np.float64) - lo) / float(hi - 1 - lo) - 1.0
    return np.concatenate([np.asarray(m6, np.float64), pos], 1).astype(np.float32)


def decode(out, lo, hi):
    """Network output rows -> (unit-Frobenius MT (S, 6), integer positions (S, 3))."""
    out = np.asarray(out, np.float64)
    m = out[:, :6]
    fro = np.sqrt((m[:, :3] ** 2).sum(1) + 2 * (m[:, 3:] ** 2).sum(1))
    m = m / np.where(fro > 0, fro, 1.0)[:, None]
    pos = np.rint((out[:, 6:] + 1.0) / 2.0 * (hi - 1 - lo) + lo).astype(np.int64)
    return m, np.clip(pos, lo, hi - 1)


class C5:
    """The C5 model on the device and shot batches drawn from it."""

    def __init__(self, wl, device="cuda"):
        self.wl, self.dev = wl, torch.device(device)
        self.grid = Grid(wl.nx, wl.ny, wl.nz, wl.dx, wl.dt, (wl.W,) * 6)
        f = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)
        self.rho = f(wl.rho)
        self.lam, self.mu = lame(f(wl.vp), f(wl.vs), self.rho)
        f0 = float(wl.f0[0])
        if np.any(wl.f0 != f0) or np.any(wl.nt != wl.nt[0]):
            raise ValueError("C5 shots share one wavelet and record length")
        self.nt = int(wl.nt[0])
        self.wavelet = M.ricker(f0, wl.dt, self.nt)
        self.cp = M.cpml_coefficients(wl.W, f0, wl.dt, wl.dx, wl.vmax, wl.nx, wl.ny, wl.nz,
                                      free_top=wl.free_top)
        self.rec = wl.rec[0]
        self.lo, self.hi = wl.extra["src_range"]

    def propagator(self, src, m6):
        S = len(src)
        sh = ShotBatch(self.grid, src, m6, np.broadcast_to(self.wavelet, (S, self.nt)),
                       np.full(S, self.nt), np.broadcast_to(self.rec, (S,) + self.rec.shape),
                       self.cp, device=self.dev)
        return Propagator(self.grid, self.lam, self.mu, self.rho, sh)

    def generate(self, idx, length, batch=256, graph_chunk=64, log=None, tune=False):
        """Network dataset (N, 3·nrec, length) BF16 and targets (N, 9) for shots idx.
        tune: autotune the forward sweeps on the first batch (cached per shape)."""
        idx = np.asarray(idx)
        nrec = self.rec.shape[0]
        data = torch.empty((len(idx), 3 * nrec, length), dtype=torch.bfloat16, device=self.dev)
        t0 = time.perf_counter()
        for i in range(0, len(idx), batch):
            part = idx[i:i + batch]
            prop = self.propagator(self.wl.src[part], self.wl.m6[part])
            if tune and i == 0:
                autotune.tune(prop, kernels=(0, 1))
                t0 = time.perf_counter()
            g, _ = prop.forward(graph_chunk=graph_chunk)
            pack_gathers(g, length, data, i)
            del prop, g
            if log:
                torch.cuda.synchronize()
                log(f"[c5] generated {i + len(part)}/{len(idx)} shots, "
                    f"{time.perf_counter() - t0:.1f} s")
        torch.cuda.synchronize()
        secs = time.perf_counter() - t0
        tg = torch.as_tensor(targets_of(self.wl.src[idx], self.wl.m6[idx], self.lo, self.hi),
                             device=self.dev)
        return data, tg, secs


def train(net: InitNet, data, targets, train_idx, val_idx, epochs, batch=64, lr=1e-3, seed=0,
          log=None, graph=True):
    """Adam on mini-batches (each step one hipGraph replay + one Adam launch when
    graph=True); returns per-epoch (train loss, validation loss)."""
    gen = torch.Generator(device=net.dev).manual_seed(seed)
    tr = torch.as_tensor(np.asarray(train_idx, np.int32), device=net.dev)
    va = torch.as_tensor(np.asarray(val_idx, np.int32), device=net.dev)
    hist = []
    nb = len(train_idx) // batch
    for ep in range(epochs):
        perm = tr[torch.randperm(len(tr), generator=gen, device=net.dev)]
        tot = torch.zeros(1, dtype=torch.float64, device=net.dev)
        for b in range(nb):
            tot += net.train_step(data, targets, perm[b * batch:(b + 1) * batch], lr, graph=graph)
        tl = float(tot) / max(nb, 1)
        vl = net.evaluate(data, targets, va)
        hist.append((tl, vl))
        if log:
            log(f"[train] epoch {ep + 1}/{epochs} train {tl:.4f} val {vl:.4f}")
    return hist


def _scale(prop, obs, m6):
    """Least-squares amplitude of the start direction m6 (one forward)."""
    prop.shots.set_m6(m6[None])
    g, _ = prop.forward()
    den = float((g.double() ** 2).sum())
    return float((g.double() * obs.double()).sum()) / den if den > 0 else 1.0


def invert_mt(prop, obs, m0, iters=12, layers=5):
    """L-BFGS on M (exact adjoint gradient, exact line search).  Returns the
    misfit after 0, 1, .. iterations and the final M."""
    m = np.asarray(m0, np.float64).copy()
    sk = np.zeros((layers, 6))
    yk = np.zeros((layers, 6))
    Js = []
    for it in range(iters + 1):
        prop.shots.set_m6(m[None])
        J, _, _, _, _, gm6 = prop.gradient(obs, strategy="auto")
        prop.release_states()
        Js.append(J)
        if it == iters:
            break
        g = gm6[0].double().cpu().numpy()
        lbfgs.compute_sk_yk(sk, yk, m, g, layers, it)
        p = -(g if it == 0 else lbfgs.L_BFGS(sk, yk, g, layers, it))
        prop.shots.set_m6(p[None])
        fp, _ = prop.forward()
        den = float((fp.double() ** 2).sum())
        if den <= 0:
            break
        m = m + (-float(np.dot(g, p)) / den) * p
    return Js, m


def ab_test(c5: C5, net: InitNet, data, heldout, iters=12, tols=(1e-2, 1e-3), log=None):
    """Iterations-to-misfit on held-out shots, in two settings.

    catalogue: the source location is known (the reference's setting); plain
    start Mmod vs the network's MT.  unknown: plain start Mmod at the centre of
    the source range vs the network's MT at the network's location.  In each
    setting J0 is the misfit of the plain start; a run reaches tol when
    J <= tol·J0 (None if it never does within ``iters``)."""
    pred = net.predict(data)            # rows of `data` are the held-out shots, in order
    pm, ppos = decode(pred.cpu().numpy(), c5.lo, c5.hi)
    centre = np.full(3, (c5.lo + c5.hi - 1) // 2)
    out = []
    for j, s in enumerate(heldout):
        true_src = c5.wl.src[s]
        obs, _ = c5.propagator(true_src[None], c5.wl.m6[s][None]).forward()
        obs = obs.clone()
        runs = {}
        for name, pos, d in (("catalogue/plain", true_src, PLAIN_START),
                             ("catalogue/network", true_src, pm[j]),
                             ("unknown/plain", centre, PLAIN_START),
                             ("unknown/network", ppos[j], pm[j])):
            prop = c5.propagator(np.asarray(pos)[None], d[None])
            a = _scale(prop, obs, d)
            runs[name], _ = invert_mt(prop, obs, a * d, iters)
            del prop
        rec = dict(shot=int(s), J=runs, loc_err_cells=float(np.linalg.norm(ppos[j] - true_src)),
                   centre_err_cells=float(np.linalg.norm(centre - true_src)), iters_to_tol={})
        for setting in ("catalogue", "unknown"):
            J0 = runs[f"{setting}/plain"][0]
            for tol in tols:
                for who in ("plain", "network"):
                    Js = runs[f"{setting}/{who}"]
                    rec["iters_to_tol"][f"{setting}/{who}@{tol:g}"] = next(
                        (i for i, J in enumerate(Js) if J <= tol * J0), None)
        out.append(rec)
        if log:
            log(f"[ab] shot {s}: location error {rec['loc_err_cells']:.1f} cells (centre "
                f"{rec['centre_err_cells']:.1f}); iterations to tol: {rec['iters_to_tol']}")
    return out


def joint_ab(c5: C5, net: InitNet, data, heldout, iters=12, sigma=3.0, tols=(1e-1, 3e-2, 1e-2),
             log=None):
    """The network seeding the joint L-BFGS of Vp, Vs, ρ and every shot's MT (the
    C4 method, fwi.invert) on the held-out shots: start model = the true model
    smoothed (Gaussian, `sigma` cells), start MTs = Mmod (plain) or the network's
    proposals (at the catalogue locations), each scaled by least squares in the
    start model.  Returns the misfit histories and the
    iterations to tol·J0, J0 = the plain start's misfit."""
    import dataclasses
    from scipy.ndimage import gaussian_filter
    from . import fwi
    wl = c5.wl
    hd = np.asarray(heldout)
    sub = dataclasses.replace(wl, name=wl.name + " (held-out shots)", src=wl.src[hd], m6=wl.m6[hd],
                              f0=wl.f0[hd], nt=wl.nt[hd], rec=wl.rec[hd])
    survey = fwi.Survey(sub, c5.dev)
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device=c5.dev)
    batch = len(hd)
    obs = fwi.observed(survey, f(wl.vp), f(wl.vs), f(wl.rho), sub.m6, batch)
    smooth = lambda a: gaussian_filter(np.asarray(a, np.float64), sigma, mode="nearest")
    vp0, vs0, rho0 = f(smooth(wl.vp)), f(smooth(wl.vs)), f(smooth(wl.rho))
    pm, _ = decode(net.predict(data).cpu().numpy(), c5.lo, c5.hi)

    def ls_scaled(m60):                 # per-shot least-squares amplitude in the start model
        g = fwi.observed(survey, vp0, vs0, rho0, m60, batch).double()
        o = obs.double()
        a = (g * o).flatten(1).sum(1) / (g * g).flatten(1).sum(1).clamp_min(1e-300)
        return m60 * a.cpu().numpy()[:, None]

    hist = {}
    for name, d in (("plain", np.tile(PLAIN_START, (len(hd), 1))), ("network", pm)):
        h, _ = fwi.invert(survey, vp0, vs0, rho0, ls_scaled(d), obs, iters, batch, log=log)
        hist[name] = [float(J) for J in h]
        survey.release_states()
    J0 = hist["plain"][0]
    reach = {f"{who}@{tol:g}": next((i for i, J in enumerate(hist[who]) if J <= tol * J0), None)
             for tol in tols for who in ("plain", "network")}
    return dict(J=hist, iters_to_tol=reach, final_J_over_J0={k: v[-1] / J0 for k, v in hist.items()},
                start_sigma_cells=sigma, shots=int(len(hd)))


def summarize_ab(ab, iters):
    """Median iterations to each tolerance (a run that never reaches it counts iters+1)."""
    keys = ab[0]["iters_to_tol"].keys()
    med = {k: float(np.median([r["iters_to_tol"][k] if r["iters_to_tol"][k] is not None else iters + 1
                               for r in ab])) for k in keys}
    reached = {k: int(sum(r["iters_to_tol"][k] is not None for r in ab)) for k in keys}
    final = {k: float(np.median([r["J"][k][-1] / r["J"][k.split("/")[0] + "/plain"][0] for r in ab]))
             for k in ab[0]["J"]}
    return dict(median_iters_to_tol=med, runs_reaching_tol=reached, median_final_J_over_J0=final)


def gemm_rate(net: InitNet, B, reps=50):
    """Throughput of the first convolution's forward pass (the largest GEMM; over the
    stored im2col matrix where the net keeps one) at batch B, timed with HIP events on
    the library's stream."""
    s = net.spec
    ci, co, Lin, lo = s.convs()[0]
    b = net._buffers(B)
    K, N = ci * s.ks, B * lo
    if "col0" in b:
        yb = b["yb0"] if s.nblocks > 1 else b["yb_last"]
        call = lambda: net._gemm(co, N, K, net.wb["W0"], K, 1, b["col0"], N, 1, b["y0"], N, bias=net.w["b0"],
                                 Cb=yb, epi=1)
    else:
        yb = b["yb0"] if s.nblocks > 1 else b["X"]
        call = lambda: _capi.check(net.L.efm_net_conv1d(
            _ptr(b["x"]), _ptr(net.wb["W0"]), _ptr(net.w["b0"]), _ptr(b["y0"]), _ptr(yb), ci, B, Lin, co, s.ks,
            s.stride, s.pad, int(s.nblocks == 1), _stream()), "efm_net_conv1d")
    call()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        call()
    e1.record()
    e1.synchronize()
    ms = e0.elapsed_time(e1) / reps
    return {"M": co, "N": N, "K": K, "ms": ms, "tflops": 2.0 * co * N * K / (ms * 1e-3) / 1e12}


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--n", type=int, default=96)
    ap.add_argument("--nt", type=int, default=1024)
    ap.add_argument("--shots", type=int, default=12288, help="training + validation shots")
    ap.add_argument("--heldout", type=int, default=8)
    ap.add_argument("--epochs", type=int, default=40)
    ap.add_argument("--batch", type=int, default=64)
    ap.add_argument("--lr", type=float, default=1e-3)
    ap.add_argument("--ab-iters", type=int, default=12)
    ap.add_argument("--no-graph", action="store_true", help="launch training steps eagerly")
    ap.add_argument("--joint-iters", type=int, default=12,
                    help="iterations of the joint Vp/Vs/rho/MT A/B (0: skip it)")
    args = ap.parse_args(argv)
    log = lambda s: print(s, file=sys.stderr, flush=True)
    dev = torch.device("cuda:0")
    total = args.shots + args.heldout
    wl = workloads.c5(n=args.n, S=total, nt=args.nt)
    c5 = C5(wl, dev)
    data, tg, gen_s = c5.generate(np.arange(args.shots), args.nt, log=log, tune=True)
    cell_steps = float(wl.nx * wl.ny * wl.nz) * args.nt * args.shots
    spec = NetSpec(cin=3 * c5.rec.shape[0], length=args.nt)
    net = InitNet(spec, seed=0, device=dev)
    nval = max(args.shots // 16, args.batch)
    tr, va = np.arange(nval, args.shots), np.arange(nval)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    hist = train(net, data, tg, tr, va, args.epochs, args.batch, args.lr, log=log,
                 graph=not args.no_graph)
    torch.cuda.synchronize()
    train_s = time.perf_counter() - t0
    steps = args.epochs * (len(tr) // args.batch)
    vai = torch.as_tensor(va.astype(np.int32), device=dev)
    err = (net.predict(data, vai) - tg[vai.long()]) ** 2
    mse_mt, mse_loc = float(err[:, :6].mean()), float(err[:, 6:].mean())
    gemm = gemm_rate(net, args.batch)
    hd = np.arange(args.shots, total)
    hdata, _, _ = c5.generate(hd, args.nt, log=None)
    ab = ab_test(c5, net, hdata, hd, iters=args.ab_iters, log=log)
    jab = None if args.joint_iters <= 0 else joint_ab(c5, net, hdata, hd, iters=args.joint_iters, log=log)
    base = float(((tg[torch.as_tensor(va, device=dev)] - tg[torch.as_tensor(tr, device=dev)].mean(0))
                  ** 2).mean())
    rep = {
        "workload": wl.name, "train_shots": int(len(tr)), "val_shots": int(len(va)),
        "heldout_shots": int(len(hd)),
        "generation_s": gen_s, "generation_cell_steps_per_s": cell_steps / gen_s,
        "epochs": args.epochs, "batch": args.batch, "train_graph": not args.no_graph,
        "train_s": train_s,
        "train_examples_per_s": steps * args.batch / train_s,
        "train_tflops": 3 * spec.flops_per_example() * steps * args.batch / train_s / 1e12,
        "val_mse_first_last": [hist[0][1], hist[-1][1]], "val_mse_predict_mean": base,
        "val_mse_mt": mse_mt, "val_mse_location": mse_loc, "gemm_conv1": gemm,
        "ab_summary": summarize_ab(ab, args.ab_iters),
        "ab": ab,
        "joint_ab": jab,
        "loc_err_cells_mean": float(np.mean([r["loc_err_cells"] for r in ab])),
        "centre_err_cells_mean": float(np.mean([r["centre_err_cells"] for r in ab])),
    }
    print(json.dumps(rep))


if __name__ == "__main__":
    main()
