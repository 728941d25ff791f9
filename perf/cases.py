"""What a user's program has the localization library do, as cases that can be timed and compared.

Outputs are the caller's buffers at their full size, with the count of rows in them.

A case names an operation ("op") and its sizes and options:

  localize   one synchronous call on host frames (lm_LocBatchedImg): upload, extraction, fit,
             frame-sorted rows and their statistics back on the host
  extract    ROI extraction of HBM-resident uint16 frames into ROI and WLE records
  fit        one-emitter BFGS fits on the reference's schedule, with CRLB, of extracted ROIs
  cascade    the reference-schedule multi-emitter cascade (1, 2 and 3 emitters) of ROIs extracted
             from dense frames
  converged  converged multi-emitter fits with FP64 model selection and full-Fisher CRLB
  frames     high-density frames to rows through the converged fitter, one HIP graph per batch
  output     what an online flush does with fitted rows: frame-sorted compaction, optionally
             consecutive-frame merging, statistics, rendering into the accumulated image
  train      one forward and backward pass of the warm-start network (its gradient)

listed() holds the measured cases, draw() more of the same ranges.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qc-storm_amd"))
import qcstorm as Q  # noqa: E402

GS2D, AS3D = Q.LOCTYPE_GS2D, Q.LOCTYPE_AS3D


def listed():
    return [
        # the smallest call: one camera frame of a small region, localized while the user focuses
        dict(name="live_256", op="localize", w=256, h=256, frames=1, R=7, loc=GS2D, multi=0, density=0.003),
        # the largest frames of a recording, 32 at a time, the default one frame per batch
        dict(name="extract_2048", op="extract", w=2048, h=2048, frames=32, batch=1, R=7, loc=GS2D, multi=0, density=0.003),
        # the online session fits each time 20,480 ROIs have accumulated (a quarter for astigmatic 3D)
        dict(name="fit_flush", op="fit", n=20480, R=7, loc=GS2D),
        # a recording fitted in one go: the largest call, an odd count
        dict(name="fit_million", op="fit", n=1000003, R=7, loc=GS2D),
        dict(name="fit_flush_3d", op="fit", n=5377, R=9, loc=AS3D),
        # wide PSFs: large ROIs, an ordinary batch of the per-call capacity, ragged
        dict(name="fit_wide", op="fit", n=100001, R=11, loc=GS2D),
        # a flush of dense frames with multi-emitter fitting on
        dict(name="cascade_flush", op="cascade", n=20480, R=7, loc=GS2D, density=0.03),
        # overlapping emitters, converged: an ordinary batch, and the elliptical model's
        dict(name="converged_2d", op="converged", n=262144, R=7, loc=GS2D),
        dict(name="converged_3d", op="converged", n=16461, R=9, loc=AS3D),
        # dense frames end to end on the device
        dict(name="frames_dense", op="frames", w=1024, h=1024, frames=10),
        # a flush's rows on their way out, at the default 5x zoom
        dict(name="output_flush", op="output", n=20480, w=2048, h=2048, loc=GS2D, merge=0),
        # training the warm-start network, at its default batch
        dict(name="train_2048", op="train", n=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["localize", "extract", "fit", "fit", "cascade", "converged", "frames", "output", "train"])
    if op == "localize":
        return dict(op=op, w=_log_int(rng, 96, 1024), h=_log_int(rng, 96, 1024), frames=rng.randint(1, 4),
                    R=rng.choice([5, 7, 7, 9, 11]), loc=rng.choice([GS2D, GS2D, AS3D]), multi=0, density=0.003)
    if op == "extract":
        w, h = _log_int(rng, 200, 2048), _log_int(rng, 200, 2048)
        return dict(op=op, w=w, h=h, frames=_log_int(rng, 1, 32), batch=rng.choice([1, 1, 2, 4]), R=rng.choice([5, 7, 7, 9, 11]),
                    loc=rng.choice([GS2D, GS2D, AS3D]), multi=rng.choice([0, 0, 1]), density=0.003)
    if op == "fit":
        R, loc = rng.choice([5, 7, 7, 9, 11, 13]), rng.choice([GS2D, GS2D, AS3D])
        top = 1000003 * 49 * 176 // (R * R * _evals(loc))   # no more pixel evaluations than the largest listed one
        return dict(op=op, n=_log_int(rng, 300, top), R=R, loc=loc)
    if op == "cascade":
        R, loc = rng.choice([5, 7, 7, 9, 11]), rng.choice([GS2D, GS2D, AS3D])
        return dict(op=op, n=_log_int(rng, 500, 20480 * 49 // (R * R)), R=R, loc=loc, density=0.03)
    if op == "converged":
        if rng.random() < 0.6:
            R = rng.choice([7, 7, 9, 11])
            return dict(op=op, n=_log_int(rng, 1000, 262144 * 49 // (R * R)), R=R, loc=GS2D)
        R = rng.choice([7, 9, 9, 11])
        return dict(op=op, n=_log_int(rng, 500, 16461 * 81 // max(R * R, 81)), R=R, loc=AS3D)
    if op == "frames":
        return dict(op=op, w=_log_int(rng, 200, 1024), h=_log_int(rng, 200, 1024), frames=rng.randint(1, 10))
    if op == "output":
        return dict(op=op, n=_log_int(rng, 500, 400000), w=_log_int(rng, 200, 2048), h=_log_int(rng, 200, 2048),
                    loc=rng.choice([GS2D, GS2D, AS3D]), merge=rng.randint(0, 1))
    return dict(op=op, n=_log_int(rng, 128, 4096))


# ---- inputs ---------------------------------------------------------------------------------
def _params(case, **kw):
    base = dict(QE=1.0, PixelSize=100.0, ROISize=case.get("R", 7), LocType=case.get("loc", GS2D), BatchedImageNum=1)
    if base["LocType"] == AS3D:
        base.update(p1_XGY=-111.11, p1_XLY=-111.11, ZDepthCorrFactor=1.0)
    base.update(kw)
    return Q.default_params(**base)


def _sim(w, h, loc, **kw):
    """Simulator settings; astigmatic emitters are brighter on less background, z over +-500 nm."""
    if loc == AS3D:
        kw = dict(dict(astig=1, photons_min=1000.0, photons_max=8000.0, bg_min=20.0, bg_max=80.0), **kw)
    return Q.default_sim(width=w, height=h, qe=1.0, **kw)


def _frames_dev(sp, seed, first, n):
    f = torch.empty((n, sp.height, sp.width), dtype=torch.int16, device="cuda")
    Q.check(Q.lib().qcs_sim_frames_dev(C.byref(sp), seed, first, n, C.c_void_p(f.data_ptr()), None), "qcs_sim_frames_dev")
    return f


def _rois_dev(sp, seed, n):
    r = torch.empty((n, Q.roi_words(sp.width)), dtype=torch.int16, device="cuda")
    truth = torch.empty((n, max(1, sp.n_per_unit_max), Q.TRUTH_FLOATS), dtype=torch.float32, device="cuda")
    Q.check(Q.lib().qcs_sim_rois_dev(C.byref(sp), seed, n, 1, C.c_void_p(r.data_ptr()), C.c_void_p(truth.data_ptr()), None),
            "qcs_sim_rois_dev")
    return r


def _extracted(ctx, case, seed, n, multi):
    """n ROI records with their WLE records, extracted from simulated frames as a session does."""
    W = 1024 if n < 60000 else 2048
    sp = _sim(W, W, case["loc"], density_per_px=case.get("density", 0.003))
    rois = torch.zeros((n, Q.roi_words(case["R"])), dtype=torch.int16, device="cuda")
    wle = torch.zeros((n, Q.WLE_FLOATS), dtype=torch.float32, device="cuda")
    p = _params(case, ImageWidth=W, ImageHigh=W, MultiEmitterFitEn=multi)
    ctx.set_params(p)
    got, frame = 0, 1
    while got < n:
        step = max(1, min(16, int((n - got) / (0.7 * case.get("density", 0.003) * W * W))))
        f = _frames_dev(sp, seed, frame, step)
        k, _ = ctx.extract_dev(f, step, frame, rois[got:], wle[got:], n - got)
        if k == 0:
            raise RuntimeError("no ROIs in the simulated frames")
        got, frame = got + k, frame + step
    return rois, wle


def _rows(case, seed):
    """Rows as a fit leaves them: frame by frame, one in 25 rejected (all zero), molecules that stay
    on for one or more frames, the values a 10 ms exposure gives."""
    n, w, h, d3 = case["n"], case["w"], case["h"], case["loc"] == AS3D
    g = torch.Generator(device="cuda").manual_seed(seed)

    def u(k, lo=0.0, hi=1.0):
        return lo + (hi - lo) * torch.rand(k, generator=g, device="cuda", dtype=torch.float32)

    per_frame = max(1.0, 0.0027 * w * h)
    nfr = max(1, int(round(n / per_frame)))
    dur = 1 + (u(n) < 0.3).int() + (u(n) < 0.1).int()
    mol = torch.repeat_interleave(torch.arange(n, device="cuda"), dur)[:n]
    start = torch.floor(u(n, 0.0, float(nfr))).int()
    first = torch.cat([torch.ones(1, dtype=torch.bool, device="cuda"), mol[1:] != mol[:-1]])
    idx = torch.arange(n, device="cuda")
    off = idx - torch.cummax(torch.where(first, idx, torch.zeros_like(idx)), 0).values
    frame = start[mol] + off.int() + 1
    sx, sy = u(n, 1.0, 1.6)[mol], u(n, 1.0, 1.6)[mol]
    sy = sy if d3 else sx
    pp = torch.exp(u(n, math.log(40.0), math.log(700.0)))
    bg = u(n, 10.0, 100.0)
    r = torch.zeros((n, Q.REC_FLOATS), dtype=torch.float32, device="cuda")
    r[:, 0] = pp
    r[:, 1] = u(n, 4.0, w - 4.0)[mol] + 0.1 * (u(n) - 0.5)
    r[:, 2] = u(n, 4.0, h - 4.0)[mol] + 0.1 * (u(n) - 0.5)
    r[:, 3] = u(n, -450.0, 450.0)[mol] if d3 else 0.0
    r[:, 4], r[:, 5] = sx, sy
    r[:, 6] = 2.0 * math.pi * pp * sx * sy
    r[:, 7] = bg
    r[:, 8] = pp / torch.sqrt(pp + bg)
    r[:, 9] = 100.0 * sx / torch.sqrt(r[:, 6]) * (1.0 + bg / pp)
    r[:, 10] = 100.0 * sy / torch.sqrt(r[:, 6]) * (1.0 + bg / pp)
    r[:, 11] = frame.float()
    r = r[torch.sort(frame, stable=True).indices].contiguous()
    r[u(n) < 0.04] = 0.0
    return r, int(frame.max().item())


def prepare(case, seed):
    op = case["op"]
    if op == "localize":
        p = _params(case, ImageWidth=case["w"], ImageHigh=case["h"], MultiEmitterFitEn=case["multi"])
        sp = _sim(case["w"], case["h"], case["loc"], density_per_px=case["density"])
        frames = _frames_dev(sp, seed, 1, case["frames"]).cpu().numpy().view(np.uint16)
        # the caller's table of a batch's rows: twice what the density gives
        table = np.zeros((64 + int(2.0 * case["density"] * frames.size), Q.REC_FLOATS), np.float32)
        return dict(case=case, ctx=Q.Context(p), frames=frames, table=table)
    if op == "extract":
        p = _params(case, ImageWidth=case["w"], ImageHigh=case["h"], MultiEmitterFitEn=case["multi"], BatchedImageNum=case["batch"])
        sp = _sim(case["w"], case["h"], case["loc"], density_per_px=case["density"])
        cap = max(256, int(2.0 * case["density"] * case["w"] * case["h"] * case["frames"]))
        return dict(case=case, ctx=Q.Context(p), frames=_frames_dev(sp, seed, 1, case["frames"]), cap=cap,
                    rois=torch.zeros((cap, Q.roi_words(case["R"])), dtype=torch.int16, device="cuda"),
                    wle=torch.zeros((cap, Q.WLE_FLOATS), dtype=torch.float32, device="cuda"))
    if op in ("fit", "cascade"):
        ctx = Q.Context(_params(case))
        multi = int(op == "cascade")
        rois, wle = _extracted(ctx, case, seed, case["n"], multi)
        return dict(case=case, ctx=ctx, rois=rois, wle=wle,
                    loc=torch.zeros(((1 + multi) * case["n"], Q.REC_FLOATS), dtype=torch.float32, device="cuda"))
    if op == "converged":
        R, kw = case["R"], dict(n_per_unit_max=3, min_sep=1.0, max_sep=4.0)
        rois = _rois_dev(_sim(R, R, case["loc"], **kw), seed, case["n"])
        return dict(case=case, ctx=Q.Context(_params(case)), rois=rois,
                    loc=torch.zeros((3 * case["n"], Q.REC_FLOATS), dtype=torch.float32, device="cuda"),
                    sel=torch.zeros(case["n"], dtype=torch.int32, device="cuda"))
    if op == "frames":
        p = _params(case, ImageWidth=case["w"], ImageHigh=case["h"], MultiEmitterFitEn=1)
        sp = _sim(case["w"], case["h"], GS2D, density_per_px=0.02, density_max_per_px=0.05, n_per_unit_max=3, min_sep=1.0, max_sep=2.5)
        st = dict(case=case, ctx=Q.Context(p), frames=_frames_dev(sp, seed, 1, case["frames"]))
        cap = 256 + int(0.038 * case["w"] * case["h"]) * case["frames"]
        st["out"] = torch.zeros((2 * cap, Q.REC_FLOATS), dtype=torch.float32, device="cuda")
        st["n"] = torch.zeros(4, dtype=torch.int32, device="cuda")
        st["start"] = torch.ones(1, dtype=torch.int32, device="cuda")
        st["graph"] = st["ctx"].graph_frames(st["frames"], case["frames"], st["start"], cap, 3, st["out"], st["n"])
        return st
    if op == "output":
        p = _params(case, ImageWidth=case["w"], ImageHigh=case["h"], ConsecFitEn=case["merge"])
        loc, last = _rows(case, seed)
        ctx = Q.Context(p)
        st = dict(case=case, ctx=ctx, loc=loc, last=last, sorted=torch.zeros_like(loc), merged=torch.zeros_like(loc),
                  kept=torch.zeros_like(loc), consec=Q.Consec(ctx) if case["merge"] else None)
        st["img"] = torch.zeros((p.SRImageHigh, p.SRImageWidth), dtype=torch.float32, device="cuda")
        st["zimg"] = torch.zeros_like(st["img"]) if case["loc"] == AS3D else None
        return st
    # train: simulated 1-3 emitter ROIs labelled by the converged fits
    p = _params(case)
    sp = _sim(7, 7, GS2D, n_per_unit_max=3, min_sep=1.0, max_sep=4.0)
    rois = _rois_dev(sp, seed, case["n"])
    labels = torch.zeros((case["n"], 16), dtype=torch.float32, device="cuda")
    Q.Context(p).label_dev(rois, case["n"], labels)
    net = Q.Net(seed=7)
    return dict(case=case, params=p, net=net, rois=rois, labels=labels)


# ---- the calls ------------------------------------------------------------------------------
def run(st):
    case = st["case"]
    op = case["op"]
    if op == "localize":
        rows, info, stats = st["ctx"].loc_batch_sync_info(st["frames"], 1)
        st["table"][:len(rows)] = rows
        return dict(rows=st["table"], count=len(rows), info=info, stats=stats)
    if op == "extract":
        n, found = st["ctx"].extract_dev(st["frames"], case["frames"], 1, st["rois"], st["wle"], st["cap"])
        return dict(rois=st["rois"], wle=st["wle"], count=n, found=found)
    if op in ("fit", "cascade"):
        rows = st["ctx"].fit_dev(st["rois"], st["wle"], case["n"], st["loc"])
        return dict(rows=st["loc"], count=rows)
    if op == "converged":
        st["ctx"].fit_mle_dev(st["rois"], case["n"], 3, st["loc"], st["sel"])
        return dict(rows=st["loc"], sel=st["sel"])
    if op == "frames":
        st["graph"].launch()
        return dict(rows=st["out"], n=st["n"])
    if op == "output":
        ctx, rows = st["ctx"], st["sorted"]
        m = ctx.compact_sorted_dev(st["loc"], case["n"], 1, st["last"], rows)
        ontime = None
        if case["merge"]:
            m, ontime = st["consec"].fit_dev(rows, m, True, st["merged"])
            rows = st["kept"]
            m = ctx.compact_dev(st["merged"], m, rows)
        stats = ctx.loc_stats_dev(rows, m)
        ctx.render_dev(rows, m, st["img"], st["zimg"])
        return dict(rows=rows, count=m, ontime=ontime, stats=stats, img=st["img"], zimg=st["zimg"])
    grad, loss = st["net"].grad_dev(st["params"], st["rois"], st["labels"], case["n"])
    return dict(grad=grad, loss=loss)


# ---- what a pass cannot do without ----------------------------------------------------------
def _evals(loc):
    """Loss evaluations of the one-emitter schedule: P parameters, It iterations."""
    P, It = (6, 11) if loc == AS3D else (5, 8)
    return 2 * P + 12 * It + 2 * P * (It - 1)


def work(case):
    op, R, n = case["op"], case.get("R", 7), case.get("n", 0)
    rec, px = 2 * Q.roi_words(R), R * R
    fit = px * 14.0 * _evals(case.get("loc", GS2D))   # FLOP per one-emitter fit: 14 per pixel of an evaluation
    if op == "localize":
        found = 0.0027 * case["w"] * case["h"] * case["frames"]
        return dict(bytes=2.0 * case["w"] * case["h"] * case["frames"] + found * 48, flops=found * fit)
    if op == "extract":
        npx = case["w"] * case["h"] * case["frames"]
        # 8 x 4 minima and sums of the background, 2 x 5 taps, 8 comparisons
        return dict(bytes=2.0 * npx + 0.0027 * npx * (rec + 24), flops=60.0 * npx)
    if op == "fit":
        return dict(bytes=n * (rec + 24.0 + 48.0), flops=n * fit)
    if op == "cascade":
        # every ROI of dense frames gets at least the two-emitter schedule (AS3D: two elliptical ones)
        P, It = (11, 16) if case["loc"] == AS3D else (8, 13)
        return dict(bytes=n * (rec + 24.0 + 48.0), flops=n * px * 16.0 * (2 * P + 12 * It + 2 * P * (It - 1)))
    if op == "converged":
        # K = 1, 2 and 3 at about 8, 15 and 20 evaluations of loss and gradient (elliptical: 13, 73 and 160)
        ev = (13 + 2 * 73 + 3 * 160) * 55.0 if case["loc"] == AS3D else (8 + 2 * 15 + 0.45 * 3 * 20) * 45.0
        return dict(bytes=n * (rec + 3 * 48.0 + 4.0), flops=n * px * ev)
    if op == "frames":
        npx = case["w"] * case["h"] * case["frames"]
        return dict(bytes=2.0 * npx + 0.018 * npx * 48, flops=60.0 * npx + 0.011 * npx * 64 * 65 * 45.0)
    if op == "output":
        # rows in and out, 49 image pixels read and written per row (twice that with a z plane)
        planes = 2 if case["loc"] == AS3D else 1
        return dict(bytes=n * (96.0 + planes * 49 * 8), flops=n * 49.0 * 25)
    # 432 kFLOP forward per ROI, twice that backward
    return dict(bytes=n * (112.0 + 64.0) + 62192 * 8.0, flops=n * 3 * 432e3)


def tolerance(case):
    op = case["op"]
    if op in ("extract", "fit", "cascade", "converged", "frames"):
        # Whole numbers, or rows gated by acceptance windows and likelihood-ratio thresholds at the
        # end of iterations that amplify the last bit: a fit either takes the same path or another
        # one, and the kernels of one model give each other's rows bit for bit.
        return "exact"
    if op == "localize":
        return dict(rel=1e-6, max=1e-5)   # rows bit for bit; the means come from 64-bit sums in any order
    if op == "output":
        return dict(rel=2e-6, max=2e-5)   # float atomics add the splats of a pixel in any order
    return dict(rel=2e-2, max=0.5)        # bf16 operands with 32-bit accumulation


# ---- the same in 64 bits --------------------------------------------------------------------
def _weights64(s, R, mle):
    d = torch.arange(R, device=s.device, dtype=torch.float64) + 0.5 - R / 2.0
    w = torch.exp(-(d * d)[None, :] / (2.0 * s * s)[:, None])
    return torch.where(mle[:, None], torch.ones_like(w), w)


def _loss64(q, w, x, loc):
    """Weighted Poisson deviance of the scaled parameters x, which it clamps, as the schedule does."""
    R = q.shape[1]
    x.clamp_(min=0.01 if loc == AS3D else 0.0)
    g = torch.arange(R, device=q.device, dtype=torch.float64) + 0.5
    sx, sy, b = x[:, 3] * 0.1, x[:, 4 if loc == AS3D else 3] * 0.1, x[:, -1] * 64.0
    ex = torch.exp(-((g[None, :] - x[:, 1:2]) ** 2) * sx[:, None])
    ey = x[:, 0:1] * 128.0 * torch.exp(-((g[None, :] - x[:, 2:3]) ** 2) * sy[:, None])
    m = ey[:, :, None] * ex[:, None, :] + b[:, None, None]
    return (w * (m - q - q * torch.log(m / q))).sum((1, 2))


def _schedule64(q, w, x, loc):
    """The reference's fixed BFGS schedule: central-difference gradients, eleven halvings of the step."""
    n, P = x.shape
    iters = 11 if loc == AS3D else 8
    D = torch.eye(P, device=q.device, dtype=torch.float64).repeat(n, 1, 1)

    def gradient():
        t, g = x.clone(), torch.zeros_like(x)
        for k in range(P):
            t[:, k] -= 0.002
            lo = _loss64(q, w, t, loc)
            t[:, k] += 0.004
            g[:, k] = (_loss64(q, w, t, loc) - lo) * 250.0
            t[:, k] -= 0.002
        return g

    g = gradient()
    d = -g
    for it in range(iters):
        d = d * (P / d.abs().sum(1, keepdim=True))
        lo = torch.full((n, 1), 1e-5, device=q.device, dtype=torch.float64)
        hi = torch.ones_like(lo)
        L0, L1 = _loss64(q, w, x + d * 1e-4, loc), _loss64(q, w, x + d, loc)
        for k in range(11):
            left = (L0 < L1)[:, None]
            mid = (lo + hi) * 0.5
            hi, lo = torch.where(left, mid, hi), torch.where(left, lo, mid)
            if k == 10:
                break
            L = _loss64(q, w, x + d * torch.where(left, hi, lo), loc)
            L1, L0 = torch.where(left[:, 0], L, L1), torch.where(left[:, 0], L0, L)
        s = d * ((lo + hi) * 0.5)
        x = (x + s).clamp_(min=0.01)
        if it == iters - 1:
            break
        g2 = gradient()
        y = g2 - g
        r = 1.0 / (s * y).sum(1)
        A = torch.eye(P, device=q.device, dtype=torch.float64) - r[:, None, None] * s[:, :, None] * y[:, None, :]
        D = (A @ D @ A.transpose(1, 2).contiguous()) + r[:, None, None] * s[:, :, None] * s[:, None, :]
        g = g2
        d = -(D * g[:, None, :]).sum(2)
    return x


def _crlb64(te, be, sx, sy, G):
    """Position bounds (pixels) from the diagonal Fisher sums with second differences of 0.02 pixels."""
    h = 0.02
    c = torch.arange(G, device=te.device, dtype=torch.float64) - G // 2
    pk = te / (2.0 * math.pi * sx * sy)

    def model(x0, y0):
        e = ((c - x0) ** 2)[None, None, :] / (2 * sx * sx)[:, None, None] + ((c - y0) ** 2)[None, :, None] / (2 * sy * sy)[:, None, None]
        return pk[:, None, None] * torch.exp(-e) + be[:, None, None]

    m0 = model(0.0, 0.0)
    out = []
    for ax in ((h, 0.0), (0.0, h)):
        p, m = model(*ax), model(-ax[0], -ax[1])
        f = ((p + m - 2 * m0) - m0 * (torch.log(p) + torch.log(m) - 2 * torch.log(m0))) / (h * h)
        out.append(torch.sqrt(1.0 / f.sum((1, 2))))
    return out


def _fit64(rois, wle, case, p):
    """Rows of the one-emitter fits of one chunk of ROI records."""
    R, loc = case["R"], case["loc"]
    n, half = rois.shape[0], R // 2
    word = rois.to(torch.int64) & 0xffff
    q = ((word[:, :R * R].double() - p.Offset) * p.KAdc).clamp(min=1.0).reshape(n, R, R)
    hdr = word[:, R * R:].double()
    e = [q[:, :, 0].sum(1), q[:, :, -1].sum(1), q[:, 0].sum(1), q[:, -1].sum(1)]
    bkg = (torch.minimum(e[0], e[1]) + torch.minimum(e[2], e[3])) / 2.0 / R
    amp = q[:, half, half] - bkg
    s = wle[:, 1:5].double()
    mle = wle[:, 5].int() == 0
    one = torch.ones_like(bkg)
    if loc == AS3D:
        wx, wy = s[:, :2].amin(1), s[:, 2:].amin(1)
        x = torch.stack([amp / 128, one * (half + 0.5), one * (half + 0.5), 5.0 / wx ** 2, 5.0 / wy ** 2, bkg / 64], 1)
        cap = torch.where(mle, one * math.inf, one * (R / 1.6 / 2.35))
        wx, wy = torch.minimum(wx, cap), torch.minimum(wy, cap)
    else:
        ws = s.amin(1).clamp(max=R / 2.0 / 2.35)
        x = torch.stack([amp / 128, one * (half + 0.5), one * (half + 0.5), 5.0 / ws ** 2, bkg / 64], 1)
        wx = wy = torch.where(mle, ws, ws / 1.2)
    w = _weights64(wy, R, mle)[:, :, None] * _weights64(wx, R, mle)[:, None, :]
    x = _schedule64(q, w, x, loc)
    pp, bg = x[:, 0] * 128.0, x[:, -1] * 64.0
    sx = torch.sqrt(5.0 / x[:, 3])
    sy = torch.sqrt(5.0 / x[:, 4]) if loc == AS3D else sx
    snr, ms = pp / torch.sqrt(pp + bg), (sx + sy) / 2
    ok = (ms <= R / 1.5 / 2.35)
    if loc == AS3D:
        ok, win = ok & (snr > 3.5) & (ms > 0.8), 2.5
        dd = sx * sx - sy * sy
        up = dd >= 0
        pc = [(getattr(p, "p%d_XGY" % k), getattr(p, "p%d_XLY" % k)) for k in range(5)]
        z = sum(torch.where(up, one * a, one * b) * dd ** k for k, (a, b) in enumerate(pc)) * p.ZDepthCorrFactor
    else:
        ok, win, z = ok & (snr > 4.0) & (ms >= 0.6), 1.5, 0.0 * one
    ok &= ((x[:, 1:3] - R / 2.0).abs() < win).all(1)
    tp = 2.0 * math.pi * pp * sx * sy
    cx, cy = _crlb64(tp, bg + p.ReadNoise_e ** 2, sx, sy, 15 if loc == AS3D else 9)
    bound = (tp > 1.0) & (bg > 1.0)
    cx, cy = torch.where(bound, cx * p.PixelSize, 100.0 * one), torch.where(bound, cy * p.PixelSize, 100.0 * one)
    rows = torch.stack([pp, x[:, 1] - half + hdr[:, 0], x[:, 2] - half + hdr[:, 1], z, sx, sy, tp, bg, snr, cx, cy,
                        hdr[:, 2] + 65536.0 * hdr[:, 3]], 1)
    none = torch.zeros(Q.REC_FLOATS, device=q.device, dtype=torch.float64)
    none[9:11] = 100.0   # a rejected row is zero but for the bound's default
    return torch.where(ok[:, None], rows, none)


def _output64(st, case):
    p, rows = st["ctx"].params, st["loc"].double()
    rows = rows[rows[:, 0] >= 2.0]
    rows = rows[torch.sort(rows[:, 11], stable=True).indices]
    d3 = case["loc"] == AS3D
    z, pix = p.PixelZoom, p.PixelSize / p.PixelZoom
    lp = (rows[:, 9] + rows[:, 10]) / 2 if d3 else rows[:, 9]
    x, y, W, H = rows[:, 1] * z, rows[:, 2] * z, p.SRImageWidth, p.SRImageHigh
    use = (rows[:, 8] >= p.SNR_th) & (lp > 0) & (x > 7) & (x < W - 8) & (y > 7) & (y < H - 8)
    pp = rows[:, 0]
    if not d3:
        pp = torch.where(lp > 30.0, torch.zeros_like(pp), pp)
    s = torch.maximum(lp, torch.full_like(lp, pix / 2)) / pix
    img = torch.zeros(W * H, dtype=torch.float64, device=rows.device)
    zimg = torch.zeros_like(img) if d3 else None
    ix, iy = torch.floor(x), torch.floor(y)
    for a in range(-3, 4):
        for b in range(-3, 4):
            v = pp * torch.exp(-0.5 * ((b - (x - ix)) ** 2 + (a - (y - iy)) ** 2) / (s * s))
            at = ((iy + a) * W + ix + b).long()
            img.index_add_(0, at[use], v[use])
            if d3:
                zimg.index_add_(0, at[use], (v * rows[:, 3])[use])
    table = torch.zeros((case["n"], Q.REC_FLOATS), dtype=torch.float64, device=rows.device)
    table[:len(rows)] = rows
    return dict(rows=table, count=None, ontime=None, stats=None, img=img.reshape(H, W), zimg=None if zimg is None else zimg.reshape(H, W))


def _train64(st):
    """Gradient of the mean loss with every product and sum in 64 bits (no bf16 rounding)."""
    f = torch.nn.functional
    p, n = st["params"], st["rois"].shape[0]
    w = torch.from_numpy(st["net"].params()).cuda().double().requires_grad_(True)
    W1, b1, W2, b2, W3, b3, W4, b4, W5, b5 = torch.split(w, [512, 32, 64 * 288, 64, 64 * 576, 64, 64 * 80, 64, 16 * 64, 16])
    q = ((st["rois"][:, :49].to(torch.int64) & 0xffff).double() - p.Offset) * p.KAdc
    q = q.clamp(min=1.0).reshape(n, 7, 7) / p.QE
    bh = (torch.minimum(q[:, 0].sum(1), q[:, 6].sum(1)) + torch.minimum(q[:, :, 0].sum(1), q[:, :, 6].sum(1))) / 14.0
    sc = (q.amax((1, 2)) - bh).clamp(min=0.0) + 1.0
    x = ((q - bh[:, None, None]) / sc[:, None, None])[:, None]
    k1 = W1.reshape(32, 16)[:, :9].reshape(32, 1, 3, 3)
    k2 = W2.reshape(64, 3, 3, 32).permute(0, 3, 1, 2)
    k3 = W3.reshape(64, 3, 3, 64).permute(0, 3, 1, 2)

    def conv(v, k, b):   # valid 3 x 3, as a sum over the taps
        s = v.shape[2] - 2
        o = sum(torch.tensordot(v[:, :, i:i + s, j:j + s], k[:, :, i, j], ([1], [1])) for i in range(3) for j in range(3))
        return f.relu(o + b).permute(0, 3, 1, 2)

    a = conv(conv(conv(x, k1, b1), k2, b2), k3, b3).reshape(n, 64)
    a = torch.cat([a, (torch.log(sc) * 0.1)[:, None], (bh / sc)[:, None]], 1)
    a = f.relu(a @ W4.reshape(64, 80)[:, :66].t() + b4)
    o = a @ W5.reshape(16, 64).t() + b5
    t = st["labels"].double()
    K = t[:, 0].long()
    use = ((K >= 1) & (K <= 3)).double()
    loss = 4.0 * f.cross_entropy(o[:, :3], (K - 1).clamp(0, 2), reduction="none")
    for k in range(3):
        e = o[:, 3 + 3 * k:6 + 3 * k] - torch.stack([t[:, 1 + 3 * k] / 7, t[:, 2 + 3 * k] / 7, t[:, 3 + 3 * k] / (2 * math.pi * sc)], 1)
        loss = loss + (K > k).double() * (49.0 * (e[:, 0] ** 2 + e[:, 1] ** 2) + e[:, 2] ** 2)
    loss = loss + (o[:, 12] - (t[:, 10] - 1.3)) ** 2 + 10.0 * (o[:, 13] - (t[:, 11] - bh) / sc) ** 2
    loss = (loss * use).sum() / n
    loss.backward()
    return dict(grad=w.grad, loss=float(loss.item()))


def exact(case, seed):
    op = case["op"]
    if op == "fit":
        st = prepare(case, seed)
        step = max(1, 3000000 // (case["R"] ** 2))
        return dict(rows=torch.cat([_fit64(st["rois"][i:i + step], st["wle"][i:i + step], case, st["ctx"].params)
                                    for i in range(0, case["n"], step)]), count=None)
    if op == "output" and not case["merge"]:
        return _output64(prepare(case, seed), case)
    if op == "train":
        return _train64(prepare(case, seed))
    # Extraction gives whole numbers.  The cascade, the converged fits and what is built on them
    # choose between models of their rows, and merging between neighbours: where 64 bits choose
    # otherwise, there are other rows, not other values.
    return None
