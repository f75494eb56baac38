"""Benchmark: plain SIRT on the distance-driven projector pair at 2048^2 x 1800 views.

One step = one fused SIRT iteration  x <- x + C * A^T(R * (b - A x)), x >= 0, with the
FP64 monitors (residual, step size, norm) computed inside the kernels -- the work of one
iteration of algorithms/art.py:sirt (art.py:212, 314-326) on one slice.

Workload: 2048 x 2048 float32 random-ellipse phantom (40 ellipses, seed 2), 1800 views
uniform over [0, 180) degrees, 2048 bins, noiseless b = A x_true computed on the GPU,
SIRT from x = 0.  Inputs are resident in HBM before timing starts.

Metric: Gupdates/s = 2 * N^2 * V * iterations / seconds / 1e9 (one pixel-view update per
projector application).  Prints ONE JSON line.

  python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]
                  [--residual-target 1e-3] [--max-residual-iters M]
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

N, V, ELLIPSES, SEED = 2048, 1800, 40, 2
HBM_PEAK_GBS = 8000.0


def alg_bytes_forward(n, v):
    # gathers (one image value per pixel-view) + x read + b, R read + work write
    return 4.0 * n * n * v + 4.0 * n * n + 3 * 4.0 * v * n


def alg_bytes_back(n, v):
    # gathers (one sinogram value per pixel-view) + work read + x, C read + x write
    return 4.0 * n * n * v + 4.0 * v * n + 3 * 4.0 * n * n


def forward_half_name(fwd_variant):
    """The forward half of a SIRT step at launch shape `fwd_variant`: the transpose for the
    column sweeps, the projection in one launch (views with few candidate pixels per bin staged
    through LDS, the wider ones along diagonals), the SIRT update pass.  Also the key of its
    traffic entry."""
    return ("transpose + dd_fwd_kernel<FAST,STORE,%d> + fwd_epi_kernel<SIRT_FWD>"
            % ([256, 128, 64][fwd_variant]))


def back_half_name(back_variant):
    """The back half (projection with the fused SIRT update) at launch shape `back_variant`."""
    return ("dd_back_kernel<FAST,SIRT_BACK,%d,%d>"
            % tuple([(64, 4), (32, 2), (32, 4), (16, 1)][back_variant]))


def measured_traffic(kernel):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 PMC summary
    (profiles/traffic_dd_sirt_2048x1800.json: FETCH_SIZE and WRITE_SIZE per dispatch,
    each scaled by the factor a 256 MiB copy kernel gives), or None when the summary
    does not cover this kernel."""
    path = os.path.join(ROOT, "profiles", "traffic_dd_sirt_2048x1800.json")
    try:
        with open(path) as f:
            table = json.load(f)
    except (OSError, ValueError):
        return None
    v = table.get("bytes_per_launch", {}).get(kernel)
    return None if v is None else float(v)


def cpu_model():
    """The host CPU's model name and logical core count (Linux /proc/cpuinfo)."""
    name = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    name = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return name, os.cpu_count()


def measured_limiter(kernel_key):
    """Shader counters of the dominant kernels from the committed rocprofv3 summary
    (profiles/counters_dd_sirt_2048x1800.json), or None."""
    path = os.path.join(ROOT, "profiles", "counters_dd_sirt_2048x1800.json")
    try:
        with open(path) as f:
            table = json.load(f)
    except (OSError, ValueError):
        return None
    return table.get("kernels", {}).get(kernel_key)


def cpu_baseline(img, c_angles, budget_views=20):
    """Reference C (radon_dd.c built with its own flags into oracle/_ref) timed on a
    bounded sample: forward + back of `budget_views` evenly spaced views at full N,
    single thread (the reference C is single-threaded)."""
    import numpy as np
    from oracle import ref, radon as O
    sub = np.ascontiguousarray(c_angles[:: max(1, len(c_angles) // budget_views)][:budget_views])
    # the wrapper fftshifts; hand it the list that shifts back to `sub`
    given = np.fft.ifftshift(sub)
    if ref.available("dd", "fast"):
        kind = "reference"
        fwd = lambda: ref.forward("dd", img, given, "fast")
        back = lambda s: ref.back("dd", s, given, "fast")
    else:
        kind = "port"
        fwd = lambda: O.dd_forward(img, given, O.FAST)
        back = lambda s: O.dd_back(s, given, O.FAST)
    t0 = time.perf_counter()
    s = fwd()
    t1 = time.perf_counter()
    back(s)
    t2 = time.perf_counter()
    secs = t2 - t0
    gups = 2.0 * img.shape[0] ** 2 * len(sub) / secs / 1e9
    model, ncpu = cpu_model()
    return {"value": round(gups, 6), "unit": "Gupdates/s", "cores": 1, "kind": kind,
            "cpu_model": model, "host_logical_cpus": ncpu,
            "sample": "forward+back of %d of the %d views at %dx%d (%.1f s fwd, %.1f s back), "
                      "single thread" % (len(sub), len(c_angles), img.shape[0], img.shape[0],
                                          t1 - t0, t2 - t1)}


def sirt_to_residual(plan, x, b, work, stats, bnorm, target, max_iters, check_every=5,
                     weights=None, t0=None):
    """Plain SIRT from x (non-negativity on) until ||A x_k - b|| / ||b|| <= target, the
    norms in FP64 on the GPU.  Each step's forward half computes the residual of the
    iterate entering it; every `check_every` steps the host reads it before the back half,
    and the run stops there with x = x_k, so `iterations` is exactly k.  The R/C setup is
    inside the timed region (``weights`` = (R, C) already computed inside it, with the
    clock started at ``t0``).  Returns the timing record."""
    import torch
    if t0 is None:
        torch.cuda.synchronize()
        t0 = time.perf_counter()
    R, C = plan.sirt_weights() if weights is None else weights
    it, rel = 0, float("inf")
    while True:
        plan.sirt_forward(x, b, R, work, stats=stats)     # residual of x_it
        if it % check_every == 0 or it == max_iters:
            rel = float(stats[0].sqrt()) / bnorm
            if rel <= target or it == max_iters:
                break
        plan.sirt_back(work, C, x, pc_beta=0.0, stats=stats)
        it += 1
    torch.cuda.synchronize()
    return {"target": target, "iterations": it, "seconds": round(time.perf_counter() - t0, 4),
            "reached": rel <= target, "residual": rel, "checked_every": check_every}


WARM_WEIGHTS = os.path.join(ROOT, "iterative_tomographic_reconstruction_algorithms_amd",
                            "weights", "unet_dd_2048x1800.npz")


def warm_start_leg(plan, b, bnorm, target, x_plain, plain_seconds, max_iters, input_iters):
    """The warm-started half of the metric: R/C setup, `input_iters` plain SIRT steps, the
    trained U-Net on that iterate (with plain SIRT's fallback: a non-finite or no-better
    output restarts from zero), then plain SIRT continues to the same residual target.
    Timed end to end (network weights are loaded and the network and its fallback check
    are run once on a zero input before the clock starts, as the one-time set-up).  Also the relative L2 distance of its result
    to the plain leg's result."""
    import torch
    from iterative_tomographic_reconstruction_algorithms_amd import warmstart as W
    net = W.load_weights(WARM_WEIGHTS)
    n, v = plan.npix, plan.nang
    dev = b.device
    work = torch.empty((v, n), dtype=torch.float32, device=dev)
    stats = torch.zeros(3, dtype=torch.float64, device=dev)
    # one-time set-up: the network and the fallback check run once on a zero input (every
    # kernel of the warm start loaded before the clock starts, as the plain leg's are)
    W.warm_start(plan, net, b[None], x_in=torch.zeros((1, n, n), device=dev), pc_beta=0.0)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    R, C = plan.sirt_weights()
    x = torch.zeros((n, n), dtype=torch.float32, device=dev)
    for _ in range(input_iters):
        plan.sirt_iterate(x, b, R, C, work, pc_beta=0.0)
    t1 = torch.cuda.Event(enable_timing=True)
    t2 = torch.cuda.Event(enable_timing=True)
    t1.record()
    x0, fell = W.warm_start(plan, net, b[None], x_in=x[None], pc_beta=0.0)
    t2.record()
    x = x0[0].contiguous()
    rec = sirt_to_residual(plan, x, b, work, stats, bnorm, target, max_iters,
                           weights=(R, C), t0=t0)
    rel = float(torch.linalg.vector_norm((x - x_plain).double())
                / torch.linalg.vector_norm(x_plain.double()))
    ratio = rec["seconds"] / plain_seconds
    return {"weights": os.path.relpath(WARM_WEIGHTS, ROOT), "input_iters": input_iters,
            "continued_iters": rec["iterations"],
            "iterations": input_iters + rec["iterations"], "seconds": rec["seconds"],
            "network_and_fallback_ms": round(t1.elapsed_time(t2), 3),
            "fell_back": bool(fell[0]), "reached": rec["reached"], "residual": rec["residual"],
            "time_vs_plain": round(ratio, 4), "rel_l2_to_plain": rel,
            "targets": {"time_vs_plain_max": round(1 / 3, 4), "rel_l2_to_plain_max": 1e-3},
            "met": {"time": ratio <= 1 / 3, "rel_l2": rel <= 1e-3}}


def _events_ms(fn, reps):
    import torch
    fn()
    torch.cuda.synchronize()
    a = torch.cuda.Event(enable_timing=True)
    b = torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(reps):
        fn()
    b.record()
    b.synchronize()
    return a.elapsed_time(b) / reps


def extra_configs(cpu=True, which=("cfg1", "cfg2", "cfg3", "cfg4", "pdss", "unet")):
    """The other workloads of the benchmark suite, measured on the GPU (opt-in):
    cfg1 ray-driven SIRT 256^2 x 304 x 100 iterations (the one-time system-matrix build
    included; the walks' per-iteration time beside it; the reference C timed on two
    iterations), distance-driven MLEM at 2048^2 x 1800 on Poisson counts, a 64-slice sample of the 1024-slice 1024^2 x 900 stack and the mixed
    256-slice launch through the persistent batch (eager and hipGraph), and CG / ADMM-TV
    per-iteration times at 1024^2 x 720 with 1% Gaussian noise; the pixel-driven and
    slant-stacking pairs at 2048^2 x 1800 ("pdss"); and the warm start's U-Net forward at
    512^2 x 64 and a training step ("unet").  "cfg3full" (not in the default list: about
    2 minutes) runs the whole 1024-slice stack for 100 iterations."""
    import numpy as np
    import torch
    from iterative_tomographic_reconstruction_algorithms_amd import solvers
    from iterative_tomographic_reconstruction_algorithms_amd.batch import Batch, Member
    from iterative_tomographic_reconstruction_algorithms_amd.core import Plan
    from iterative_tomographic_reconstruction_algorithms_amd.phantom import (
        angles_deg, ellipses, ellipsoid_slices)
    dev = torch.device("cuda", 0)
    out = {}

    def dd_plan(n, v):
        return Plan("dd", n, np.fft.fftshift((angles_deg(v) * np.pi / 180).astype(np.float32)))

    if "cfg1" in which:
        # cfg1: ray-driven SIRT, 100 iterations from zero, non-negativity on
        n1, v1 = 256, 304
        img1 = ellipses(n1, 10, seed=1)
        ang1 = (angles_deg(v1) * np.pi / 180).astype(np.float32)
        p1 = Plan("rd", n1, ang1)
        b1 = p1.forward(torch.from_numpy(img1).to(dev))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        mat_bytes = p1.rd_matrix("build")     # what the first iteration call does by itself
        t_build = (time.perf_counter() - t0) * 1e3
        R1, C1 = p1.sirt_weights()
        x1 = torch.zeros((n1, n1), device=dev)
        w1 = torch.empty_like(b1)
        st1 = torch.zeros(3, dtype=torch.float64, device=dev)
        t_it = _events_ms(lambda: p1.sirt_iterate(x1, b1, R1, C1, w1, pc_beta=0.0, stats=st1), 100)
        cfg1 = {"workload": "ray-driven SIRT 256x256, 304 views, 100 iterations, x0=0, pc on",
                "gpu_seconds_100_iters": round((t_it * 100 + t_build) / 1e3, 4),
                "gpu_ms_per_iter": round(t_it, 4),
                "system_matrix_build_ms": round(t_build, 2),
                "system_matrix_bytes": mat_bytes}
        p1.rd_matrix("drop")
        cfg1["gpu_ms_per_iter_walks"] = round(
            _events_ms(lambda: p1.sirt_iterate(x1, b1, R1, C1, w1, pc_beta=0.0, stats=st1), 20), 4)
        if cpu:
            from oracle import ref, radon as O
            b1h = b1.cpu().numpy()
            x1h = np.zeros((n1, n1), np.float32)
            use_ref = ref.available("rd", "fast")
            fw = (lambda z: ref.forward("rd", z, ang1, "fast")) if use_ref else \
                 (lambda z: O.rd_forward(z, ang1, O.FAST))
            bw = (lambda z: ref.back("rd", z, ang1, "fast")) if use_ref else \
                 (lambda z: O.rd_back(z, ang1, O.FAST))
            t0 = time.perf_counter()
            for _ in range(2):   # one SIRT iteration = forward, back, monitoring forward
                r = b1h - fw(x1h)
                x1h = x1h + bw(r)
                fw(x1h)
            secs = (time.perf_counter() - t0) / 2
            cfg1["cpu_seconds_100_iters_extrapolated"] = round(secs * 100, 2)
            cfg1["cpu_kind"] = "reference" if use_ref else "port"
            cfg1["cpu_sample"] = "2 iterations timed single-threaded, x50"
        out["cfg1_rd_sirt_256x304"] = cfg1

    if "cfg2" in which:
        # cfg2 MLEM: Poisson counts I0 * A x / max(A x) with I0 = 1e4, from ones
        n2, v2 = 2048, 1800
        p2 = dd_plan(n2, v2)
        from iterative_tomographic_reconstruction_algorithms_amd import autotune
        autotune.tune(p2, nslices=1, reps=2, use_cache=False)
        ax2 = p2.forward(torch.from_numpy(ellipses(n2, 40, seed=2)).to(dev))
        gen = torch.Generator(device=dev).manual_seed(2)
        b2 = torch.poisson(1e4 * ax2 / ax2.max(), generator=gen)
        inv_d2 = p2.mlem_weights()
        x2 = torch.ones((n2, n2), device=dev)
        w2 = torch.empty_like(b2)
        st2 = torch.zeros(3, dtype=torch.float64, device=dev)
        t_m = _events_ms(lambda: p2.mlem_iterate(x2, b2, inv_d2, w2, stats=st2), 20)
        out["cfg2_dd_mlem_2048x1800"] = {
            "workload": "distance-driven MLEM 2048x2048, 1800 views, Poisson counts (I0 = 1e4), x0 = 1",
            "gpu_ms_per_iter": round(t_m, 4),
            "gupdates_per_s": round(2.0 * n2 * n2 * v2 / (t_m * 1e-3) / 1e9, 1),
            "gpu_seconds_200_iters": round(t_m * 200 / 1e3, 3)}
        del p2, ax2, b2, inv_d2, x2, w2

    if "cfg3" in which:
        # cfg3a: 64 of the 1024 slices of a 1024^2 x 900 ellipsoid stack, one persistent batch
        n3, v3, nz3 = 1024, 900, 64
        p3 = dd_plan(n3, v3)
        vol = torch.from_numpy(ellipsoid_slices(n3, 1024, 60, seed=3000, first=480, count=nz3))
        b3 = p3.forward(vol.to(dev))
        del vol
        m3 = Member(p3, b3)
        bt = Batch([m3], pc_beta=0.0)
        t3 = _events_ms(bt.iterate, 5)
        g3 = bt.graph(iters=1)
        t3g = _events_ms(g3.launch, 5)
        g3.close()
        ups = 2.0 * n3 * n3 * v3 * nz3
        out["cfg3_stack_1024x900"] = {
            "workload": "persistent batched SIRT, 64 of 1024 slices of 1024^2 x 900 views",
            "ms_per_iter": round(t3, 3), "ms_per_iter_graph": round(t3g, 3),
            "gupdates_per_s": round(ups / t3 / 1e6, 1),
            "seconds_100_iters_1024_slices_extrapolated": round(t3 * 16 * 100 / 1e3, 2)}
        bt.close()
        del m3, b3

        # cfg3b: one mixed launch of 256 slices, sizes x view counts, 16 slices each
        members, ups = [], 0.0
        for n in (256, 512, 1024, 2048):
            for v in (180, 360, 720, 1440):
                p = dd_plan(n, v)
                imgs = torch.from_numpy(np.stack([ellipses(n, 10, seed=k) for k in range(2)]))
                b = p.forward(imgs.to(dev)).repeat(8, 1, 1).contiguous()
                members.append(Member(p, b))
                ups += 2.0 * n * n * v * 16
        bm = Batch(members, pc_beta=0.0)
        tm = _events_ms(bm.iterate, 3)
        gm = bm.graph(iters=1)
        tmg = _events_ms(gm.launch, 3)
        gm.close()
        out["cfg3_mixed_256_slices"] = {
            "workload": "one persistent launch: 16 slices each of {256,512,1024,2048}^2 x "
                        "{180,360,720,1440} views", "ms_per_iter": round(tm, 3),
            "ms_per_iter_graph": round(tmg, 3), "gupdates_per_s": round(ups / tm / 1e6, 1)}
        bm.close()
        del members

    if "cfg4" in which:
        # cfg4: CG and ADMM-TV at 1024^2 x 720, Gaussian noise of 1% of the largest value
        n4, v4 = 1024, 720
        p4 = dd_plan(n4, v4)
        from iterative_tomographic_reconstruction_algorithms_amd import autotune
        shapes4 = autotune.tune(p4, nslices=1, reps=2, use_cache=False)
        b4 = p4.forward(torch.from_numpy(ellipses(n4, 10, seed=4)).to(dev))
        gen = torch.Generator(device=dev).manual_seed(4)
        b4 = (b4 + 0.01 * float(b4.max()) * torch.randn(b4.shape, device=dev, generator=gen)).contiguous()
        x4 = torch.zeros((n4, n4), device=dev)
        t_cg = _events_ms(lambda: solvers.cg(p4, x4.clone(), b4, 10), 1) / 10
        t_admm = _events_ms(lambda: solvers.admm_tv(p4, x4.clone(), b4, 5, n_inner=4), 1) / 5
        out["cfg4_cg_admm_1024x720"] = {
            "workload": "CG and ADMM-TV (4 inner CG steps per outer step), 1024^2 x 720, "
                        "1% Gaussian noise, FP64 scalars on the GPU",
            "shapes": {"fwd": shapes4["fwd"], "back": shapes4["back"]},
            "cg_ms_per_iter": round(t_cg, 3), "admm_ms_per_outer_iter": round(t_admm, 3),
            "cg_seconds_300_iters": round(t_cg * 0.3, 2),
            "admm_seconds_300_iters": round(t_admm * 0.3, 2)}
    if "cfg3full" in which:
        # the whole stack: 1024 slices of 1024^2 x 900 views, 100 SIRT iterations in one
        # persistent batch.  The projector's cost does not depend on the content, so the 1024
        # slices are 16 copies of 64 distinct ellipsoid slices (generating 1024 on the host
        # takes minutes); b = A x_true on the GPU.
        n3, v3 = 1024, 900
        p3 = dd_plan(n3, v3)
        base = torch.from_numpy(ellipsoid_slices(n3, 1024, 60, seed=3000, first=480, count=64))
        b3 = torch.empty((1024, v3, n3), dtype=torch.float32, device=dev)
        for k in range(16):
            b3[64 * k:64 * (k + 1)] = p3.forward(base.to(dev))
        del base
        bt = Batch([Member(p3, b3)], pc_beta=0.0)
        bt.iterate()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for it in range(100):
            bt.iterate()
            if (it + 1) % 10 == 0:
                torch.cuda.synchronize()
                print("cfg3full: %d iterations, %.1f s" % (it + 1, time.perf_counter() - t0),
                      file=sys.stderr, flush=True)
        torch.cuda.synchronize()
        secs = time.perf_counter() - t0
        out["cfg3_full_1024x1024x900"] = {
            "workload": "persistent batched SIRT, all 1024 slices of 1024^2 x 900 views, "
                        "100 iterations (after one untimed)",
            "seconds_100_iters": round(secs, 2), "ms_per_iter": round(secs * 10, 2),
            "gupdates_per_s": round(2.0 * n3 * n3 * v3 * 1024 * 100 / secs / 1e9, 1)}
        bt.close()
        del b3
    if "pdss" in which:
        # the facade's other two operator pairs at the headline geometry, method 1
        from iterative_tomographic_reconstruction_algorithms_amd.phantom import angles_deg as _ad
        n5, v5 = 2048, 1800
        ang5 = (_ad(v5) * np.pi / 180).astype(np.float32)
        img5 = torch.from_numpy(ellipses(n5, 40, seed=2)).to(dev)
        res = {}
        for oper in ("pd", "ss"):
            p5 = Plan(oper, n5, ang5, method=1)
            s5 = p5.forward(img5)
            t_f = _events_ms(lambda: p5.forward(img5, out=s5), 2)
            t_b = _events_ms(lambda: p5.back(s5), 2)
            res[oper] = {"forward_ms": round(t_f, 3), "back_ms": round(t_b, 3),
                         "gupdates_per_s": round(2.0 * n5 * n5 * v5 / ((t_f + t_b) * 1e-3) / 1e9, 1)}
            del p5, s5
        out["pd_ss_2048x1800"] = dict(workload="pixel-driven and slant-stacking pairs (method 1), "
                                               "2048^2 x 1800, forward and back per call", **res)
    if "unet" in which:
        # the warm start's network at cfg5's inference shape (512^2, batch 64) and a
        # training step on 8 crops of 256^2; FLOPs of the 3x3 convolutions only
        from iterative_tomographic_reconstruction_algorithms_amd.unet import CONVS, UNet
        net = UNet(seed=0)

        def conv_flops(nb, h, w):
            lvl = {"0": 1, "1": 2, "2": 4, "3": 8}
            return sum(2.0 * nb * (h // lvl[nm[1]]) * (w // lvl[nm[1]]) * co * 9 * ci
                       for nm, ci, co in CONVS)
        img = torch.rand((64, 512, 512), device=dev)
        t_fwd = _events_ms(lambda: net(img), 3)
        del img
        # the weight gradients of every 3x3 layer at the same shape (random BF16 operands)
        from iterative_tomographic_reconstruction_algorithms_amd import _lib as L
        from iterative_tomographic_reconstruction_algorithms_amd.core import stream_handle
        t_wg = 0.0
        lvl = {"0": 1, "1": 2, "2": 4, "3": 8}
        for nm, ci, co in CONVS:
            hh = 512 // lvl[nm[1]]
            xw = torch.randn((64, hh, hh, ci), device=dev).to(torch.bfloat16)
            dyw = torch.randn((64, hh, hh, co), device=dev).to(torch.bfloat16)
            dw = torch.zeros((co, 9, ci), device=dev)
            dbw = torch.zeros(co, device=dev)
            pw = [ctypes.c_void_p(t.data_ptr()) for t in (xw, dyw, dw, dbw)]
            t_wg += _events_ms(lambda: L.check(L.lib().itomo_unet_wgrad(
                pw[0], pw[1], 64, hh, hh, ci, co, pw[2], pw[3], stream_handle()), "wgrad"), 3)
            del xw, dyw, dw, dbw
        xi = torch.rand((8, 256, 256), device=dev)
        yi = torch.rand((8, 256, 256), device=dev)
        t_step = _events_ms(lambda: net.train_step(xi, yi, lr=1e-4), 20)
        f_fwd = conv_flops(64, 512, 512)
        out["unet_512x64"] = {
            "workload": "U-Net forward, 64 images of 512^2 (1.95 M parameters, BF16 on the "
                        "matrix cores); training step on 8 crops of 256^2",
            "forward_ms": round(t_fwd, 3), "conv_tflop_per_forward": round(f_fwd / 1e12, 3),
            "forward_tflops": round(f_fwd / t_fwd / 1e9, 1),
            "wgrad_ms": round(t_wg, 3), "wgrad_tflops": round(f_fwd / t_wg / 1e9, 1),
            "train_step_ms_8x256": round(t_step, 3),
            "train_step_tflops_8x256": round(3 * conv_flops(8, 256, 256) / t_step / 1e9, 1)}
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--residual-target", type=float, default=1e-3)
    ap.add_argument("--pmc-calibration", action="store_true",
                    help="after the timed steps, copy a 256 MiB float32 array 3 times "
                         "(a kernel of known traffic for scaling FETCH_SIZE / WRITE_SIZE)")
    ap.add_argument("--extra-configs", action="store_true",
                    help="also measure the other configurations of the suite (minutes)")
    ap.add_argument("--extra-only", default="cfg1,cfg2,cfg3,cfg4,pdss,unet",
                    help="with --extra-configs: the configurations to run (comma list)")
    ap.add_argument("--no-warm-start", dest="warm_start", action="store_false",
                    help="skip the warm-started leg (runs when the trained weights exist)")
    ap.add_argument("--warm-input-iters", type=int, default=40,
                    help="plain SIRT steps before the network (the network's input)")
    ap.add_argument("--max-residual-iters", type=int, default=600,
                    help="also time plain SIRT from zero to the residual target, the R/C "
                         "setup included, for at most this many iterations (0: skip)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the library has no multi-GPU path (--gpus %d "
              "requested)" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    from iterative_tomographic_reconstruction_algorithms_amd import autotune
    from iterative_tomographic_reconstruction_algorithms_amd.core import Plan
    from iterative_tomographic_reconstruction_algorithms_amd.phantom import angles_deg, ellipses

    torch.cuda.set_device(0)
    dev = torch.device("cuda", 0)
    img = ellipses(N, ELLIPSES, seed=SEED)
    facade = (angles_deg(V) * np.pi / 180).astype(np.float32)
    c_angles = np.fft.fftshift(facade)
    plan = Plan("dd", N, c_angles)
    # launch shapes from the autotuner (timed here, not read from a cache)
    shapes = autotune.tune(plan, nslices=1, reps=2, use_cache=False)
    x_true = torch.from_numpy(img).to(dev)
    b = plan.forward(x_true)
    R, C = plan.sirt_weights()
    x = torch.zeros((N, N), dtype=torch.float32, device=dev)
    work = torch.empty((V, N), dtype=torch.float32, device=dev)
    stats = torch.zeros(3, dtype=torch.float64, device=dev)
    bnorm = float(torch.linalg.vector_norm(b.double()))

    for _ in range(args.warmup):
        plan.sirt_iterate(x, b, R, C, work, pc_beta=0.0, stats=stats)
    torch.cuda.synchronize()

    K = args.steps
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3 * K)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(K):
        ev[3 * k].record()
        plan.sirt_forward(x, b, R, work, stats=stats)
        ev[3 * k + 1].record()
        plan.sirt_back(work, C, x, pc_beta=0.0, stats=stats)
        ev[3 * k + 2].record()
    torch.cuda.synchronize()
    secs = time.perf_counter() - t0
    fwd_ms = sum(ev[3 * k].elapsed_time(ev[3 * k + 1]) for k in range(K)) / K
    back_ms = sum(ev[3 * k + 1].elapsed_time(ev[3 * k + 2]) for k in range(K)) / K
    ms_per_step = secs * 1e3 / K
    gups = 2.0 * N * N * V * K / secs / 1e9
    resid_rel = float(stats[0].sqrt()) / bnorm

    fwd_name = forward_half_name(shapes["fwd"])
    back_name = back_half_name(shapes["back"])
    if back_ms >= fwd_ms:
        dom, dom_ms, dom_bytes = back_name, back_ms, alg_bytes_back(N, V)
    else:
        dom, dom_ms, dom_bytes = fwd_name, fwd_ms, alg_bytes_forward(N, V)
    achieved = dom_bytes / (dom_ms * 1e-3) / 1e9
    pair_gbs = (alg_bytes_forward(N, V) + alg_bytes_back(N, V)) / ((fwd_ms + back_ms) * 1e-3) / 1e9
    line = {
        "metric": "SIRT Gupdates/s & s-to-residual 1e-3 (plain vs warm-start) @2048²×1800 views",
        "value": round(gups, 3),
        "unit": "Gupdates/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32 (FP64 monitors)",
        "data": "synthetic",
        "config": {"workload": "plain SIRT, distance-driven pair, 2048x2048 image, 1800 views "
                               "over [0,180), 2048 bins, 40-ellipse phantom (seed 2), noiseless, "
                               "x0=0, non-negativity on", "npix": N, "nang": V, "slices": 1,
                   "shapes": {"fwd": shapes["fwd"], "back": shapes["back"],
                              "fwd_ms": shapes["fwd_ms"], "back_ms": shapes["back_ms"]}},
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": round(achieved, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                     "traffic": measured_traffic(dom),
                     # achieved counts algorithmic bytes: one 4-byte operand gather per
                     # pixel-view plus the compulsory streams; the gathers are served by
                     # LDS and L2, so HBM moves far less (traffic) and the kernels are
                     # limited by VALU issue and LDS (measured below)
                     "accounting": "algorithmic bytes: 4 B gathered per pixel-view + compulsory "
                                   "input/output streams, per launch",
                     "limiter": {"forward": measured_limiter("forward_one_launch"),
                                 "back": measured_limiter("back")},
                     "pair": {"what": "forward + back of one SIRT step",
                              "alg_bytes": alg_bytes_forward(N, V) + alg_bytes_back(N, V),
                              "achieved": round(pair_gbs, 1),
                              "frac": round(pair_gbs / HBM_PEAK_GBS, 4)}},
        "kernels_ms": {"sirt_forward": round(fwd_ms, 4), "sirt_back": round(back_ms, 4)},
        "residual_after_timed_steps": resid_rel,
    }

    if args.pmc_calibration:
        src = torch.rand(64 << 20, device=dev)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        line["pmc_calibration"] = {"copy_bytes_read": src.numel() * 4,
                                   "copy_bytes_written": dst.numel() * 4}

    if args.max_residual_iters > 0:
        x.zero_()
        torch.cuda.synchronize()
        plain = sirt_to_residual(plan, x, b, work, stats, bnorm, args.residual_target,
                                 args.max_residual_iters)
        line["plain_sirt_to_residual"] = plain
        if args.warm_start and os.path.exists(WARM_WEIGHTS):
            line["warm_sirt_to_residual"] = warm_start_leg(
                plan, b, bnorm, args.residual_target, x.clone(), plain["seconds"],
                args.max_residual_iters, args.warm_input_iters)

    if args.extra_configs:
        line["extra"] = extra_configs(cpu=not args.no_cpu_baseline,
                                      which=tuple(args.extra_only.split(",")))

    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(img, c_angles)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
