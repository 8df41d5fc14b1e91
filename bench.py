"""Headline benchmark: G pair-interactions/s of the direct Biot-Savart velocity evaluation.

Workload (one step = one full velocity evaluation): 1,048,576 particles in 64 Lamb-Oseen
blobs acting on themselves (particle targets, kernelu_0v_0b) plus on 65,536 tracers (point
targets, kernelu_0v_0p), Gaussian core, fp32 split-precision pair arithmetic with fp64
accumulation. Inputs are synthetic (seeded) and resident in HBM before timing starts.

Also reported on the same line: the plain fp64 form's rate, the split form's error against
the fp64 sum of every pair (all targets) and against the CPU oracle (a target subsample), the
adjoint/forward time ratio on the 250k-particle / 4,096-probe adjoint workload, the dominant
kernel's roofline position, and the reference CPU path timed on this host.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

# treecode opening angle and expansion order: the fastest pair with error near 1e-10 on the
# 1M-particle blob workload (0.6/28: 1.2e-10 against 0.5/20: 2.7e-10, and faster)
TREE_THETA, TREE_ORDER = 0.6, 28
METRIC = "G pair-interactions/s at N=1M (fp32-split vs fp64, err vs fp64); adjoint/fwd"
PEAK_FP32 = 157.3e12   # MI355X dense FP32 vector, FLOP/s (includes packed FP32)
ORACLE_TARGETS = 4096  # particle targets checked against the CPU oracle (all 1M sources each)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def pair_sum(src, tgt, tr, most=262144):
    """The fp64 velocity of device tensors src at tgt pair by pair: the no-allocation entry, which takes
    no clusters, adding `most` sources and targets at a time."""
    import ctypes

    import torch

    from omega2d_amd._cabi import call
    from omega2d_amd.device import env_for
    u, v = (torch.zeros(tgt[0].numel(), dtype=torch.float64, device=tgt[0].device) for _ in range(2))
    env = env_for(u.device, "gauss", "fp64", "vel")
    p = lambda a: None if a is None else ctypes.c_void_p(a.data_ptr())
    for i in range(0, u.numel(), most):
        cut = slice(i, i + most)
        t = [None if a is None else a[cut].contiguous() for a in (*tgt, tr)]
        for j in range(0, src[0].numel(), most):
            s = [a[j:j + most].contiguous() for a in src]
            call("o2d_hip_points_on_points_noalloc_dev_d", ctypes.byref(env), s[0].numel(),
                 *[p(a) for a in s], t[0].numel(), *[p(a) for a in t], p(u[cut]), p(v[cut]), None, None)
    return u, v


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--fp64-steps", type=int, default=1)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0,
                    help="target CPU time of the bounded reference-baseline sample")
    ap.add_argument("--n", type=int, default=1 << 20, help="particles (default 2^20)")
    ap.add_argument("--only", choices=["split"], default=None,
                    help="run only the split-form steps (short runs under a profiler)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="BYTES",
                    help="run one device-to-device copy of BYTES (HBM counter calibration) "
                         "and exit")
    args = ap.parse_args()
    if args.copy_calibration:
        return copy_calibration(args.copy_calibration)

    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus {args.gpus}); the multi-GPU "
              "layout (targets sharded, sources all-gathered) is a design that is not run here.",
              file=sys.stderr)
        return 2

    import torch
    import omega2d_amd as o2d
    from omega2d_amd import device as dv
    from omega2d_amd import workloads as wl
    from omega2d_amd._cabi import (KT_ADJOINT, KT_NBODY_PLAIN, KT_NBODY_PLAIN_PT,
                                   KT_NBODY_SPLIT, KT_SPLIT_PREP,
                                   timing_enable, timing_read)

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    w = wl.c2_blobs(n=args.n)
    n, nt = len(w["x"]), len(w["tx"])
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    sx, sy, ss, sr = T(w["x"]), T(w["y"]), T(w["s"]), T(w["r"])
    tx, ty = T(w["tx"]), T(w["ty"])
    pairs = float(n) * n + float(nt) * n
    flops_b = o2d.flops_per_pair("gauss", False)   # 19: particle targets
    flops_p = o2d.flops_per_pair("gauss", True)    # 17: point targets
    flops = float(n) * n * flops_b + float(nt) * n * flops_p + 2.0 * (n + nt)
    log(f"workload {w['name']}: {n} particles + {nt} tracers, {pairs:.4e} pairs per step")

    pu = torch.zeros(n, dtype=torch.float64, device=dev)
    pv = torch.zeros_like(pu)
    qu = torch.zeros(nt, dtype=torch.float64, device=dev)
    qv = torch.zeros_like(qu)

    def step(precision):
        pu.zero_()
        pv.zero_()
        qu.zero_()
        qv.zero_()
        dv.points_on_points(sx, sy, ss, sr, sx, sy, sr, core="gauss", precision=precision,
                            tu=pu, tv=pv)
        dv.points_on_points(sx, sy, ss, sr, tx, ty, None, core="gauss", precision=precision,
                            tu=qu, tv=qv)

    # ---- split form: warmup, then exactly K timed steps
    for i in range(args.warmup):
        step("split")
    torch.cuda.synchronize()
    for c in (KT_NBODY_SPLIT, KT_SPLIT_PREP):
        timing_read(c)
    timing_enable(True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        step("split")
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    timing_enable(False)
    k_ms, k_n = timing_read(KT_NBODY_SPLIT)
    prep_ms, prep_n = timing_read(KT_SPLIT_PREP)
    ms_split = (t1 - t0) * 1e3 / args.steps
    value = pairs / (ms_split * 1e-3) / 1e9
    log(f"split: {ms_split:.2f} ms/step, {value:.1f} G-int/s; particle-target kernel "
        f"{k_ms / max(k_n, 1):.3f} ms x{k_n}, prep {prep_ms / max(prep_n, 1):.3f} ms x{prep_n}")
    su, sv_, squ, sqv = (a.cpu().numpy() for a in (pu, pv, qu, qv))
    if args.only == "split":
        print(json.dumps({"only": "split", "ms_per_step": round(ms_split, 3),
                          "value": round(value, 2), "kernel_ms": round(k_ms / max(k_n, 1), 4)}),
              flush=True)
        return 0

    # ---- the same pairs in a random order (particles and tracers each permuted): the kernels
    # sort both internally, so the rate should not depend on the caller's order
    rng_p = np.random.default_rng(7)
    pp, pq = rng_p.permutation(n), rng_p.permutation(nt)
    px_, py_, ps_, pr_ = (T(w[k][pp]) for k in ("x", "y", "s", "r"))
    ptx, pty = T(w["tx"][pq]), T(w["ty"][pq])

    def step_shuffled():
        pu.zero_()
        pv.zero_()
        qu.zero_()
        qv.zero_()
        dv.points_on_points(px_, py_, ps_, pr_, px_, py_, pr_, core="gauss", precision="split",
                            tu=pu, tv=pv)
        dv.points_on_points(px_, py_, ps_, pr_, ptx, pty, None, core="gauss", precision="split",
                            tu=qu, tv=qv)

    step_shuffled()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        step_shuffled()
    torch.cuda.synchronize()
    ms_shuf = (time.perf_counter() - t0) * 1e3 / args.steps
    hu, hv, hqu, hqv = (a.cpu().numpy() for a in (pu, pv, qu, qv))
    err_shuf = float(np.sqrt((np.sum((hu - su[pp]) ** 2) + np.sum((hv - sv_[pp]) ** 2)
                              + np.sum((hqu - squ[pq]) ** 2) + np.sum((hqv - sqv[pq]) ** 2))
                             / (np.sum(su ** 2) + np.sum(sv_ ** 2) + np.sum(squ ** 2)
                                + np.sum(sqv ** 2))))
    log(f"shuffled order: {ms_shuf:.2f} ms/step ({ms_shuf / ms_split:.3f} of the ordered time), "
        f"results vs ordered {err_shuf:.3e}")
    del px_, py_, ps_, pr_, ptx, pty

    # ---- plain fp64 form
    step("fp64")
    torch.cuda.synchronize()
    timing_read(KT_NBODY_PLAIN)
    timing_enable(True)
    t0 = time.perf_counter()
    for i in range(args.fp64_steps):
        step("fp64")
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    timing_enable(False)
    k64_ms, k64_n = timing_read(KT_NBODY_PLAIN)
    ms_64 = (t1 - t0) * 1e3 / args.fp64_steps
    value_64 = pairs / (ms_64 * 1e-3) / 1e9
    fu, fv, fqu, fqv = (a.cpu().numpy() for a in (pu, pv, qu, qv))

    # errors are against the fp64 sum of every pair: the fp64 form and the treecode share their cells
    ref = [a.cpu().numpy() for a in (*pair_sum((sx, sy, ss, sr), (sx, sy), sr),
                                     *pair_sum((sx, sy, ss, sr), (tx, ty), None))]

    def err_of(*got):
        return float(np.sqrt(sum(np.sum((g - r) ** 2) for g, r in zip(got, ref))
                             / sum(np.sum(r ** 2) for r in ref)))

    err_fp64, err_form = err_of(su, sv_, squ, sqv), err_of(fu, fv, fqu, fqv)
    log(f"fp64: {ms_64:.2f} ms/step, {value_64:.1f} G-int/s; split/fp64 = {ms_64 / ms_split:.2f}x;"
        f" err vs fp64 pairs: split {err_fp64:.3e}, fp64 form {err_form:.3e}")

    # ---- split error against the CPU oracle on a target subsample
    err_oracle = None
    try:
        import oracle as O
        rng = np.random.default_rng(0)
        sub = np.sort(rng.choice(n, ORACLE_TARGETS, replace=False))
        ou, ov = O.points_on_points("gauss", w["x"], w["y"], w["s"], w["r"], w["x"][sub],
                                    w["y"][sub], w["r"][sub])
        err_oracle = float(np.sqrt((np.sum((su[sub] - ou) ** 2) + np.sum((sv_[sub] - ov) ** 2))
                                   / (np.sum(ou ** 2) + np.sum(ov ** 2))))
        err64_oracle = float(np.sqrt((np.sum((fu[sub] - ou) ** 2) + np.sum((fv[sub] - ov) ** 2))
                                     / (np.sum(ou ** 2) + np.sum(ov ** 2))))
        log(f"oracle subsample ({ORACLE_TARGETS} targets): split err {err_oracle:.3e}, "
            f"fp64 err {err64_oracle:.3e}")
    except Exception as e:  # the comparison is left out where the oracle is not built
        log(f"oracle check skipped: {e}")
        err64_oracle = None

    # ---- adjoint / forward on the adjoint workload (fp64 both)
    a = wl.c4_adjoint()
    ax, ay, as_, ar, atx, aty = (T(a[k]) for k in ("x", "y", "s", "r", "tx", "ty"))
    au = torch.zeros(len(a["tx"]), dtype=torch.float64, device=dev)
    av = torch.zeros_like(au)
    grads = tuple(torch.zeros(len(a["x"]), dtype=torch.float64, device=dev) for _ in range(4))

    def fwd():
        au.zero_()
        av.zero_()
        dv.points_on_points(ax, ay, as_, ar, atx, aty, None, core="gauss", tu=au, tv=av)

    def adj():
        for g in grads:
            g.zero_()
        dv.points_on_points_adjoint(ax, ay, as_, ar, atx, aty, 2 * au, 2 * av, core="gauss",
                                    out=grads)

    fwd()
    adj()
    torch.cuda.synchronize()
    timing_read(KT_NBODY_PLAIN_PT)
    timing_read(KT_ADJOINT)
    timing_enable(True)
    reps = 5
    t0 = time.perf_counter()
    for i in range(reps):
        fwd()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    for i in range(reps):
        adj()
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    timing_enable(False)
    ms_fwd, ms_adj = (t1 - t0) * 1e3 / reps, (t2 - t1) * 1e3 / reps
    kf_ms, kf_n = timing_read(KT_NBODY_PLAIN_PT)
    ka_ms, ka_n = timing_read(KT_ADJOINT)
    log(f"adjoint workload: fwd {ms_fwd:.3f} ms, adjoint {ms_adj:.3f} ms, ratio {ms_adj / ms_fwd:.2f}")

    # ---- the same evaluation through the treecode (summation_t barneshut, theta 0.6, order 28):
    # time per evaluation and error against the fp64 sum of every pair over every target
    def tree_step():
        pu.zero_()
        pv.zero_()
        qu.zero_()
        qv.zero_()
        dv.points_on_points_tree(sx, sy, ss, sr, sx, sy, sr, core="gauss", theta=TREE_THETA, order=TREE_ORDER,
                                 tu=pu, tv=pv)
        dv.points_on_points_tree(sx, sy, ss, sr, tx, ty, None, core="gauss", theta=TREE_THETA, order=TREE_ORDER,
                                 tu=qu, tv=qv)

    tree_step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        tree_step()
    torch.cuda.synchronize()
    ms_tree = (time.perf_counter() - t0) * 1e3 / args.steps
    err_tree = err_of(*(a.cpu().numpy() for a in (pu, pv, qu, qv)))
    log(f"treecode: {ms_tree:.2f} ms/step, {pairs / (ms_tree * 1e-3) / 1e9:.1f} equivalent "
        f"G-int/s, err vs fp64 {err_tree:.3e}")

    # ---- the other measured configurations: one Ralston RK3 step of 4M particles (C5) and
    # Ralston RK2 steps of the 200k wake around the 2,048-panel circle (C3), device-resident
    del pu, pv, qu, qv, sx, sy, ss, sr, tx, ty
    torch.cuda.empty_cache()
    c5 = c5_rk3_step(T)
    torch.cuda.empty_cache()
    c3 = c3_rk2_steps(T, args.steps)

    # ---- roofline of the dominant kernel: the split launch with particle targets (N x N pairs,
    # 19 flops each in the reference's convention plus 2 per target), timed by the library's
    # HIP events around each such launch on its stream
    main_ms = k_ms / max(k_n, 1)
    flops_main = float(n) * n * flops_b + 2.0 * n
    achieved = flops_main / (main_ms * 1e-3) / 1e12
    roofline = {"bound": "valu", "achieved": round(achieved, 3),
                "peak": PEAK_FP32 / 1e12, "unit": "TFLOP/s",
                "frac": round(achieved * 1e12 / PEAK_FP32, 4),
                "traffic": measured_traffic(),
                "kernel": "nbody32_kernel<Gaussian, particle targets>",
                "flops_per_pair": flops_b, "kernel_ms": round(main_ms, 4)}

    # ---- CPU baseline: the reference's own OpenMP path (S=float, A=double), bounded sample
    cpu = None
    cpu_rows = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(w, args.cpu_seconds)
        cpu_rows = cpu_reference_c3(args.cpu_seconds / 10.0)

    out = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "G pair-interactions/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_split, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "1,048,576 particles in 64 Lamb-Oseen blobs (self, particle "
                               "targets) + 65,536 tracers, Gaussian core sigma=7.8125e-5, one "
                               "velocity evaluation, fp32 split pair math + fp64 accumulation",
                   "particles": n, "tracers": nt, "pairs_per_step": pairs, "core": "gaussian",
                   "parallelism": "single GPU"},
        "fp64_plain": {"value": round(value_64, 2), "ms_per_step": round(ms_64, 3),
                       "kernel_ms": round(k64_ms / max(k64_n, 1), 4),
                       "err_vs_pairs": err_form,
                       "note": "sources beyond the compact cutoff by clusters, to rounding: the "
                               "value is an equivalent rate"},
        "shuffled": {"value": round(pairs / (ms_shuf * 1e-3) / 1e9, 2),
                     "ms_per_step": round(ms_shuf, 3),
                     "time_over_ordered": round(ms_shuf / ms_split, 4),
                     "err_vs_ordered": err_shuf,
                     "note": "the same pairs with particles and tracers randomly permuted"},
        "split_over_fp64": round(ms_64 / ms_split, 3),
        "err_vs_fp64": err_fp64,
        "err_vs_oracle_subsample": err_oracle,
        "fp64_err_vs_oracle_subsample": err64_oracle,
        "adjoint_over_fwd": round(ms_adj / ms_fwd, 3),
        "adjoint_workload": {"particles": len(a["x"]), "probes": len(a["tx"]),
                             "fwd_ms": round(ms_fwd, 3), "adjoint_ms": round(ms_adj, 3),
                             "fwd_kernel_ms": round(kf_ms / max(kf_n, 1), 4),
                             "adjoint_kernel_ms": round(ka_ms / max(ka_n, 1), 4)},
        "split_prep_ms": round(prep_ms / max(prep_n, 1), 4),
        "treecode": {"theta": TREE_THETA, "order": TREE_ORDER, "ms_per_step": round(ms_tree, 3),
                     "equivalent_value": round(pairs / (ms_tree * 1e-3) / 1e9, 1),
                     "err_vs_fp64": err_tree,
                     "note": "same evaluation, O(N log N) with fp64 moments; not the headline"},
        "c5_rk3": c5,
        "c3_rk2": c3,
        "roofline": roofline,
        "cpu_baseline": cpu,
        "cpu_reference_c3": cpu_rows,
    }
    print(json.dumps(out), flush=True)
    return 0


def c5_rk3_step(T):
    """One Ralston RK3 step (src/Convection.h:472-598) of the 4,194,304-particle shear layer:
    three split-form velocity evaluations (Rosenhead-Moore, particle targets) and the fp64
    position updates; the error of the first stage's velocity against the fp64 form on a
    16,384-target subsample."""
    import torch
    from omega2d_amd import device_step as ds
    from omega2d_amd import flops_per_pair, workloads as wl
    from omega2d_amd._cabi import KT_NBODY_SPLIT, timing_enable, timing_read
    w = wl.c5_shear_layer()
    n = len(w["x"])
    x0, y0, s, r = T(w["x"]), T(w["y"]), T(w["s"]), T(w["r"])
    st = ds.Stepper(x0.clone(), y0.clone(), s, r, core="rm", precision="split", fs=w["fs"])
    st.vels(x0, y0)  # untimed: the library's buffers for this size
    torch.cuda.synchronize()
    timing_read(KT_NBODY_SPLIT)
    timing_enable(True)
    t0 = time.perf_counter()
    st.step(w["dt"], 3)
    torch.cuda.synchronize()
    t = time.perf_counter() - t0
    timing_enable(False)
    kms, kn = timing_read(KT_NBODY_SPLIT)
    rng = np.random.default_rng(4)
    sub = torch.from_numpy(np.sort(rng.choice(n, 16384, replace=False))).to(x0.device)
    from omega2d_amd import device as dv
    u6, v6 = dv.points_on_points(x0, y0, s, r, x0[sub].contiguous(), y0[sub].contiguous(),
                                 r[sub].contiguous(), core="rm", precision="fp64")
    c = 0.5 / np.pi
    us, vs = st.stages[0]
    du, dvv = us[sub] - c * u6, vs[sub] - c * v6
    err = float(torch.sqrt((du * du + dvv * dvv).sum() / (c * c * (u6 * u6 + v6 * v6).sum())))
    pairs = float(n) * n
    k_ms = kms / max(kn, 1)
    fl = flops_per_pair("rm", False) * pairs + 2.0 * n
    log(f"C5 RK3 step: {t * 1e3:.1f} ms, {3 * pairs / t / 1e9:.1f} G-int/s; evaluation kernel "
        f"{k_ms:.1f} ms ({fl / (k_ms * 1e-3) / PEAK_FP32:.3f} of FP32 peak); split error vs "
        f"fp64 on 16,384 targets {err:.3e}")
    return {"workload": "4,194,304 particles in a perturbed shear layer, Rosenhead-Moore core "
                        "radius 0.002, one Ralston RK3 step dt=0.01: three split-form evaluations"
                        " + fp64 position updates",
            "ms_per_step": round(t * 1e3, 2), "G_int_s": round(3 * pairs / t / 1e9, 1),
            "eval_kernel_ms": round(k_ms, 3), "evals_timed": kn,
            "frac_fp32_peak": round(fl / (k_ms * 1e-3) / PEAK_FP32, 4),
            "err_vs_fp64_16k": err}


def c3_rk2_steps(T, steps):
    """Ralston RK2 steps (src/Convection.h:390-466) of the 200,000-particle wake around the
    2,048-panel circle (vortex panels, augmented 2049^2 system), all on the device: each stage
    solves the BEM (points on panels, right-hand side, LU solve), sums the wake on itself in the
    split form (Vatistas n=2) and the panels on the wake, moves the wake in fp64 and clears the
    inner layer. The matrix is assembled and factored once (timed as setup)."""
    import torch
    from omega2d_amd import device_step as ds
    from omega2d_amd import workloads as wl
    from omega2d_amd._cabi import (KT_NBODY_SPLIT, KT_NEAR, KT_PANEL_RHS, KT_PANELS,
                                   timing_enable, timing_read)
    w = wl.c3_circle_wake()
    ips = 0.005
    x, y, s, r = T(w["x"]), T(w["y"]), T(w["s"]), T(w["r"])
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    body = ds.Body(w["nx"], w["ny"], w["idx"], nunk=1)
    torch.cuda.synchronize()
    t_setup = time.perf_counter() - t0
    st = ds.Stepper(x, y, s, r, core="v2", precision="split", fs=w["fs"], body=body, ips=ips)
    for _ in range(2):
        st.step(0.01, 2)
    torch.cuda.synchronize()
    cls = {"particles_split": KT_NBODY_SPLIT, "panels_on_particles": KT_PANELS,
           "points_on_panels": KT_PANEL_RHS, "clear_inner": KT_NEAR}
    for c in cls.values():
        timing_read(c)
    timing_enable(True)
    t0 = time.perf_counter()
    for _ in range(steps):
        st.step(0.01, 2)
    torch.cuda.synchronize()
    t = (time.perf_counter() - t0) / steps
    timing_enable(False)
    parts = {k: round(timing_read(c)[0] / steps, 3) for k, c in cls.items()}
    log(f"C3 RK2 step (device path): {t * 1e3:.2f} ms/step, setup {t_setup * 1e3:.1f} ms; "
        f"kernel ms per step {parts}")
    return {"workload": "2,048-panel circle (vortex panels, augmented 2049^2 LU) + 200,000 wake "
                        "particles, Vatistas n=2 split form, Ralston RK2 dt=0.01, inner layer "
                        "cleared at spacing 0.005; device-resident",
            "ms_per_step": round(t * 1e3, 3), "steps": steps,
            "setup_ms": round(t_setup * 1e3, 2), "kernel_ms_per_step": parts}


def measured_traffic():
    """HBM bytes per launch of the dominant kernel, from the FETCH_SIZE / WRITE_SIZE runs
    recorded in profiles/ (each counter scaled by what it reads for a copy of known size)."""
    p = os.path.join(ROOT, "profiles", "nbody32_c2_split.traffic.json")
    try:
        with open(p) as f:
            return json.load(f)["bytes_per_launch"]
    except (OSError, KeyError, ValueError):
        return None


def copy_calibration(nbytes):
    """One device-to-device copy of a known size: FETCH_SIZE/WRITE_SIZE of this dispatch over
    nbytes gives the factor that turns those counters into HBM bytes."""
    import torch
    n = nbytes // 8
    a = torch.ones(n, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes": n * 8}), flush=True)
    return 0


def cpu_baseline(w, seconds):
    """The reference's points_affect_points<float,double> (OpenMP, compiled from its sources by
    oracle/Makefile) on a bounded target sample of the same workload, scaled to pairs/s."""
    try:
        import oracle as O
    except Exception as e:
        log(f"cpu baseline skipped: {e}")
        return None
    threads = int(os.environ.get("OMP_NUM_THREADS", "0")) or len(os.sched_getaffinity(0))
    n = len(w["x"])
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)
    sx, sy, ss, sr = f32(w["x"]), f32(w["y"]), f32(w["s"]), f32(w["r"])
    if O.have_ref("gauss"):
        kind, fn = "reference", lambda m: O.ref_points_on_points(
            sx, sy, ss, sr, sx[:m], sy[:m], sr[:m], "vel", dtype=np.float32, core="gauss")
        label = ("reference points_affect_points<float,double> built with its exponential "
                 "(Gaussian) core define, particle targets, the GPU line's workload")
    else:
        kind, fn = "port", lambda m: O.points_on_points(
            "gauss", w["x"], w["y"], w["s"], w["r"], w["x"][:m], w["y"][:m], w["r"][:m])
        label = "fp64 C restatement, Gaussian core, particle targets"
    m = max(threads * 4, 64)
    t0 = time.perf_counter()
    fn(m)
    dt = time.perf_counter() - t0
    rate = m * float(n) / dt
    m2 = int(min(n, max(m, seconds * rate / n)))
    t0 = time.perf_counter()
    fn(m2)
    dt = time.perf_counter() - t0
    rate = m2 * float(n) / dt
    log(f"cpu baseline ({kind}): {m2} targets x {n} sources in {dt:.2f} s = {rate / 1e9:.3f} "
        f"G-int/s on {threads} threads")
    return {"value": round(rate / 1e9, 4), "unit": "G pair-interactions/s", "cores": threads,
            "kind": kind, "sample": f"{m2} of {n} particle targets x {n} sources, {dt:.1f} s; "
                                    f"{label}; OpenMP x86 env (the Vc env cannot be built offline)"}


def _bounded_rate(fn, total_units, per_call_units, seconds, start=8):
    """Units per second of fn(m) (m targets of per_call_units work each), timed on a sample of
    about `seconds` of CPU work."""
    m = start
    t0 = time.perf_counter()
    fn(m)
    dt = time.perf_counter() - t0
    rate = m * per_call_units / max(dt, 1e-9)
    m = int(min(total_units, max(m, seconds * rate / per_call_units)))
    t0 = time.perf_counter()
    fn(m)
    dt = time.perf_counter() - t0
    return m, dt, m * per_call_units / dt


def cpu_reference_c3(seconds):
    """The reference's own CPU loops (compiled from its sources by oracle/Makefile, OpenMP) for the
    per-stage pieces of the C3 workload (2,048 panels, 200,000 wake particles, Vatistas n=2, the
    reference's compiled-in core), each on a bounded target sample, in (target, source) pairs
    per second. The library's times for the same pieces come from
    `python bench_configs.py --configs c3`."""
    try:
        import oracle as O
        from omega2d_amd import workloads as wl
    except Exception as e:
        log(f"C3 cpu rows skipped: {e}")
        return None
    if not O.have_ref():
        return None
    threads = int(os.environ.get("OMP_NUM_THREADS", "0")) or len(os.sched_getaffinity(0))
    w = wl.c3_circle_wake()
    npan, nw = len(w["idx"]) // 2, len(w["x"])
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    x, y, s, r = f32(w["x"]), f32(w["y"]), f32(w["s"]), f32(w["r"])
    vs = np.full(npan, 1e-3, np.float32)
    rows = {}
    m, dt, rate = _bounded_rate(
        lambda k: O.ref_points_on_points(x, y, s, r, x[:k], y[:k], r[:k], "vel",
                                         dtype=np.float32), nw, nw, seconds, start=64)
    rows["particles_on_particles"] = {"pairs_s": round(rate, 1), "sample": f"{m} targets"}
    m, dt, rate = _bounded_rate(
        lambda k: O.ref_panels_on_points(w["nx"], w["ny"], w["idx"], vs, vs, x[:k], y[:k],
                                         dtype=np.float32), nw, npan, seconds, start=256)
    rows["panels_on_points"] = {"pairs_s": round(rate, 1), "sample": f"{m} targets"}
    m, dt, rate = _bounded_rate(
        lambda k: O.ref_points_on_panels(x, y, s, r, w["nx"], w["ny"], w["idx"][:2 * k],
                                         dtype=np.float32), npan, nw, seconds, start=4)
    rows["points_on_panels"] = {"pairs_s": round(rate, 1), "sample": f"{m} panels"}
    m, dt, rate = _bounded_rate(
        lambda k: O.ref_nearest_distances(w["nx"], w["ny"], w["idx"], w["x"][:k], w["y"][:k]),
        nw, npan, seconds, start=256)
    rows["nearest_distances"] = {"pairs_s": round(rate, 1), "sample": f"{m} targets"}
    log("C3 reference CPU rows: " + ", ".join(f"{k} {v['pairs_s'] / 1e9:.3f} G/s"
                                               for k, v in rows.items()))
    return {"threads": threads, "unit": "(target, source) pairs/s", "workload":
            "C3: 2,048-panel circle, 200,000 wake particles, Vatistas n=2, S=float", **rows}


if __name__ == "__main__":
    sys.exit(main())
