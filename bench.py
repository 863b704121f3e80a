#!/usr/bin/env python
"""Throughput of the Position-Based Fluids step on one MI355X.

Workload (the headline configuration): a 1,000,000-particle dam break -- a 100^3 lattice at
spacing 0.05 with +-0.005 seeded jitter in a [0,10]x[0,6]x[0,5] box, rest density 6378, h = 0.1,
relaxation 600, artificial pressure k = 0.1, n = 4, delta_q = 0.2 h, XSPH c = 0.01,
dt = 0.0083, gravity -9.8 y, 4 Jacobi iterations -- stepped by the HIP solver (libakua.so)
with its inputs resident in HBM.  A step is one PBFSolver::step (predict, hash, sort, neighbour
lists, 4 x (density/lambda, position correction), update, wall damping, vorticity confinement,
XSPH); the timed region launches one hipGraph per step.

Printed: one JSON line with the throughput (particle-substeps/s), the roofline of the dominant
kernel (algorithmic bytes per launch / mean launch time from HIP events on the solver's stream,
against the 8 TB/s HBM peak), the maximum and mean density-constraint error after the timed
steps, and the CPU oracle timed on the host's cores on a bounded sample of the same workload.

Also reported, each in its own object of the same line:
  learned   -- learned warm start vs plain solver at equal error.  The headline parameter set
               drives the 1M column into a degenerate state (max density error ~88 after 100
               steps, velocities in the hundreds to thousands), where density error says
               nothing, so the comparison runs on the same 1M scene with the reference
               application's own solver parameters (PBFConfig defaults) at a 2 ms substep: plain
               with 1-4 iterations and learned with J = 1, 2 (networks from
               akuaengine_amd/networks, trained by akuaengine_amd/train_warm_start.py), 300
               steps each, density error sampled every 25 steps.
  learned_8m -- the same comparison on the 8M two-column scene (plain with 3 and 4 iterations,
               learned with J = 1 and the 1M-trained network), 150 steps each.
  dam_break_8m, batched_256 -- throughput of the 8M two-column scene and of 256 independent
               scenes in one batched solver.

Usage: python bench.py [--steps K] [--warmup W] [--gpus 1] [--cpu-seconds S] [--no-cpu-baseline]
                       [--no-learned] [--no-extra]
                       [--tuning block,level,hashBits,layoutBits,interval[,balanceTile[,slabBatch[,fuseSweep[,laneGroup[,workQueue]]]]]]
"""
from __future__ import annotations

import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "particle-substeps/sec at 1M particles, learned vs plain, max density err ≤1%"
HBM_PEAK_GBPS = 8000.0

# Algorithmic bytes per particle of each kernel (FP32 structure of arrays, every array element a
# pass must stream counted once; neighbour positions are gathered and counted as cache-resident;
# nbar = measured mean neighbour count, the neighbour list is 4 bytes per entry).
#   density/lambda : x* 12 + count 4 + density 4 + lambda 4 + list 4 nbar
#   delta/correct  : x* 12 + lambda 4 + count 4 + x* out 12 + list 4 nbar
#   last iteration : the above + update and damping (x 12 in, x 12 + v 12 out, ids 8) 48
#   neighbours     : x* 12 + count 4 + list 4 nbar
#   vorticity      : x 12 + v 12 + count 4 + omega 12 + list 4 nbar
#   confinement    : x 12 + omega 12 + rho 4 + v 12 + count 4 + v out 12 + list 4 nbar
#   xsph           : x 12 + v 12 + rho 4 + count 4 + v out 12 + list 4 nbar
#   predict/hash 44, gather (reorder) 72, each sort kernel 16 per pass over 3 kernels, table 8
BYTES = {
    "density_lambda": lambda nb: 24 + 4 * nb,
    "delta_correct": lambda nb: 32 + 4 * nb,
    "delta_correct_update": lambda nb: 80 + 4 * nb,
    "neighbours": lambda nb: 16 + 4 * nb,
    "vorticity": lambda nb: 40 + 4 * nb,
    "confinement": lambda nb: 56 + 4 * nb,
    "xsph": lambda nb: 44 + 4 * nb,
    "predict_hash": lambda nb: 44,
    "order": lambda nb: 116,  # predict/hash and move together (launch_order, launch_tally)
    "gather": lambda nb: 72,
    "rs_hist": lambda nb: 4,
    "rs_scan": lambda nb: 0,
    "rs_scatter": lambda nb: 16,
    "rs_onesweep": lambda nb: 16,
    "fill_table": lambda nb: 8,
    "tile_queue": lambda nb: 4,
}


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def _cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _oracle_rate(O, scene, cfg, corr, dt, budget_s: float, max_steps: int, label: str):
    """Steps of the FP32 oracle from the scene's initial state until the budget is spent (at
    least one step, at most max_steps): (particle-substeps/s, steps, seconds)."""
    o = O.Oracle(scene.n, cfg, corr, 32)
    o.set_state(scene.pos, scene.vel, scene.mass)
    steps, t0 = 0, time.perf_counter()
    while True:
        o.step(dt, scene.box_min, scene.box_max, 1)
        steps += 1
        el = time.perf_counter() - t0
        if steps == 1 or steps % 50 == 0:
            log(f"[bench] cpu oracle {label} step {steps}: {el:.1f} s")
        if el >= budget_s or steps >= max_steps:
            break
    return scene.n * steps / el, steps, el


def cpu_baseline(scene, cfg, corr, dt, budget_s: float):
    """The FP32 CPU oracle (OpenMP over particles) on the same 1M workload from its initial
    state: steps until the time budget is spent (at least one).  Beside it: one step of the 1M
    scene on one thread, and the 27k dam break (all 200 steps on every thread, a bounded sample
    on one thread), with the host's CPU model and core count."""
    from akuaengine_amd import scenes
    from oracle import oracle as O
    threads = O.max_threads()
    rate, steps, el = _oracle_rate(O, scene, cfg, corr, dt, budget_s, 50, "1M")
    out = {"value": rate, "unit": "particle-substeps/s", "cores": threads, "kind": "port",
           "sample": f"{steps} steps of the 1M dam break from its initial state, FP32 oracle, "
                     f"{threads} OpenMP threads, {el:.1f} s",
           "host": {"cpu_model": _cpu_model(), "nproc": os.cpu_count(), "threads": threads}}
    small = scenes.dam_break_27k()
    r27, s27, e27 = _oracle_rate(O, small, cfg, corr, dt, 60.0, 200, "27k")
    out["dam_break_27k"] = {"value": r27, "steps": s27, "seconds": round(e27, 2), "threads": threads}
    O.set_threads(1)
    try:
        r1, s1, e1 = _oracle_rate(O, scene, cfg, corr, dt, 0.0, 1, "1M one thread")
        out["one_thread_1m"] = {"value": r1, "steps": s1, "seconds": round(e1, 2)}
        r1s, s1s, e1s = _oracle_rate(O, small, cfg, corr, dt, 8.0, 200, "27k one thread")
        out["one_thread_27k"] = {"value": r1s, "steps": s1s, "seconds": round(e1s, 2)}
    finally:
        O.set_threads(threads)
    return out


def time_steps(s, dt, bmin, bmax, steps: int) -> float:
    """Seconds of `steps` steps, synchronised on both sides."""
    s.synchronize()
    t0 = time.perf_counter()
    s.step_n(dt, bmin, bmax, steps)
    s.synchronize()
    return time.perf_counter() - t0


def learned_comparison(log_steps: int = 300, sample: int = 25, skip: int = 50, only: str = None,
                       scene: str = "1m", plain_iters=(4, 3, 2, 1), learned_js=(1, 2),
                       physics: str = "reference"):
    """Plain solver with 1-4 iterations and learned warm start with J = 1, 2 on the 1M scene (or
    the 8M two-column scene, scene="8m").  physics "reference": the reference application's
    parameters at a 2 ms substep; "dam_break": the dam-break workload's own parameter set at its
    8.3 ms step.  The networks are the ones trained on 1M scenes with the same physics.  only: run
    just one configuration ("plain_I<n>" or "learned_J<n>") and return its record."""
    from dataclasses import replace
    from akuaengine_amd import learned, scenes
    from akuaengine_amd.solver import PBFSolver
    from akuaengine_amd.train_warm_start import PHYSICS
    cfg, corr, dt = PHYSICS[physics]()
    sc = scenes.dam_break_8m() if scene == "8m" else scenes.dam_break_1m()
    if only:  # load just the network the configuration uses
        kind, n = only.split("_")
        learned_js = (int(n[1:]),) if kind == "learned" else ()
    stem = "reference" if physics == "reference" else "benchmark"
    nets = {}
    for J in learned_js:
        path = os.path.join(learned.NETWORK_DIR, f"dam_break_1m_{stem}_J{J}.npy")
        if os.path.exists(path):
            with open(os.path.splitext(path)[0] + ".json") as f:
                meta = json.load(f)
            nets[J] = (learned.load_network(path), meta)
        else:
            from akuaengine_amd.train_warm_start import train
            log(f"[bench] training the J={J} network (no file at {path})")
            nets[J] = train(physics, J, log=log)

    # every variant runs the default setting: the autotuner's short plain trials picked settings
    # (a layout refresh interval of 2) that made both the plain and the learned steps slower here

    def run(I, J=None):
        s = PBFSolver(sc.n, replace(cfg, solverIterations=I), corr)
        s.set_state(sc.pos, sc.vel, sc.mass)
        if J is not None:
            net, meta = nets[J]
            s.set_network(net)
            s.set_learned(True, meta["gate_ratio_p90"], 0.01, "max", J)
        errs, t, done = [], 0.0, 0
        while done < log_steps:
            el = time_steps(s, dt, sc.box_min, sc.box_max, sample)
            if done >= skip:
                t += el
            done += sample
            errs.append(s.density_error())
        ms = t / (log_steps - skip) * 1e3
        errs = [[float(a), float(b)] for a, b in errs]
        r = {"iterations": I, "ms_per_step": round(ms, 4), "value": round(sc.n / ms * 1e3, 1),
             "density_error_max_avg": round(sum(e[0] for e in errs) / len(errs), 5),
             "density_error_mean_avg": round(sum(e[1] for e in errs) / len(errs), 6),
             "density_error_final": [round(errs[-1][0], 5), round(errs[-1][1], 6)]}
        if J is not None:
            st = s.learned_stats()
            r.update({"learned_iterations": J, "fallback_steps": st["fallbacks"],
                      "gate": {"statistic": "max", "ratio": round(nets[J][1]["gate_ratio_p90"], 4),
                               "tolerance": 0.01}})
        log(f"[bench] {scene} {'learned J=%d' % J if J else 'plain I=%d' % I}: {ms:.3f} ms/step, "
            f"error max {r['density_error_max_avg']:.4f} mean {r['density_error_mean_avg']:.5f}")
        return r

    if only:
        kind, n = only.split("_")
        return {only: run(int(n[1:])) if kind == "plain" else run(4, int(n[1:]))}
    plain = {f"plain_I{I}": run(I) for I in plain_iters}
    learned_runs = {f"learned_J{J}": run(4, J) for J in learned_js}
    out = {"workload": f"dam_break_{scene}_{'reference_substep' if physics == 'reference' else 'benchmark_parameters'}",
           "particles": sc.n, "dt": dt,
           "parameters": ("PBFConfig/LambdaCorrParams defaults (PBFConfig.h:10-29)" if physics == "reference"
                          else "the dam-break workload's set: rest density 6378, k 0.1, n 4, "
                               "delta_q 0.2 h, dt 0.0083"),
           "steps": log_steps, "timed_steps": log_steps - skip, "error_samples_every": sample,
           **plain, **learned_runs}
    # equal error: the cheapest plain solver whose time-averaged errors are both no larger
    for name, r in learned_runs.items():
        ok = [p for p in plain.values() if p["density_error_max_avg"] <= r["density_error_max_avg"]
              and p["density_error_mean_avg"] <= r["density_error_mean_avg"]]
        best = min(ok, key=lambda p: p["ms_per_step"]) if ok else None
        r["speedup_vs_plain_I4"] = round(plain["plain_I4"]["ms_per_step"] / r["ms_per_step"], 4)
        r["speedup_vs_plain_at_equal_error"] = (
            round(best["ms_per_step"] / r["ms_per_step"], 4) if best else None)
        r["plain_at_equal_error"] = f"plain_I{best['iterations']}" if best else None
    out["max_density_error_le_1pct"] = {
        k: v["density_error_max_avg"] <= 0.01 for k, v in {**plain, **learned_runs}.items()}
    return out


def full_run(tuning, total: int = 500, edges=(0, 10, 100, 200, 300, 400, 500)):
    """The headline workload's whole run: the 1M dam break from its initial state for 500 steps
    (the run the workload defines) at the given setting, timed per window of steps with the
    device synchronised at the window edges; the mean over steps 10-500 and the density error
    at the end."""
    from akuaengine_amd import scenes
    from akuaengine_amd.config import DAM_BREAK_DT, dam_break_params
    from akuaengine_amd.solver import PBFSolver
    cfg, corr = dam_break_params(4)
    dt = DAM_BREAK_DT
    sc = scenes.dam_break_1m()
    s = PBFSolver(sc.n, cfg, corr)
    s.set_state(sc.pos, sc.vel, sc.mass)
    s.set_tuning(**tuning)
    windows, t_after10 = [], 0.0
    for a, b in zip(edges[:-1], edges[1:]):
        el = time_steps(s, dt, sc.box_min, sc.box_max, b - a)
        windows.append({"steps": [a, b], "ms_per_step": round(el / (b - a) * 1e3, 4)})
        if a >= 10:
            t_after10 += el
    emax, emean = s.density_error()
    n_after = edges[-1] - 10
    out = {"particles": sc.n, "steps": total, "windows": windows,
           "ms_per_step_10_500": round(t_after10 / n_after * 1e3, 4),
           "value_10_500": round(sc.n * n_after / t_after10, 1), "unit": "particle-substeps/s",
           "density_error_at_500": {"max": round(emax, 5), "mean": round(emean, 6)}}
    log(f"[bench] 500-step run: {out['ms_per_step_10_500']:.3f} ms/step over steps 10-500, windows "
        + ", ".join(f"{w['steps'][0]}-{w['steps'][1]}: {w['ms_per_step']:.3f}" for w in windows))
    del s
    return out


def extra_workloads(steps: int = 20, warmup: int = 3):
    """Throughput of the 27k dam break (the reference's CPU-runnable scene, all 200 steps), of the
    8M two-column scene and of the 256-scene batch (plain, 4 iterations), the cost of the wall
    samples and of headless rendering."""
    import numpy as np
    from akuaengine_amd import scenes
    from akuaengine_amd.config import DAM_BREAK_DT, dam_break_params
    from akuaengine_amd.solver import BatchSolver, PBFSolver
    cfg, corr = dam_break_params(4)
    dt = DAM_BREAK_DT
    out = {}
    # the 27k dam break from its initial state, all 200 steps, at the autotuner's setting (the
    # tuner's trials start from the initial state and restore it); the CPU baseline times the same
    sc = scenes.dam_break_27k()
    s = PBFSolver(sc.n, cfg, corr)
    s.set_state(sc.pos, sc.vel, sc.mass)
    tuning = s.autotune(dt, sc.box_min, sc.box_max, trialSteps=5)
    el = time_steps(s, dt, sc.box_min, sc.box_max, 200)
    emax, emean = s.density_error()
    out["dam_break_27k"] = {"particles": sc.n, "steps": 200, "ms_per_step": round(el / 200 * 1e3, 4),
                            "value": round(sc.n * 200 / el, 1), "unit": "particle-substeps/s",
                            "tuning": tuning, "density_error_after_200": [float(emax), float(emean)]}
    log(f"[bench] 27k: {el / 200 * 1e3:.3f} ms/step")
    del s
    sc = scenes.dam_break_8m()
    s = PBFSolver(sc.n, cfg, corr)
    s.set_state(sc.pos, sc.vel, sc.mass)
    s.step_n(dt, sc.box_min, sc.box_max, warmup)
    tuning = s.autotune(dt, sc.box_min, sc.box_max, trialSteps=3)
    s.step_n(dt, sc.box_min, sc.box_max, 1)
    el = time_steps(s, dt, sc.box_min, sc.box_max, steps)
    out["dam_break_8m"] = {"particles": sc.n, "steps": steps, "ms_per_step": round(el / steps * 1e3, 4),
                           "value": round(sc.n * steps / el, 1), "unit": "particle-substeps/s",
                           "tuning": tuning}
    log(f"[bench] 8M: {el / steps * 1e3:.3f} ms/step")
    del s
    scs = scenes.batched_scenes(256, seed=3)
    counts = [x.n for x in scs]
    b = BatchSolver(counts, cfg, corr)
    b.set_state(np.concatenate([x.pos for x in scs]), np.concatenate([x.vel for x in scs]))
    for i, x in enumerate(scs):
        b.set_box(i, x.box_min, x.box_max)
    b.step_batch(dt, warmup)
    b.autotune(dt, trialSteps=3)  # on a developed state, as the single scenes
    b.step_batch(dt, 1)
    b.synchronize()
    t0 = time.perf_counter()
    b.step_batch(dt, steps)
    b.synchronize()
    el = time.perf_counter() - t0
    total = int(sum(counts))
    out["batched_256"] = {"scenes": 256, "particles": total, "steps": steps,
                          "ms_per_step": round(el / steps * 1e3, 4), "value": round(total * steps / el, 1),
                          "unit": "particle-substeps/s", "tuning": b.get_tuning()}
    log(f"[bench] batched 256 scenes ({total} particles): {el / steps * 1e3:.3f} ms/step")
    del b
    out["boundary_1m"] = boundary_cost(steps, warmup)
    out["render_1280x720"] = render_cost()
    return out


def render_cost(images: int = 10):
    """Wall time of akua_render per 1280x720 image, the copy of the 2.8 MB image to the host
    included: the application scene from the default camera (27k particles, 50-pixel sprites), and
    the 1M dam break from (5, 4, 16), where its whole 10 x 6 x 5 box is in view."""
    from akuaengine_amd import scenes
    from akuaengine_amd.config import dam_break_params
    from akuaengine_amd.solver import PBFSolver, default_camera
    cfg, corr = dam_break_params(4)
    res = {"width": 1280, "height": 720, "point_size": 50.0, "images": images}
    for key, sc, eye in (("app_dam_break", scenes.app_dam_break(), None),
                         ("dam_break_1m", scenes.dam_break_1m(), (5.0, 4.0, 16.0))):
        s = PBFSolver(sc.n, cfg, corr)
        s.set_state(sc.pos, sc.vel, sc.mass)
        cam = default_camera()
        if eye is not None:
            cam.position[:] = list(eye)
        s.render(cam, 1280, 720)
        t0 = time.perf_counter()
        for _ in range(images):
            s.render(cam, 1280, 720)
        el = time.perf_counter() - t0
        res[f"ms_per_image_{key}"] = round(el / images * 1e3, 3)
        del s
    log(f"[bench] render 1280x720: {res['ms_per_image_app_dam_break']:.2f} ms (27k), "
        f"{res['ms_per_image_dam_break_1m']:.2f} ms (1M)")
    return res


def boundary_cost(steps: int, warmup: int):
    """The 1M dam break with and without two layers of wall samples (same tuning): the cost of
    the boundary terms in the density/lambda and position-delta passes."""
    from akuaengine_amd import scenes
    from akuaengine_amd.config import DAM_BREAK_DT, dam_break_params
    from akuaengine_amd.solver import PBFSolver
    cfg, corr = dam_break_params(4)
    dt = DAM_BREAK_DT
    sc = scenes.dam_break_1m()
    res = {"particles": sc.n, "steps": steps, "layers": 2}
    for layers in (0, 2):
        s = PBFSolver(sc.n, cfg, corr)
        s.set_state(sc.pos, sc.vel, sc.mass)
        s.set_boundary(layers)
        s.step_n(dt, sc.box_min, sc.box_max, warmup)
        el = time_steps(s, dt, sc.box_min, sc.box_max, steps)
        key = "boundary" if layers else "plain"
        res[f"ms_per_step_{key}"] = round(el / steps * 1e3, 4)
        if layers:
            res["samples"] = int(len(s.debug_boundary()[1]))
        del s
    res["overhead"] = round(res["ms_per_step_boundary"] / res["ms_per_step_plain"] - 1.0, 4)
    log(f"[bench] 1M with wall samples: {res['ms_per_step_boundary']:.3f} ms/step "
        f"(plain {res['ms_per_step_plain']:.3f})")
    return res


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--timing-steps", type=int, default=10,
                    help="steps with per-kernel HIP events after the timed region")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-learned", action="store_true")
    ap.add_argument("--no-extra", action="store_true")
    ap.add_argument("--no-full-run", action="store_true",
                    help="skip the 500-step run of the headline workload (profiling runs: one solver "
                         "per process)")
    ap.add_argument("--tuning", default=None,
                    help="block,level,hashBits,layoutBits,interval: apply this setting instead of "
                         "autotuning (every setting gives identical results; for profiling runs, "
                         "whose own timings would steer the tuner)")
    ap.add_argument("--learned-run", default=None,
                    help="run only this configuration of the learned comparison (plain_I1..4, "
                         "learned_J1, learned_J2), print its record and exit (for profiling)")
    ap.add_argument("--learned-physics", default="reference", choices=("reference", "dam_break"),
                    help="parameter set of --learned-run")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: --gpus {args.gpus} is not supported (the solver runs "
              f"on one device; it has no multi-GPU decomposition).", file=sys.stderr)
        return 2

    if args.learned_run:
        print(json.dumps(learned_comparison(only=args.learned_run, physics=args.learned_physics)))
        return 0

    from akuaengine_amd import _lib, scenes
    from akuaengine_amd.config import DAM_BREAK_DT, dam_break_params
    from akuaengine_amd.solver import PBFSolver

    cfg, corr = dam_break_params(4)
    dt = DAM_BREAK_DT
    sc = scenes.dam_break_1m()
    log(f"[bench] workload dam_break_1m N={sc.n}")
    s = PBFSolver(sc.n, cfg, corr)
    s.set_state(sc.pos, sc.vel, sc.mass)
    # tune on a developed state (the initial lattice is unrepresentatively regular), then warm up
    s.step_n(dt, sc.box_min, sc.box_max, args.warmup)
    if args.tuning:
        v = [int(x) for x in args.tuning.split(",")]
        b_, l_, h_, d_, i_ = v[:5]
        s.set_tuning(block=b_, layoutLevel=l_, hashDigitBits=h_, layoutDigitBits=d_,
                     layoutInterval=i_, balanceTile=v[5] if len(v) > 5 else 0,
                     slabBatch=v[6] if len(v) > 6 else 0, fuseSweep=v[7] if len(v) > 7 else 0,
                     laneGroup=v[8] if len(v) > 8 else 0, workQueue=v[9] if len(v) > 9 else 0)
        tuning = s.get_tuning()
    else:
        # 10 timed steps per trial (twice): the best settings differ by 1-3% here
        tuning = s.autotune(dt, sc.box_min, sc.box_max, trialSteps=10)
    log(f"[bench] tuning {tuning}")

    s.step_n(dt, sc.box_min, sc.box_max, args.warmup)
    s.synchronize()
    log(f"[bench] warm-up {args.warmup} steps done; timing {args.steps} steps")
    t0 = time.perf_counter()
    s.step_n(dt, sc.box_min, sc.box_max, args.steps)
    s.synchronize()
    elapsed = time.perf_counter() - t0
    nbar = s.mean_neighbours()
    value = sc.n * args.steps / elapsed
    log(f"[bench] {elapsed * 1e3 / args.steps:.3f} ms/step, {value:.4e} particle-substeps/s, nbar {nbar:.2f}")

    # per-kernel device time: HIP events around every launch on the solver's stream
    s.set_timing(True)
    s.reset_timing()
    s.step_n(dt, sc.box_min, sc.box_max, args.timing_steps)
    times = s.get_timing()
    s.set_timing(False)
    nbar_t = s.mean_neighbours()
    steps_t = args.timing_steps
    kernels = {}
    for name, (ms, launches) in times.items():
        per_launch = ms / launches
        b = BYTES.get(name, lambda nb: 0)(nbar_t) * sc.n
        kernels[name] = {"ms_per_launch": round(per_launch, 5), "launches_per_step": launches // steps_t,
                         "ms_per_step": round(ms / steps_t, 5),
                         "achieved_gbps": round(b / (per_launch * 1e-3) / 1e9, 1) if b else None}
    dominant = max(kernels, key=lambda k: kernels[k]["ms_per_step"])

    def roof(name):
        bpp = BYTES[name](nbar_t)
        per_launch_s = kernels[name]["ms_per_launch"] * 1e-3
        achieved = bpp * sc.n / per_launch_s / 1e9
        return {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBPS, 4), "traffic": None, "kernel": name,
                "bytes_per_particle": round(bpp, 2), "particles_per_launch": sc.n}

    roofline = roof(dominant)
    roof_dl = roof("density_lambda")
    step_bytes = sum(BYTES.get(k, lambda nb: 0)(nbar_t) * v["launches_per_step"] for k, v in kernels.items())
    ms_step = elapsed * 1e3 / args.steps
    roof_step = {"bytes_per_particle_step": round(step_bytes, 1),
                 "achieved": round(step_bytes * sc.n / (ms_step * 1e-3) / 1e9, 1),
                 "frac": round(step_bytes * sc.n / (ms_step * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4)}
    traffic_file = os.path.join(ROOT, "profiles", "traffic.json")
    if os.path.exists(traffic_file):
        with open(traffic_file) as f:
            tr = json.load(f)
        for r in (roofline, roof_dl):
            t = tr.get(r["kernel"])
            if t:
                r["traffic"] = t["bytes_per_launch"]

    gbps = ctypes.c_double(0.0)
    _lib.check(_lib.load().akua_stream_copy_bandwidth(1 << 30, 20, ctypes.byref(gbps)))
    emax, emean = s.density_error()
    log(f"[bench] density error after the timed steps: max {emax:.4f} mean {emean:.5f}")

    del s
    run500 = None if args.no_full_run else full_run(tuning)
    learned_out = None if args.no_learned else learned_comparison()
    # the learned workload at its own stated parameters (the dam-break set, dt 0.0083), where the
    # column degenerates (see learned_config4["note"]): measured and reported as such
    learned_c4 = None
    if not args.no_learned:
        learned_c4 = learned_comparison(physics="dam_break", plain_iters=(4, 3, 2, 1, 8),
                                        learned_js=(1,))
        learned_c4["degenerate"] = True
        learned_c4["note"] = ("at these parameters the plain solver degenerates: its max density error "
                              "reaches the tens (4 iterations) to the thousands (1 or 8 iterations), "
                              "with clumps at the 128-neighbour cap; more iterations make it worse, not "
                              "better, so no plain iteration count may reach the learned step's error")
    # the 8M scene of the learned workload: plain 4 and 3 iterations against the J = 1 network
    learned_8m = None if args.no_learned or args.no_extra else learned_comparison(
        log_steps=150, sample=25, skip=25, scene="8m", plain_iters=(4, 3), learned_js=(1,))
    extra = {} if args.no_extra else extra_workloads()

    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(sc, cfg, corr, dt, args.cpu_seconds)

    out = {
        "metric": METRIC, "value": round(value, 1), "unit": "particle-substeps/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms_step, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp32",
        "data": "synthetic",
        "config": {"workload": "dam_break_1m_plain", "particles": sc.n, "solver": "plain",
                   "solverIterations": cfg.solverIterations, "dt": dt, "restDensity": cfg.restDensity,
                   "corr_k": corr.k, "corr_n": corr.n, "corr_delta_q": corr.delta_q,
                   "box_max": list(sc.box_max), "parallelism": "single-gpu", "tuning": tuning},
        "roofline": roofline,
        "roofline_density_lambda": roof_dl,
        "roofline_step": roof_step,
        "stream_copy_gbps": round(gbps.value, 1),
        "mean_neighbours": round(nbar_t, 3),
        "density_error": {"max": round(emax, 5), "mean": round(emean, 6),
                          "definition": "max/mean over particles of max(0, rho/rho0 - 1), exact SPH "
                                        "density at the positions after the timed steps"},
        "kernels": kernels,
        "full_run_500": run500,
        "learned": learned_out,
        "learned_config4": learned_c4,
        "learned_8m": learned_8m,
        **extra,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out))
    return 0


if __name__ == "__main__":
    sys.exit(main())
