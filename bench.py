"""Benchmark: simulation steps per second of the ADMM contact step on one MI355X,
run to ADMM residual <= 1e-4 (capped at admm_max_iter), with the roofline of
the global solve's measured kernel (the direct solve's dense-top product, or
the PCG SpMV) and the FP64 CPU oracle timed on the host beside it.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload cloth256|tetbox|cloth32]
    python bench.py --copy-calibration     # plain device copy of known size (for rocprofv3 --pmc scaling)

Prints one JSON line.  A "step" is one simulation time step of the whole scene
(detection, local/contact/global ADMM iterations) on synthetic geometry with
positions resident in HBM.
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "sim steps/s at ADMM residual \u22641e-4, plain vs learned warm-start; % HBM peak"
HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
COPY_BYTES = 1 << 28   # calibration copy: 256 MiB read + 256 MiB written per launch
COPY_LAUNCHES = 20


def spmv_bytes(n: int, nnz_off: int) -> int:
    """Algorithmic bytes of one launch of the fused PCG direction + SpMV kernel
    (k_cg_dir_spmv: p' = z + beta p, q = A p', 3 interleaved FP32 columns):
    off-diagonal values + column ids (8 B each), row pointers (4(n+1)), diagonal
    (4n), z and p read once (24n), p' and q written (24n); the per-block
    partial sums are negligible."""
    return 8 * nnz_off + 4 * (n + 1) + 4 * n + 24 * n + 24 * n


def top_bytes(top_cols: int, top_sq: int) -> int:
    """Algorithmic bytes of one launch of the direct solve's dense-top product
    (k_chol_top): S^-1 read once (4 sum m^2), and per top entry its assembled
    right-hand side (12, written by k_chol_top_f), its place (4) and the
    correction (12)."""
    return 4 * top_sq + 28 * top_cols


def measured_traffic(workload: str, kernel: str) -> tuple[int | None, str | None]:
    """HBM bytes per launch of the roofline kernel from the committed PMC
    summary (FETCH_SIZE + WRITE_SIZE per dispatch, scaled by the copy-kernel
    factor), if one exists for this workload."""
    path = os.path.join(ROOT, "profiles", f"pmc_{kernel}_{workload}.md")
    if not os.path.exists(path):
        return None, None
    m = re.search(r"traffic_bytes_per_launch:\s*([0-9]+)", open(path).read())
    return (int(m.group(1)), os.path.relpath(path, ROOT)) if m else (None, None)


def profile_kernel_avg_ms(workload: str, kernel: str) -> tuple[float | None, str | None]:
    """Average duration (ms) of `kernel` (all template variants, weighted by
    calls) in the committed rocprofv3 kernel-trace summary of this workload."""
    path = os.path.join(ROOT, "profiles", f"kernel_trace_{workload}.md")
    if not os.path.exists(path):
        return None, None
    calls = total = 0.0
    for line in open(path):
        cells = [c.strip() for c in line.strip().strip("|").split("|")]
        if len(cells) >= 3 and re.match(re.escape(kernel) + r"(<|$)", cells[0]):
            calls += float(cells[1])
            total += float(cells[2])
    return (total / calls, os.path.relpath(path, ROOT)) if calls else (None, None)


def measured_step_traffic(workload: str) -> tuple[int | None, str | None]:
    """HBM bytes of one whole step (every kernel), from the committed PMC
    summary: FETCH_SIZE + WRITE_SIZE summed over all dispatches of two runs
    that differ only in their number of timed steps, the difference divided
    by the step difference, scaled by the copy-kernel factors."""
    path = os.path.join(ROOT, "profiles", f"pmc_step_{workload}.md")
    if not os.path.exists(path):
        return None, None
    m = re.search(r"traffic_bytes_per_step:\s*([0-9]+)", open(path).read())
    return (int(m.group(1)), os.path.relpath(path, ROOT)) if m else (None, None)


def copy_calibration() -> int:
    """A plain device-to-device copy of COPY_BYTES, launched COPY_LAUNCHES
    times: under rocprofv3 --pmc its FETCH_SIZE / WRITE_SIZE per dispatch give
    the counters' scale against a known byte count."""
    import torch

    a = torch.empty(COPY_BYTES // 4, dtype=torch.float32, device="cuda:0").uniform_()
    b = torch.empty_like(a)
    for _ in range(COPY_LAUNCHES):
        b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes_read": COPY_BYTES, "copy_bytes_written": COPY_BYTES, "launches": COPY_LAUNCHES}))
    return 0


def _cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _oracle_run(prec: int, scene, cfg, state, tracks, frame: int, seconds: float) -> dict:
    """Steps the oracle (prec 64: FP64; prec 32: the FP32 twin) from `state`
    for about `seconds` (at least one step); steps/s, ms per step and the
    phase split (detection, local, contact, global)."""
    from oracle.pyoracle import Oracle

    o = Oracle(scene.mesh(), cfg, prec=prec)
    for first, count, pos, quat in tracks:
        o.add_rigid_track(first, count, pos[frame:], quat[frame:])
    x, v, ue, uc = state
    o.set_state(x, v)
    o.set_duals(ue, uc)
    t0 = time.perf_counter()
    steps, iters = 0, 0
    ph = np.zeros(4)
    while True:
        st = o.step()
        steps += 1
        iters += st["iterations"]
        ph += [st["dcd_ms"], st["local_ms"], st["contact_ms"], st["global_ms"]]
        if time.perf_counter() - t0 > seconds:
            break
    dt = time.perf_counter() - t0
    return {"value": steps / dt, "ms_per_step": 1e3 * dt / steps, "steps": steps, "admm_iterations": iters, "seconds": dt,
            "phase_ms": dict(zip(("detection", "local", "contact", "global"), [round(float(t), 2) for t in ph / steps]))}


def cpu_baseline(workload: str, scene, cfg, state, tracks, frame: int, seconds: float) -> dict:
    """The CPU restatement of the reference's CPU backend (prefactored sparse
    LLT, OpenMP local step and broad phase) on the host cores, started from
    the GPU's state at the beginning of its timed region (obstacle tracks
    resumed at the same frame): the FP64 oracle for about `seconds`, then its
    FP32 twin (the reference's own precision) for about half that."""
    cores = os.cpu_count() or 1
    threads = int(os.environ.get("OMP_NUM_THREADS", cores))
    f64 = _oracle_run(64, scene, cfg, state, tracks, frame, seconds)
    f32 = _oracle_run(32, scene, cfg, state, tracks, frame, seconds / 2)
    return {"value": f64["value"], "unit": "steps/s", "cores": threads, "kind": "port",
            "sample": f"{workload}: {f64['steps']} FP64 oracle steps ({f64['admm_iterations']} ADMM iterations) from the GPU's "
                      f"state at the start of its timed region, {f64['seconds']:.1f} s",
            "cpu_model": _cpu_model(), "host_cpus": cores, "ms_per_step": f64["ms_per_step"], "phase_ms": f64["phase_ms"],
            "fp32_twin": {k: f32[k] for k in ("value", "ms_per_step", "steps", "phase_ms")}}


MLP_FLOPS_FWD = 2 * (10 * 128 + 2 * 128 * 128 + 128 * 2)  # per sample, algorithmic (unpadded)
BF16_PEAK_TFLOPS = 2500.0


def learned_leg(pa, args, scene, cfg, tracks, plain_stats, plain_value) -> dict:
    """The same run with the committed warm-start network (mode 1, default
    judge): a fresh backend, the same warm-up, the same timed steps.  Also the
    network's own MFMA throughput (forward; forward + backward + Adam) on a
    batch of 8192 contact rows."""
    from parallel_admm_amd import warm_start as ws

    model = ws.Model.load()
    b = pa.ADMMBackendHIP.from_scene(scene, cfg)
    for first, count, pos, quat in tracks:
        b.add_rigid_track(first, count, pos, quat, frames_per_step=1)
    b.set_sync_to_host(False)
    for _ in range(args.warmup):
        b.step()
    ws.apply(b, model, 1)
    st = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        st.append(b.step())
    wall = time.perf_counter() - t0
    sl, sp = ws.summary(st, wall), ws.summary(plain_stats, args.steps / plain_value)
    net = pa.MLP(0)
    net.set_params(model.params)
    rows = 8192
    fwd_ms, train_ms = net.time_ms(0, rows, 200), net.time_ms(1, rows, 200)
    fwd_tf = MLP_FLOPS_FWD * rows / (fwd_ms * 1e-3) / 1e12
    train_tf = 3 * MLP_FLOPS_FWD * rows / (train_ms * 1e-3) / 1e12
    print(f"[bench] learned warm start: {sl['steps_per_s']:.2f} steps/s, ADMM iters {sl['admm_iters_mean']:.1f} "
          f"(+{sl['admm_iters_incl_wasted'] - sl['admm_iters_mean']:.1f} abandoned), converged {sl['converged']}, "
          f"fallbacks {sl['fallbacks']}; MLP forward {fwd_ms * 1e3:.1f} us / train step {train_ms * 1e3:.1f} us per 8192 rows",
          file=sys.stderr, flush=True)
    return {
        "value": sl["steps_per_s"], "unit": "steps/s", "speedup_vs_plain": sl["steps_per_s"] / plain_value,
        "admm_iters_mean": sl["admm_iters_mean"], "admm_iters_incl_abandoned": sl["admm_iters_incl_wasted"],
        "plain_admm_iters_mean": sp["admm_iters_mean"],
        "iteration_ratio_plain_over_learned": sp["admm_iters_mean"] / max(sl["admm_iters_incl_wasted"], 1e-9),
        "converged_steps": sl["converged"], "plain_converged_steps": sp["converged"],
        "final_residual_mean": sl["final_residual_mean"], "plain_final_residual_mean": sp["final_residual_mean"],
        "fallback_steps": sl["fallbacks"], "seeded_detections": sl["seeded"],
        "model": {k: model.meta.get(k) for k in ("samples", "epochs", "batch", "lr", "seed", "data_seed", "source")},
        "mlp_roofline": {"bound": "mfma", "unit": "TFLOP/s", "peak": BF16_PEAK_TFLOPS, "rows": rows,
                         "forward_ms": fwd_ms, "forward_achieved": fwd_tf, "forward_frac": fwd_tf / BF16_PEAK_TFLOPS,
                         "train_step_ms": train_ms, "train_achieved": train_tf, "train_frac": train_tf / BF16_PEAK_TFLOPS},
    }


def uncapped_leg(pa, workload: str, scene, cfg, tracks, state, frame: int, steps: int, tol: float, cap: int = 1000) -> dict:
    """The timed steps again from the same start state (obstacle tracks
    resumed at the same frame) with the iteration cap lifted to `cap`: ADMM
    iterations each step needs to reach the residual tolerance, and the
    steps/s at that tolerance."""
    c = config_for_copy(cfg)
    c.admm_max_iter = cap
    c.residual_tol = tol
    b = pa.ADMMBackendHIP.from_scene(scene, c)
    for first, count, pos, quat in tracks:
        b.add_rigid_track(first, count, pos[frame:], quat[frame:], frames_per_step=1)
    b.set_sync_to_host(False)
    x, v, ue, uc = state
    b.set_state(x, v)
    b.set_duals(ue, uc)
    stats = []
    t0 = time.perf_counter()
    for _ in range(steps):
        stats.append(b.step())
    wall = time.perf_counter() - t0
    it = np.array([s["iterations"] for s in stats])
    out = {"steps_per_s": steps / wall, "ms_per_step": 1e3 * wall / steps, "admm_max_iter": cap,
           "admm_iters_mean": float(it.mean()), "admm_iters_p50": float(np.median(it)), "admm_iters_max": int(it.max()),
           "converged_steps": int(sum(s["converged"] for s in stats)), "steps": steps,
           "pcg_iters_per_step": float(np.mean([s["global_iters"] for s in stats]))}
    print(f"[bench] {workload} uncapped (cap {cap}): {out['steps_per_s']:.2f} steps/s, ADMM iterations to {tol:g} mean "
          f"{out['admm_iters_mean']:.1f} (max {out['admm_iters_max']}), converged {out['converged_steps']}/{steps}",
          file=sys.stderr, flush=True)
    return out


def config_for_copy(cfg):
    from parallel_admm_amd import AdmmConfig

    return AdmmConfig(**vars(cfg))


def dense_leg(pa, steps: int, warmup: int, tol: float) -> dict:
    """cloth256 at the config's contact density: the workload's scene with a
    24-column flap of the cloth folded back over it (configs.folded_flap_state,
    101,804 contacts), the same solver settings and obstacle track.  Every
    step starts from that state at rest with zero duals (the contact response
    lifts the flap to the contact distance within a step, after which the
    resting layers hover at the detection threshold), so each timed step
    detects the full contact set: `warmup` untimed steps, then `steps` timed
    one by one, and the phase split of one more."""
    from parallel_admm_amd.configs import config_for, folded_flap_state, workload_tracks

    scene = pa.Scene.generate(3)
    cfg = config_for("cloth256")
    cfg.residual_tol = tol
    cfg.residual_interval = 1
    b = pa.ADMMBackendHIP.from_scene(scene, cfg)
    for first, count, pos, quat in workload_tracks("cloth256", scene, warmup + steps + 8):
        b.add_rigid_track(first, count, pos, quat, frames_per_step=1)
    b.set_sync_to_host(False)
    x0 = folded_flap_state(scene)
    v0 = np.zeros_like(x0)
    ue, uc = b.get_duals()
    ue0, uc0 = np.zeros_like(ue), np.zeros_like(uc)

    def restart():
        b.set_state(x0, v0)
        b.set_duals(ue0, uc0)

    for _ in range(warmup):
        restart()
        b.step()
    stats, wall = [], 0.0
    for _ in range(steps):
        restart()
        t0 = time.perf_counter()
        stats.append(b.step())
        wall += time.perf_counter() - t0
    restart()
    b.set_profiling(2)
    st = b.step()
    ph = b.phase_times()
    b.set_profiling(0)
    nc = [s["n_contacts_max"] for s in stats]
    out = {"steps_per_s": steps / wall, "ms_per_step": 1e3 * wall / steps, "steps": steps, "warmup": warmup,
           "step_peak_contacts_min": int(min(nc)), "step_peak_contacts_max": int(max(nc)),
           "last_detection_contacts_mean": float(np.mean([s["n_contacts"] for s in stats])),
           "admm_iters_mean": float(np.mean([s["iterations"] for s in stats])),
           "converged_steps": int(sum(s["converged"] for s in stats)),
           "pcg_iters_per_step": float(np.mean([s["global_iters"] for s in stats])),
           "phase_ms": dict(zip(("detection", "local", "contact", "rhs", "global", "other"), (round(float(v), 3) for v in ph))),
           "phase_step_iterations": st["iterations"]}
    print(f"[bench] cloth256 folded flap: {out['steps_per_s']:.2f} steps/s, {out['step_peak_contacts_min']}.."
          f"{out['step_peak_contacts_max']} contacts at the step's densest detection, "
          f"ADMM iters {out['admm_iters_mean']:.1f}; phases " + ", ".join(f"{v:.2f}" for v in ph), file=sys.stderr, flush=True)
    return out


def full_run_leg(pa, workload: str, scene, frames: int) -> dict:
    """The workload's whole run from its initial state (cloth256: 300 frames,
    fall, draping and folding over the sphere and the rotating cylinder) on a
    fresh backend, with the same settings as the timed steps: the rate over
    all frames, the contact peak and the ADMM iterations early and late."""
    from parallel_admm_amd.configs import config_for, workload_tracks

    cfg = config_for(workload)
    cfg.residual_tol = 1e-4
    b = pa.ADMMBackendHIP.from_scene(scene, cfg)
    b.set_sync_to_host(False)
    for first, count, pos, quat in workload_tracks(workload, scene, frames + 8):
        b.add_rigid_track(first, count, pos, quat)
    stats, wall_f = [], []
    t0 = time.perf_counter()
    for _ in range(frames):
        ts = time.perf_counter()
        stats.append(b.step())
        wall_f.append(time.perf_counter() - ts)
    wall = time.perf_counter() - t0
    x, _ = b.get_state()
    it = np.array([s["iterations"] for s in stats], float)
    nc = np.array([s["n_contacts_max"] for s in stats], float)
    q = max(1, frames // 10)
    # the window of `win` consecutive frames with the most contacts
    win = min(20, frames)
    csum = np.convolve(nc, np.ones(win), "valid")
    w0 = int(np.argmax(csum))
    wsec = float(np.sum(wall_f[w0:w0 + win]))
    out = {"frames": frames, "steps_per_s": frames / wall, "seconds": wall,
           "contacts_max": int(nc.max()), "contacts_max_frame": int(np.argmax(nc)), "contacts_last": int(stats[-1]["n_contacts"]),
           "admm_iters_first_tenth": float(it[:q].mean()), "admm_iters_last_tenth": float(it[-q:].mean()),
           "converged_steps": int(sum(s["converged"] for s in stats)), "state_finite": bool(np.isfinite(x).all()),
           "peak_window": {"first_frame": w0, "frames": win, "contacts_mean": float(nc[w0:w0 + win].mean()),
                           "steps_per_s": win / wsec, "admm_iters_mean": float(it[w0:w0 + win].mean())}}
    print(f"[bench] {workload} whole run: {frames} frames in {wall:.1f} s = {out['steps_per_s']:.1f} steps/s, contacts max "
          f"{out['contacts_max']}, ADMM iterations {out['admm_iters_first_tenth']:.1f} -> {out['admm_iters_last_tenth']:.1f}; "
          f"peak window frames {w0}..{w0 + win - 1}: {out['peak_window']['contacts_mean']:.0f} contacts, "
          f"{out['peak_window']['steps_per_s']:.1f} steps/s", file=sys.stderr, flush=True)
    return out


def batch_leg(pa, count: int, warmup: int, steps: int, solo_sample: int = 16, graphs: int = 0, precond: int | None = None) -> dict:
    """The batched workload: `count` cloths (side ~ U{16..96}, drop ~ U(0.2,
    0.6) m, sphere radius ~ U(0.1, 0.3) m, mu ~ U(0.1, 0.6); generator seed 0;
    h = 1/60, 30 ADMM iterations) merged into one scene and stepped together.
    Beside it, a sample of the same scenes stepped one at a time with the
    single-scene backend (same settings and warm-up): their per-scene step
    times give the p50/p99 and the one-at-a-time throughput."""
    from parallel_admm_amd.configs import config_for
    from parallel_admm_amd.warm_start import batch_member_scenes

    members = list(batch_member_scenes(count, seed=0))
    t0 = time.perf_counter()
    merged = pa.Scene.merge([sc for _, sc in members])
    cfg = config_for("batch")
    cfg.max_contacts = 1 << 23
    cfg.graphs = graphs
    if precond is not None:
        cfg.precond = precond
    b = pa.ADMMBackendHIP.from_scene(merged, cfg)
    mus = np.array([par["mu"] for par, _ in members])
    b.set_scene_mu(mus, merged.segments())
    b.set_sync_to_host(False)
    setup_s = time.perf_counter() - t0
    for _ in range(warmup):
        b.step()
    print(f"[bench] batch of {count}: set-up {setup_s:.1f} s, warmup {warmup} steps done", file=sys.stderr, flush=True)
    stats = []
    t1 = time.perf_counter()
    for _ in range(steps):
        stats.append(b.step())
    wall = time.perf_counter() - t1
    its, _ = b.batch_stats(count)
    b.set_profiling(2)
    b.step()
    ph = b.phase_times()
    b.set_profiling(0)
    # one-at-a-time sample: every (count // solo_sample)-th scene
    idx = list(range(0, count, max(1, count // solo_sample)))[:solo_sample] if solo_sample > 0 else []
    solo_ms = []
    for k in idx:
        par, sc = members[k]
        c = config_for("batch")
        c.mu = par["mu"]
        c.precond = cfg.precond
        sb = pa.ADMMBackendHIP.from_scene(sc, c)
        sb.set_sync_to_host(False)
        for _ in range(warmup):
            sb.step()
        ts = time.perf_counter()
        for _ in range(steps):
            sb.step()
        solo_ms.append(1000.0 * (time.perf_counter() - ts) / steps)
    solo_ms = np.array(solo_ms if solo_ms else [float("nan")])
    sizes = np.array([par["side"] for par, _ in members])
    out = {
        "scenes": count, "vertices": merged.info["n_all"], "dynamic_vertices": merged.info["n_dyn"],
        "mu_per_scene": {"min": float(mus.min()), "max": float(mus.max()), "distribution": "U(0.1, 0.6), generator seed 0"},
        "side_min": int(sizes.min()), "side_max": int(sizes.max()), "generator_seed": 0,
        "steps": steps, "warmup": warmup, "setup_s": setup_s,
        "batched_steps_per_s": steps / wall, "scene_steps_per_s": count * steps / wall, "ms_per_batched_step": 1000.0 * wall / steps,
        "per_scene_step_ms_in_batch": 1000.0 * wall / steps,
        "phase_ms": dict(zip(("detection", "local", "contact", "rhs", "global", "other"), (float(v) for v in ph))),
        "contacts_last": stats[-1]["n_contacts"],
        "pcg_iters_to_own_tol_p50": float(np.percentile(its, 50)), "pcg_iters_to_own_tol_p99": float(np.percentile(its, 99)),
        "solo_sample": len(idx), "solo_step_ms_p50": float(np.percentile(solo_ms, 50)), "solo_step_ms_p99": float(np.percentile(solo_ms, 99)),
        "solo_scene_steps_per_s": float(1000.0 / solo_ms.mean()),
        "batch_speedup_vs_one_at_a_time": float((count * steps / wall) / (1000.0 / solo_ms.mean())),
        "global_solve": ("direct: one supernodal Cholesky factor per scene (a forest), solved level by level for all "
                         "scenes at once" if cfg.precond == 2 else "AMG-PCG over the block-diagonal batch, stopped per scene"),
        "pcg_iteration_pairs_as_hip_graphs": bool(cfg.graphs),
    }
    print(f"[bench] batch of {count}: {out['batched_steps_per_s']:.2f} batched steps/s = {out['scene_steps_per_s']:.0f} scene-steps/s; "
          f"one at a time {out['solo_scene_steps_per_s']:.0f} scene-steps/s (step ms p50 {out['solo_step_ms_p50']:.1f}, "
          f"p99 {out['solo_step_ms_p99']:.1f}); phases {', '.join(f'{v:.1f}' for v in ph)}", file=sys.stderr, flush=True)
    return out


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="cloth256", choices=["cloth256", "tetbox", "cloth32", "batch512"],
                    help="batch512: only the batched leg (512 uneven cloths stepped together)")
    ap.add_argument("--tol", type=float, default=1e-4)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=20.0)
    ap.add_argument("--copy-calibration", action="store_true")
    ap.add_argument("--no-learned", action="store_true", help="skip the learned warm-start leg")
    ap.add_argument("--batch-scenes", type=int, default=512, help="scenes in the batched leg (0 skips it)")
    ap.add_argument("--batch-steps", type=int, default=5)
    ap.add_argument("--batch-warmup", type=int, default=20)
    ap.add_argument("--batch-solo", type=int, default=16, help="scenes of the batch also stepped one at a time")
    ap.add_argument("--full-run-frames", type=int, default=300,
                    help="cloth256: also run the workload's whole run (300 frames) on a fresh backend and report its rate (0 skips it)")
    ap.add_argument("--uncapped-cap", type=int, default=1000,
                    help="the timed steps again with the ADMM iteration cap lifted to this (0 skips it)")
    ap.add_argument("--dense-steps", type=int, default=10,
                    help="cloth256: timed steps of the folded-flap state at ~1e5 contacts (0 skips it)")
    ap.add_argument("--batch-precond", type=int, default=None, choices=[0, 1, 2],
                    help="global solve of the batched leg (default: the batch config's)")
    ap.add_argument("--batch-graphs", type=int, default=0, choices=[0, 1],
                    help="1: replay the batched PCG iteration pairs as HIP graphs (0: launch every kernel, the default)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the scene runs on one device; multi-GPU sharding is not built)", file=sys.stderr)
        return 2
    if args.copy_calibration:
        return copy_calibration()

    import parallel_admm_amd as pa
    from parallel_admm_amd.configs import SCENE_KIND, config_for, workload_tracks

    if args.workload == "batch512":
        bl = batch_leg(pa, args.batch_scenes or 512, args.batch_warmup, args.batch_steps, args.batch_solo, args.batch_graphs,
                       args.batch_precond)
        print(json.dumps({
            "metric": "scene steps/s of the batched workload (512 uneven cloths stepped together, mu per scene)",
            "value": bl["scene_steps_per_s"], "unit": "scene-steps/s", "n_gpus": 1, "steps": args.batch_steps,
            "warmup": args.batch_warmup, "ms_per_step": bl["ms_per_batched_step"], "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "fp32", "data": "synthetic", "config": {"workload": "batch512", "parallelism": "single GPU"},
            "batch": bl}), flush=True)
        return 0

    scene = pa.Scene.generate(SCENE_KIND[args.workload])
    cfg = config_for(args.workload)
    cfg.residual_tol = args.tol
    cfg.residual_interval = 1
    backend = pa.ADMMBackendHIP.from_scene(scene, cfg)
    # moving obstacles of the workload, one frame per step, long enough for the whole run
    tracks = workload_tracks(args.workload, scene, args.warmup + args.steps + 64)
    for first, count, pos, quat in tracks:
        backend.add_rigid_track(first, count, pos, quat, frames_per_step=1)
    backend.set_sync_to_host(False)
    for _ in range(args.warmup):
        backend.step()
    print(f"[bench] {args.workload}: warmup {args.warmup} steps done", file=sys.stderr, flush=True)
    state = (*backend.get_state(), *backend.get_duals())
    backend.set_profiling(1)
    backend.kernel_time(reset=True)
    stats = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        stats.append(backend.step())
    t1 = time.perf_counter()
    spmv_ms, spmv_launches = backend.kernel_time()
    backend.set_profiling(0)
    elapsed = t1 - t0
    ms_per_step = 1000.0 * elapsed / args.steps
    iters = [s["iterations"] for s in stats]
    conv = sum(s["converged"] for s in stats)
    print(f"[bench] timed {args.steps} steps in {elapsed:.3f} s; ADMM iters mean {np.mean(iters):.1f}, "
          f"converged {conv}/{args.steps}, contacts last {stats[-1]['n_contacts']}", file=sys.stderr, flush=True)

    # one extra (untimed) step with phase events, for the breakdown on stderr
    backend.set_profiling(2)
    st = backend.step()
    ph = backend.phase_times()
    backend.set_profiling(0)
    print("[bench] phase ms of one step (detection, local, contact, rhs, global, other): "
          + ", ".join(f"{v:.2f}" for v in ph) + f"; iterations {st['iterations']}, PCG {st['global_iters']}",
          file=sys.stderr, flush=True)

    # roofline of the PCG SpMV (the global solve's kernel moving the most bytes per launch)
    sizes = backend.sizes()
    n = sizes["n_dyn"]
    nnz_off = sizes["nnz_a_off"]
    direct = cfg.precond == 2
    roofline_kernel = "k_chol_top" if direct else "k_cg_dir_spmv"
    bytes_launch = top_bytes(sizes["chol_top_cols"], sizes["chol_top_sq"]) if direct else spmv_bytes(n, nnz_off)
    # Kernel duration: every SpMV launch inside the timed region is bracketed
    # by its own pair of HIP events on the backend's stream (spmv_ms, the
    # in-situ average; it includes each launch's dispatch).  Beside it: 200
    # back-to-back launches on the state the timed region left, and the
    # average of the committed rocprofv3 kernel trace of this workload.
    b2b_ms = backend.spmv_time(200)
    achieved = bytes_launch / (spmv_ms * 1e-3) / 1e9 if spmv_ms > 0 else 0.0
    traffic, traffic_src = measured_traffic(args.workload, roofline_kernel)
    prof_ms, prof_src = profile_kernel_avg_ms(args.workload, roofline_kernel)
    step_bytes, step_src = measured_step_traffic(args.workload)

    uncapped = None
    if args.uncapped_cap > 0:
        uncapped = uncapped_leg(pa, args.workload, scene, cfg, tracks, state, args.warmup, args.steps, args.tol, args.uncapped_cap)

    dense = None
    if args.dense_steps > 0 and args.workload == "cloth256":
        dense = dense_leg(pa, args.dense_steps, 2, args.tol)

    learned = None if args.no_learned else learned_leg(pa, args, scene, cfg, tracks, stats, args.steps / elapsed)

    full = None
    if args.full_run_frames > 0 and args.workload == "cloth256":
        full = full_run_leg(pa, args.workload, scene, args.full_run_frames)

    batch = None
    if args.batch_scenes > 0:
        try:
            batch = batch_leg(pa, args.batch_scenes, args.batch_warmup, args.batch_steps, args.batch_solo, args.batch_graphs,
                              args.batch_precond)
        except Exception as e:  # reported, not fatal to the headline line
            batch = {"error": f"{type(e).__name__}: {e}"}
            print(f"[bench] batched leg failed: {e}", file=sys.stderr, flush=True)

    cpu = None
    if not args.no_cpu_baseline:
        print(f"[bench] CPU oracle baseline (~{args.cpu_seconds:.0f} s) ...", file=sys.stderr, flush=True)
        cpu = cpu_baseline(args.workload, scene, cfg, state, tracks, args.warmup, args.cpu_seconds)

    out = {
        "metric": METRIC,
        "value": args.steps / elapsed,
        "unit": "steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {
            "workload": args.workload,
            "vertices": scene.info["n_all"],
            "dynamic_vertices": n,
            "constraint_rows": scene.info["m_rows"],
            "residual_tol": args.tol,
            "admm_max_iter": cfg.admm_max_iter,
            "stop": f"ADMM residual <= {args.tol:g} or {cfg.admm_max_iter} iterations (the workload's iteration count), "
                    "whichever comes first; the uncapped leg lifts the cap",
            "capped_steps": args.steps - conv,
            "warm_start": "plain (cold-start contact duals per detection)",
            "moving_obstacles": len(tracks),
            "admm_iters_mean": float(np.mean(iters)),
            "converged_steps": conv,
            "contacts_last": stats[-1]["n_contacts"],
            "contacts_per_step_max": int(max(s["n_contacts_max"] for s in stats)),
            "global_solve": ("direct: supernodal Cholesky factored once at set-up, level-scheduled FP32 triangular solves "
                             "with dense tree tops, on the FP64 residual" if direct else "AMG-PCG (FP32) on the FP64 residual"),
            "global_solves_per_step": float(np.mean([s["global_iters"] for s in stats])) if direct else None,
            "pcg_iters_per_step": None if direct else float(np.mean([s["global_iters"] for s in stats])),
            "parallelism": "single GPU",
        },
        "roofline": {
            "bound": "hbm",
            "kernel": roofline_kernel,
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": traffic,
            "traffic_source": traffic_src,
            "bytes_per_launch": bytes_launch,
            "avg_launch_ms": spmv_ms,
            "timing": "HIP events around every launch in the timed region (includes each launch's dispatch)",
            "launches": spmv_launches,
            "back_to_back_ms": b2b_ms,
            "back_to_back_frac": (bytes_launch / (b2b_ms * 1e-3) / 1e9) / HBM_PEAK_GBS if b2b_ms > 0 else None,
            "rocprof_avg_ms": prof_ms,
            "rocprof_frac": (bytes_launch / (prof_ms * 1e-3) / 1e9) / HBM_PEAK_GBS if prof_ms else None,
            "rocprof_source": prof_src,
        },
        "whole_step": None if step_bytes is None else {
            "hbm_bytes_per_step": step_bytes, "source": step_src,
            "achieved_GBs": step_bytes / (ms_per_step * 1e-3) / 1e9,
            "frac": step_bytes / (ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS,
        },
        "uncapped": uncapped,
        "dense_contacts": dense,
        "cpu_baseline": cpu,
        "learned": learned,
        "full_run": full,
        "batch": batch,
    }
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
