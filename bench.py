"""Benchmark: batched VSWRM parameter sweep, fused float32 vs plain float64.

Workload (one GPU): 4096 independent visual-flocking replicas on a 64 x 64
grid of ALP0 x BET0 in [0.1, 3] x [0.1, 3]; N = 50 agents, R = 512 rays,
radius 5, 707 x 707 periodic arena (density 1e-4), GAM 0.1, V0 1, ALP1 =
BET1 = 0.09, reference (sequential) update order, per-replica seeds
10000 + b, synthetic uniform start.  A step is one kernel launch advancing
every replica by one simulation step (captured in a HIP graph and replayed).

Prints ONE JSON line: the fused kernel's agent-steps/s (``value``), the plain
float64 kernel's rate on the same workload, the one-step error between them,
the roofline of the fused kernel and the CPU baseline (the oracle, one
process per core, a bounded sample of the same replicas).
"""
from __future__ import annotations

import argparse
import json
import multiprocessing as mp
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "agent-steps/s: batched FP32 vs plain FP64 GPU at fixed error; % VALU peak"
B_SIDE, N, R, W = 64, 50, 512, 707.0
PAD, RADIUS = 30.0, 5
VALU_PEAK_TOPS = 256 * 64 * 2.4e9 / 1e12   # MI355X lane-ops/s: 256 CU x 64 lanes x 2.4 GHz


def ops_per_agent_step(n, r):
    """Algorithmic lane-ops per agent-step: pair geometry 40 per other agent,
    17 per ray, 20 per agent (transcendentals count 1)."""
    return 40 * (n - 1) + 17 * r + 20


def make_workload(n_rep_side=B_SIDE):
    from abm_amd.vf import VFConfig
    a = np.linspace(0.1, 3.0, n_rep_side)
    cfgs, xs, ys, ths = [], [], [], []
    for i in range(n_rep_side):
        for j in range(n_rep_side):
            b = i * n_rep_side + j
            cfgs.append(VFConfig(n_agents=N, n_rays=R, width=W, height=W, window_pad=PAD,
                                 boundary="infinite", GAM=0.1, V0=1.0, ALP0=float(a[i]),
                                 ALP1=0.09, BET0=float(a[j]), BET1=0.09))
            rng = np.random.RandomState(10000 + b)
            xs.append(rng.uniform(PAD, PAD + W, N))
            ys.append(rng.uniform(PAD, PAD + W, N))
            ths.append(rng.uniform(0, 2 * np.pi, N))
    f32 = lambda v: np.concatenate(v).astype(np.float32).astype(np.float64)
    return cfgs, f32(xs), f32(ys), f32(ths)


def time_steps(sw, steps, warmup, use_graph=True, per_graph=10):
    """Average time (ms) of one step over `steps` steps, after `warmup` untimed
    steps.  With graphs, up to `per_graph` consecutive steps are captured in
    one HIP graph (the step kernels back to back, no host launch between
    them; fewer when that leaves at least five replays to take the spread
    of); each replay is bracketed by events on the launch stream and its time
    divided by its steps.  Returns (mean, median, wall-clock per step); the
    quartiles of the per-replay times are left in ``time_steps.last_iqr``."""
    import torch
    for _ in range(warmup):
        sw.step()
    torch.cuda.synchronize()
    graph = None
    reps = max(1, steps)
    per = 1
    if use_graph:
        # steps per graph: the largest divisor of `steps` up to per_graph, so
        # exactly `steps` steps are timed
        cap = max(1, min(per_graph, steps // 5 if steps >= 5 else steps))
        per = max(d for d in range(1, cap + 1) if steps % d == 0)
        reps = max(1, steps // per)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            sw.step()                       # one eager launch on the capture stream
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(per):
                sw.step()
        torch.cuda.synchronize()
    run = graph.replay if graph is not None else sw.step
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(reps)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(reps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(reps):
        starts[i].record()
        run()
        ends[i].record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    per_step = [s.elapsed_time(e) / per for s, e in zip(starts, ends)]
    time_steps.last_iqr = [float(v) for v in np.percentile(per_step, [25, 75])]
    time_steps.last_replays = (reps, per)
    return float(np.mean(per_step)), float(np.median(per_step)), wall * 1e3 / (reps * per)


def valu_instructions_per_agent_step():
    """VALU wave instructions the fused kernel issues per agent-step on this
    workload (rocprofv3 SQ_INSTS_VALU per launch / agent-steps), recorded next
    to the profile summaries; None if not recorded."""
    path = os.path.join(ROOT, "profiles", "traffic_vswrm_sweep_4096x50x512.json")
    try:
        with open(path) as f:
            return float(json.load(f)["valu_wave_instructions_per_agent_step"]["f32"])
    except (OSError, KeyError, ValueError):
        return None


def traffic_bytes():
    """HBM bytes per launch of the fused kernel on this workload, as measured by
    rocprofv3 FETCH_SIZE / WRITE_SIZE (scaled by a device copy of known size)
    and recorded next to the profile summaries; None if not recorded."""
    path = os.path.join(ROOT, "profiles", "traffic_vswrm_sweep_4096x50x512.json")
    try:
        with open(path) as f:
            return float(json.load(f)["bytes_per_launch"]["f32"])
    except (OSError, KeyError, ValueError):
        return None


# ------------------------------------------------------------ CPU baseline
def _cpu_worker(args):
    core, rep, steps = args
    try:
        os.sched_setaffinity(0, {core})
    except (AttributeError, OSError):
        pass
    from oracle import vf_oracle as vo
    a = np.linspace(0.1, 3.0, B_SIDE)
    i, j = divmod(rep, B_SIDE)
    rng = np.random.RandomState(10000 + rep)
    x = rng.uniform(PAD, PAD + W, N)
    y = rng.uniform(PAD, PAD + W, N)
    th = rng.uniform(0, 2 * np.pi, N)
    v = np.zeros(N)
    p = vo.VFParams(GAM=0.1, V0=1.0, ALP0=float(a[i]), ALP1=0.09, BET0=float(a[j]), BET1=0.09,
                    BOUNDARY="infinite")
    ags = vo.make_agents(x, y, th, v, RADIUS, R, (-np.pi, np.pi), W, W, PAD, p)
    vo.group_update(ags, p)                          # warm-up step
    t0 = time.perf_counter()
    for _ in range(steps):
        vo.group_update(ags, p)
    dt = time.perf_counter() - t0
    return steps * N / dt


def host_cpu():
    """os.cpu_count(), the cores this process may run on, and the CPU model
    (from /proc/cpuinfo, the line lscpu reports as the model name)."""
    model = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    aff = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else os.cpu_count()
    return {"cpu_count": os.cpu_count(), "affinity_cores": aff, "model": model}


# One GPU's share of the host: the GPU box gives each GPU 16 cores, whatever
# os.cpu_count() reports there, so the baseline uses at most 16 processes.
CPU_SHARE = 16


def cpu_baseline(seconds=15.0):
    """The oracle on the host cores, one process per core, one replica each."""
    cores = sorted(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else list(range(os.cpu_count()))
    cores = cores[:CPU_SHARE]
    # size the sample: calibrate one step on one core
    from oracle import vf_oracle as vo  # noqa: F401
    steps = max(2, int(seconds / 0.12))
    steps = min(steps, 60)
    with mp.get_context("spawn").Pool(len(cores)) as pool:
        rates = pool.map(_cpu_worker, [(c, k * 61 % (B_SIDE * B_SIDE), steps)
                                       for k, c in enumerate(cores)])
    return {"value": float(sum(rates)), "unit": "agent-steps/s", "cores": len(cores),
            "kind": "port", "host": host_cpu(),
            "sample": (f"oracle (numpy restatement of the reference step), {len(cores)} processes "
                       f"pinned one per core (at most {CPU_SHARE}: one GPU's share of the host), "
                       f"one replica each (N={N}, R={R}, torus) for {steps} steps after 1 "
                       f"warm-up; per-core rate {np.mean(rates):.1f} agent-steps/s")}


def _line(args, workload, value, ms, dtype, config, **extra):
    out = {"metric": METRIC, "value": value, "unit": "agent-steps/s", "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": dtype, "data": "synthetic",
           "config": dict(workload=workload, **config)}
    out.update(extra)
    print(json.dumps(out), flush=True)


def other_workload(args):
    """Measurements of the other configurations (not the headline line)."""
    import torch
    from abm_amd.vf import VFConfig, VFSwarm
    from abm_amd.forage import ForageConfig, ForageSwarm, ResourceWorld, WorldConfig
    f32 = lambda a: np.asarray(a).astype(np.float32).astype(np.float64)
    if args.workload == "single":
        Ns, Rs, Ws = 100, 1024, 1000.0
        rng = np.random.RandomState(42)
        x, y = f32(rng.uniform(PAD, PAD + Ws, Ns)), f32(rng.uniform(PAD, PAD + Ws, Ns))
        th = f32(rng.uniform(0, 2 * np.pi, Ns))
        cfg = VFConfig(n_agents=Ns, n_rays=Rs, width=Ws, height=Ws, boundary="infinite", ALP0=1.0,
                       BET0=0.5)
        res = {}
        for prec in ("f32", "f64"):
            sw = VFSwarm([cfg], x, y, th, 0.0, radius=5, precision=prec)
            res[prec] = time_steps(sw, args.steps, args.warmup, not args.no_graph)[0]

        class PlainStep:   # every pair in float64: the float64 step that counts its near ties
            step = staticmethod(lambda: sw.step(count=True))
        res["plain"] = time_steps(PlainStep, args.steps, args.warmup, not args.no_graph)[0]
        ops = ops_per_agent_step(Ns, Rs) * Ns
        _line(args, f"single VSWRM replica N={Ns}, R={Rs}, 1000x1000 torus, reference order", Ns / (res["f32"] * 1e-3),
              res["f32"], "f32", {"replicas": 1, "agents_per_replica": Ns, "rays": Rs},
              plain_f64={"agent_steps_per_s": Ns / (res["plain"] * 1e-3), "ms_per_step": res["plain"]},
              speedup_vs_plain_f64=res["plain"] / res["f32"], speedup_vs_float64=res["f64"] / res["f32"],
              float64={"agent_steps_per_s": Ns / (res["f64"] * 1e-3), "ms_per_step": res["f64"]},
              roofline={"bound": "valu", "achieved": ops / (res["f32"] * 1e-3) / 1e12,
                        "peak": VALU_PEAK_TOPS, "unit": "Tops/s",
                        "frac": ops / (res["f32"] * 1e-3) / 1e12 / VALU_PEAK_TOPS, "traffic": None,
                        "note": "one replica occupies one workgroup: latency-bound by design"})
    elif args.workload == "large":
        Nl, Rl, Wl = 8192, 2048, 4000.0
        rng = np.random.RandomState(7)
        x, y = f32(rng.uniform(PAD, PAD + Wl, Nl)), f32(rng.uniform(PAD, PAD + Wl, Nl))
        th = f32(rng.uniform(0, 2 * np.pi, Nl))
        cfg = VFConfig(n_agents=Nl, n_rays=Rl, width=Wl, height=Wl, boundary="infinite", ALP0=1.0,
                       BET0=0.5)
        cpu = None if args.no_cpu else large_cpu_sample(x, y, th, Nl, Rl, Wl, min(args.cpu_seconds, 10.0))
        sw = VFSwarm([cfg], x, y, th, 0.5, radius=2, precision="f32")

        class Sync:
            step = staticmethod(lambda: sw.step(order="synchronous"))
        ms = time_steps(Sync, args.steps, args.warmup, not args.no_graph)[0]
        iqr = getattr(time_steps, "last_iqr", None)
        # the reference's order: the chain step (segments of 256 agents moved
        # in id order by one workgroup, the pairs decided over the GPU)
        sq = VFSwarm([cfg], x, y, th, 0.5, radius=2, precision="f32")
        k_seq = max(5, min(args.steps // 5, 40))
        ms_seq = time_steps(sq, k_seq, min(args.warmup, 5), not args.no_graph)[0]
        iqr_seq = getattr(time_steps, "last_iqr", None)
        kernels_seq = sorted(sq.last_kernels())
        # the same order on the 16-wave kernel (one workgroup, every pose in
        # LDS, each agent's pairs decided in its turn), for comparison
        sb = VFSwarm([cfg], x, y, th, 0.5, radius=2, precision="f32")
        sb.set_launch(16)
        ms_big = time_steps(sb, 5, 2, not args.no_graph)[0]
        # pairs a step must decide: those inside the exact visibility cut-off
        # r cot(2 pi / R) (beyond it floor(proj_size / 2) = 0 and nothing is
        # drawn, vf_supcalc.py:116-117), torus images, from the start state
        cut = 2.0 / np.tan(2 * np.pi / Rl)
        eff = 0
        for i0 in range(0, Nl, 512):
            dx = np.abs(x[i0:i0 + 512, None] - x[None, :])
            dy = np.abs(y[i0:i0 + 512, None] - y[None, :])
            dx = np.minimum(dx, Wl - dx)
            dy = np.minimum(dy, Wl - dy)
            eff += int(((dx * dx + dy * dy) <= cut * cut).sum())
        eff -= Nl                                   # each agent with itself
        ops = 40 * eff + (17 * Rl + 20) * Nl
        ach = ops / (ms_seq * 1e-3) / 1e12
        ach_sync = ops / (ms * 1e-3) / 1e12
        note = ("lane-ops of the pairs inside the visibility cut-off (40 each) and of every agent's "
                "rays (17 each) and update (20)")
        extra = {"cpu_baseline": cpu} if cpu is not None else {}
        _line(args, f"one flock N={Nl}, R={Rl}, radius 2, 4000x4000 torus, reference order (chain "
                    f"step: agents moved in id order, pairs decided over the GPU)",
              Nl / (ms_seq * 1e-3), ms_seq, "f32", {"replicas": 1, "agents_per_replica": Nl, "rays": Rl,
                                                     "order": "sequential"},
              ms_per_step_iqr=iqr_seq, kernels=kernels_seq,
              sixteen_wave_kernel={"ms_per_step": ms_big, "speedup": ms_big / ms_seq},
              roofline={"bound": "valu", "achieved": ach, "peak": VALU_PEAK_TOPS, "unit": "Tops/s",
                        "frac": ach / VALU_PEAK_TOPS, "traffic": None,
                        "note": note + "; the id-order chain runs on one workgroup (one segment at a "
                                       "time): latency-bound"},
              synchronous_order={"agent_steps_per_s": Nl / (ms * 1e-3), "ms_per_step": ms,
                                 "ms_per_step_iqr": iqr, "kernel": "wide (grid cells, one wave per agent)",
                                 "roofline_frac": ach_sync / VALU_PEAK_TOPS,
                                 "note": "not the reference's order: every field from the step's "
                                         "start poses"},
              effective_pairs_per_step=eff, nominal_pairs_per_step=Nl * (Nl - 1),
              pair_ray_evals_per_s=eff * Rl / (ms_seq * 1e-3),
              nominal_pair_ray_evals_per_s=Nl * (Nl - 1) * Rl / (ms_seq * 1e-3), **extra)
    elif args.workload == "cs":
        return cs_workload(args)
    elif args.workload == "c1":
        return c1_workload(args)
    elif args.workload == "c5overlay":
        return c5_overlay_workload(args)
    else:   # mixed ragged batch: even replicas forage, odd replicas flock
        cpu = None if args.no_cpu else mixed_cpu_baseline(args.cpu_seconds)
        vf_cfgs, fg_cfgs, vx, fx_ = [], [], [], []
        for b, (n, r) in enumerate(mixed_shapes()):
            side = 100.0 * np.sqrt(n)
            srng = np.random.RandomState(20000 + b)
            pos = (f32(srng.uniform(PAD, PAD + side, n)), f32(srng.uniform(PAD, PAD + side, n)),
                   f32(srng.uniform(0, 2 * np.pi, n)))
            if b % 2:
                vf_cfgs.append(VFConfig(n_agents=n, n_rays=r, width=side, height=side,
                                        boundary="infinite", ALP0=1.0, BET0=0.5))
                vx.append(pos)
            else:
                fg_cfgs.append(ForageConfig(n_agents=n, n_rays=r, width=side, height=side,
                                            vision_range=2000.0))
                fx_.append(pos)
        cat = lambda L, i: np.concatenate([p[i] for p in L])
        vsw = VFSwarm(vf_cfgs, cat(vx, 0), cat(vx, 1), cat(vx, 2), 0.5, radius=5, precision="f32")
        fsw = ForageSwarm(fg_cfgs, cat(fx_, 0), cat(fx_, 1), cat(fx_, 2), radius=10,
                          rngs=[np.random.RandomState(30000 + i) for i in range(len(fg_cfgs))])
        # each foraging replica runs the whole loop body: 10 patches of radius
        # 30, quality U[0.5, 1], 200..1000 units, regenerated when depleted
        # (the generators on the device: no host work or synchronisation per step)
        world = ResourceWorld(fsw, [WorldConfig(N_resc=10, patch_radius=30, min_resc_quality=0.5,
                                                max_resc_quality=1.0, teleport_exploit=False)
                                    for _ in fg_cfgs], device_rng=True)
        world.create_resources()
        chosen, chosen_ms = vsw.autotune(trial_steps=3)
        ms_vf = time_steps(vsw, args.steps, args.warmup, not args.no_graph)[0]
        vf_kernels = sorted(vsw.last_kernels())
        for _ in range(min(args.warmup, 3)):
            world.step()
        torch.cuda.synchronize()
        n_fs = max(3, min(args.steps, 20))
        t0 = time.perf_counter()
        for _ in range(n_fs):
            world.step()
        torch.cuda.synchronize()
        ms_fg = (time.perf_counter() - t0) * 1e3 / n_fs
        world.sync_rng()
        n_vf = int(vsw.batch.info.n_agents_total)
        n_fg = int(fsw.info.n_agents_total)
        ms = ms_vf + ms_fg
        ops_vf = sum(c.n_agents * ops_per_agent_step(c.n_agents, c.n_rays) for c in vf_cfgs)
        ach = ops_vf / (ms_vf * 1e-3) / 1e12
        extra = {"roofline": {"bound": "valu", "achieved": ach, "peak": VALU_PEAK_TOPS, "unit": "Tops/s",
                              "frac": ach / VALU_PEAK_TOPS, "traffic": None,
                              "kernel": "flocking half (the autotuned launch), lane-ops of every "
                                        "flocking agent-step over its graph-replay time"}}
        if cpu is not None:
            extra["cpu_baseline"] = cpu
        _line(args, "2000 ragged replicas (N log-uniform 8..512, R in {256,512,1024}, side 100*sqrt(N)): "
                    "odd replicas flock (fused float32), even replicas forage (float64) among 10 "
                    "resource patches each (interaction, regeneration and update on the device)",
              (n_vf + n_fg) / (ms * 1e-3), ms, "f32+f64",
              {"replicas": 2000, "agents_flocking": n_vf, "agents_foraging": n_fg},
              flocking={"agent_steps_per_s": n_vf / (ms_vf * 1e-3), "ms_per_step": ms_vf,
                        "ms_per_step_iqr": getattr(time_steps, "last_iqr", None),
                        "launch": {"autotuned": chosen, "trial_ms": chosen_ms, "kernels": vf_kernels,
                                   "note": "abm_vf_set_launch value: 32 the push kernel for every "
                                           "replica, 0 the size classes, 1/2/4 the per-replica "
                                           "kernel, -1/-2/-4 the grouped kernel"}},
              foraging={"agent_steps_per_s": n_fg / (ms_fg * 1e-3), "ms_per_step_wall": ms_fg},
              **extra)


def large_cpu_sample(x, y, th, N, R, W, seconds):
    """The oracle on one core for the 8192-agent flock: VFAgent.update of a
    sample of agents (each sees all 8191 others), scaled to a step.  The
    reference itself cannot hold this flock: its field is an (N-1) x R
    float64 matrix per agent (vf_supcalc.py:38), 134 MB here."""
    from oracle import vf_oracle as vo
    p = vo.VFParams(ALP0=1.0, BET0=0.5, BOUNDARY="infinite")
    v = np.full(N, 0.5)
    t0, n = time.perf_counter(), 0
    while n < 1 or (time.perf_counter() - t0 < seconds and n < 50):
        vo.agent_view_step(x, y, th, v, 2, (n * 997) % N, R, (-np.pi, np.pi), W, W, PAD, p)
        n += 1
    per = (time.perf_counter() - t0) / n
    return {"value": 1.0 / per, "unit": "agent-steps/s", "cores": 1, "kind": "port",
            "sample": f"oracle VFAgent.update of {n} agents of the 8192-agent flock ({per:.2f} s "
                      f"each, one core); a whole step would take {per * N / 3600:.1f} h"}


def mixed_shapes():
    """(N, R) of the 2000 ragged replicas: N log-uniform in [8, 512], R in
    {256, 512, 1024}; even replicas forage, odd replicas flock."""
    rng = np.random.RandomState(20000)
    out = []
    for b in range(2000):
        n = int(round(np.exp(rng.uniform(np.log(8), np.log(512)))))
        r = int(rng.choice([256, 512, 1024]))
        out.append((n, r))
    return out


def _mixed_cpu_worker(args):
    core, b, seconds = args
    try:
        os.sched_setaffinity(0, {core})
    except (AttributeError, OSError):
        pass
    n, r = mixed_shapes()[b]
    side = 100.0 * np.sqrt(n)
    srng = np.random.RandomState(20000 + b)
    x, y, th = srng.uniform(PAD, PAD + side, n), srng.uniform(PAD, PAD + side, n), srng.uniform(0, 2 * np.pi, n)
    if b % 2:
        from oracle import vf_oracle as vo
        p = vo.VFParams(ALP0=1.0, BET0=0.5, BOUNDARY="infinite")
        ags = vo.make_agents(x, y, th, np.full(n, 0.5), 5, r, (-np.pi, np.pi), side, side, PAD, p)
        step = lambda: vo.group_update(ags, p)
    else:
        from oracle import forage_oracle as fo
        fp = fo.ForageParams()
        ags = [fo.ForageAgent(i, 10, (x[i], y[i]), th[i], r, (-np.pi, np.pi), side, side, PAD, 2000.0,
                              False, True, fp) for i in range(n)]
        np.random.seed(30000 + b)
        world = fo.ForageWorld(ags, side, side, PAD, 10, 30, 200, 1000, 0.5, 1.0, teleport_exploit=False)
        step = world.step
    t0, k = time.perf_counter(), 0
    while k < 1 or (time.perf_counter() - t0 < seconds and k < 50):
        step()
        k += 1
    return n, (time.perf_counter() - t0) / k


def mixed_cpu_baseline(seconds=15.0):
    """The oracle on the uneven batch: one replica per core (at most one
    GPU's share of the host), sampled across the N / R mix (8 flocking and 8
    foraging replicas spread over the sorted costs), each for at least one
    step; the rate is sum(N) / sum(seconds per step) per core, times the
    cores."""
    cores = sorted(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else list(range(os.cpu_count()))
    cores = cores[:CPU_SHARE]
    shapes = mixed_shapes()
    pick = []
    for parity in (1, 0):
        idx = sorted((b for b in range(len(shapes)) if b % 2 == parity),
                     key=lambda b: shapes[b][0] * shapes[b][0] + shapes[b][0] * shapes[b][1])
        half = len(cores) // 2
        pick += [idx[int((i + 0.5) * len(idx) / half)] for i in range(half)]
    with mp.get_context("spawn").Pool(len(cores)) as pool:
        res = pool.map(_mixed_cpu_worker, [(c, b, seconds / 3) for c, b in zip(cores, pick)])
    per_core = sum(n for n, _ in res) / sum(t for _, t in res)
    return {"value": per_core * len(cores), "unit": "agent-steps/s", "cores": len(cores), "kind": "port",
            "host": host_cpu(),
            "sample": f"oracle (VSWRM group_update / ForageWorld.step) on {len(pick)} replicas of the "
                      f"batch spread over its cost range, one per core, at least one step each; "
                      f"ratio estimate sum(N) / sum(s per step) = {per_core:.1f} agent-steps/s per core"}


def cs_workload(args):
    """Cooperative-signalling perception of every agent of 1000 replicas
    (N=50, R=1200, FOV 0.45 pi, 600x600 arena): the crowding density (sum over
    the 49 others, max_proj_size = 0.5 R) and the signalling density (maximum
    over 20 current signallers and 4 remembered steps of 20, decayed meters)."""
    import torch
    from abm_amd.cs import CSProjection
    B, N, R, Wc, S, MEM = 1000, 50, 1200, 600.0, 20, 5
    fov = (-0.45 * np.pi, 0.45 * np.pi)
    rng = np.random.RandomState(77)
    dev = torch.device("cuda")
    pos = rng.uniform(PAD, PAD + Wc, (B, N, 2))
    th = rng.uniform(0, 2 * np.pi, (B, N))
    focal = np.concatenate([pos, np.full((B, N, 1), 10.0), th[..., None]], axis=2).reshape(-1, 4)
    # crowding: the others of the same replica
    idx = np.array([[j for j in range(N) if j != k] for k in range(N)])
    crowd_obj = pos[:, idx, :].reshape(-1, 2)
    crowd_off = np.arange(B * N + 1, dtype=np.int64) * (N - 1)
    # signalling: S current positions and MEM-1 remembered steps (the same for
    # every agent of a replica; the kernel takes one list per focal agent)
    sig_pos = rng.uniform(PAD, PAD + Wc, (B, MEM, S, 2))
    sig_met = rng.uniform(0, 1, (B, MEM, S)) * (1 - np.arange(MEM) / MEM)[None, :, None]
    sig_obj = np.repeat(sig_pos.reshape(B, 1, MEM * S, 2), N, axis=1).reshape(-1, 2)
    sig_m = np.repeat(sig_met.reshape(B, 1, MEM * S), N, axis=1).reshape(-1)
    sig_off = np.arange(B * N + 1, dtype=np.int64) * (MEM * S)
    T = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)
    F, CO, CF, SO, SM, SF = (T(focal), T(crowd_obj), T(crowd_off, torch.int64), T(sig_obj), T(sig_m),
                             T(sig_off, torch.int64))
    norm = torch.full((B * N,), float(N), dtype=torch.float64, device=dev)
    crowd = CSProjection(R, fov, 0.5 * R, check_offsets=False)
    sig = CSProjection(R, fov, None, check_offsets=False)
    out_c = torch.empty((B * N, R), dtype=torch.float64, device=dev)
    out_s = torch.empty((B * N, R), dtype=torch.float64, device=dev)
    s = torch.cuda.current_stream()

    def step():
        crowd.sum(F, CF, CO, norm, out=out_c, stream=s)
        sig.max(F, SF, SO, SM, out=out_s, stream=s)
    for _ in range(max(2, args.warmup // 10)):
        step()
    torch.cuda.synchronize()
    k = max(3, min(args.steps, 20))
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(s)
    for _ in range(k):
        step()
    e1.record(s)
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / k
    cells = B * N * ((N - 1) + MEM * S) * R
    _line(args, f"cooperative-signalling perception: {B} replicas x N={N} x R={R}, FOV 0.45 pi, "
                f"crowding (49 others) + signalling ({MEM * S} remembered signallers)",
          B * N / (ms * 1e-3), ms, "f64", {"replicas": B, "agents_per_replica": N, "rays": R},
          object_ray_cells_per_s=cells / (ms * 1e-3),
          note="agent-steps/s counts focal agents whose two projections were computed")


C1_ENV = dict(T_w=0.5, Eps_w=3.0, g_w=0.085, B_w=0.0, w_max=1.0, T_u=0.5, Eps_u=1.0, g_u=0.085,
              B_u=0.0, u_max=1.0, S_wu=0.25, S_uw=0.01, Tau=10, F_N=0.5, F_R=0.5, exp_vel_max=3.0,
              exp_theta_min=-0.5, exp_theta_max=0.5, reloc_theta_max=1.8, exp_stop_ratio=0.175)
C1_WORLD = dict(N_resc=10, patch_radius=30, min_resc_perpatch=200, max_resc_perpatch=1000,
                min_resc_quality=0.5, max_resc_quality=1.0, teleport_exploit=False)


def _c1_start(seed, N=10, W=500):
    """Simulation.create_agents of the C1 case (sims.py:526-532): positions
    from randint, orientations from uniform, on the replica's own stream."""
    g = np.random.RandomState(seed)
    x, y, th = [], [], []
    for _ in range(N):
        x.append(float(g.randint(PAD - 10, W + PAD - 10)))
        y.append(float(g.randint(PAD - 10, W + PAD - 10)))
        th.append(g.uniform(0, 2 * np.pi))
    return g, x, y, th


def c1_workload(args):
    """The reference's own CPU case (C1): collective foraging, N=10 agents of
    radius 10, 10 patches (radius 30, quality U[0.5, 1]) in a 500x500
    reflective arena, R=1200 over 2 pi, the .env decision values; the whole
    loop body (resources, regeneration, Agent.update) per step on the device,
    one replica as the reference runs it and 1000 seeds in one batch, with the
    generators on the device (and, for one replica, on the host).  The
    oracle's ForageWorld (numpy, one core) is timed first on the same case."""
    from oracle import forage_oracle as fo
    N, R, W = 10, 1200, 500
    p = fo.ForageParams(**C1_ENV)
    g, x, y, th = _c1_start(42)
    ags = [fo.ForageAgent(i, 10, (x[i], y[i]), th[i], R, (-np.pi, np.pi), W, W, PAD, 2000.0, False,
                          True, p, pooling_time=0) for i in range(N)]
    np.random.set_state(g.get_state())
    world = fo.ForageWorld(ags, W, W, PAD, 10, 30, 200, 1000, 0.5, 1.0, regenerate=True,
                           teleport_exploit=False)
    world.step()
    t0, n_cpu = time.perf_counter(), 0
    while time.perf_counter() - t0 < min(args.cpu_seconds, 10.0):
        world.step()
        n_cpu += 1
    cpu_rate = n_cpu * N / (time.perf_counter() - t0)

    import torch
    from abm_amd.forage import ForageConfig, ForageSwarm, ResourceWorld, WorldConfig
    cfg = ForageConfig(n_agents=N, n_rays=R, width=W, height=W, window_pad=PAD, vision_range=2000.0,
                       **{k: v for k, v in C1_ENV.items()})

    def run(n_rep, steps, warmup, device_rng=True):
        starts = [_c1_start(42 + b) for b in range(n_rep)]
        sw = ForageSwarm([cfg] * n_rep, sum((s[1] for s in starts), []), sum((s[2] for s in starts), []),
                         sum((s[3] for s in starts), []), radius=10, rngs=[s[0] for s in starts])
        rw = ResourceWorld(sw, [WorldConfig(**C1_WORLD)] * n_rep, device_rng=device_rng)
        rw.create_resources()
        for _ in range(warmup):
            rw.step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            rw.step()
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) * 1e3 / steps
        rw.sync_rng()
        return ms

    k = max(20, min(args.steps, 1000))
    ms1 = run(1, k, max(5, args.warmup // 10))
    ms1_host = run(1, k, max(5, args.warmup // 10), device_rng=False)
    msb = run(1000, max(10, k // 10), 3)
    _line(args, "C1 collective foraging: N=10, R=1200, 10 patches (radius 30, quality U[0.5, 1]), "
                "500x500 walls; resource loop and Agent.update on the device, one replica",
          N / (ms1 * 1e-3), ms1, "f64", {"replicas": 1, "agents_per_replica": N, "rays": R},
          batched_1000_seeds={"agent_steps_per_s": 1000 * N / (msb * 1e-3), "ms_per_step_wall": msb},
          host_generators={"agent_steps_per_s": N / (ms1_host * 1e-3), "ms_per_step_wall": ms1_host,
                           "note": "numpy generators peeked and skipped on the host every step"},
          cpu_baseline={"value": cpu_rate, "unit": "agent-steps/s", "cores": 1, "kind": "port",
                        "sample": f"oracle ForageWorld (numpy restatement of the loop body), the same "
                                  f"C1 world, {n_cpu} steps on one core"},
          note="wall time per step; the replicas' MT19937 generators live on the device "
               "(written back to numpy after the timed steps)")


C5_WORLD = dict(N_resc=64, patch_radius=30, min_resc_perpatch=200, max_resc_perpatch=1000,
                min_resc_quality=0.5, max_resc_quality=1.0, teleport_exploit=False)


def _c5_start(seed, N=8192, W=4000, r=2):
    """Simulation.create_agents (sims.py:526-532) for the large population:
    randint positions over [pad - r, W + pad - r), uniform orientations."""
    g = np.random.RandomState(seed)
    x, y, th = [], [], []
    for _ in range(N):
        x.append(float(g.randint(PAD - r, W + PAD - r)))
        y.append(float(g.randint(PAD - r, W + PAD - r)))
        th.append(g.uniform(0, 2 * np.pi))
    return g, x, y, th


def c5_cpu_sample(N, R, W, r, seconds):
    """The oracle on one core for the large population: Agent.update of a
    sample of agents inside the full 8192-agent world plus one resource
    interaction pass, scaled to a whole step (one reference step would take
    minutes)."""
    from oracle import forage_oracle as fo
    p = fo.ForageParams(**C1_ENV)
    g, x, y, th = _c5_start(7, N, W, r)
    ags = [fo.ForageAgent(i, r, (x[i], y[i]), th[i], R, (-np.pi, np.pi), W, W, PAD, 2000.0, False,
                          True, p, pooling_time=0) for i in range(N)]
    np.random.set_state(g.get_state())
    world = fo.ForageWorld(ags, W, W, PAD, 64, 30, 200, 1000, 0.5, 1.0, regenerate=True,
                           teleport_exploit=False)
    # the interaction's membership pass: every patch against every agent
    t0 = time.perf_counter()
    groups = [[a for a in ags if fo.distance(q, a) < q.radius] for q in world.patches]
    t_inter = time.perf_counter() - t0
    del groups
    t0, n = time.perf_counter(), 0
    while time.perf_counter() - t0 < seconds and n < N:
        fo.agent_update(ags[(n * 997) % N], ags)
        n += 1
    t_agent = (time.perf_counter() - t0) / n
    step_s = N * t_agent + t_inter
    return {"value": N / step_s, "unit": "agent-steps/s", "cores": 1, "kind": "port",
            "sample": f"oracle Agent.update of {n} agents sampled from the 8192-agent world "
                      f"({t_agent * 1e3:.1f} ms each) plus one membership pass of the resource "
                      f"loop ({t_inter:.1f} s), scaled to one step ({step_s:.0f} s) on one core"}


def c5_overlay_workload(args):
    """The foraging overlay of the large flock: the collective-foraging loop
    body (resource interaction and regeneration, sims.py:789-858, then
    Agent.update in id order, sims.py:861) for one population of N=8192
    agents of radius 2, R=2048 over 2 pi, on the 4000x4000 arena with walls
    (the foraging agent's only boundary, agent.py:279), 64 resource patches
    of radius 30 with quality U[0.5, 1] and 200..1000 units, the C1 decision
    values, vision range 2000, generators on the device.  The replica
    exceeds one workgroup's LDS, so the update runs over the whole GPU."""
    import torch
    from abm_amd.forage import ForageConfig, ForageSwarm, ResourceWorld, WorldConfig
    N, R, W, r = 8192, 2048, 4000, 2
    cpu = None if args.no_cpu else c5_cpu_sample(N, R, W, r, min(args.cpu_seconds, 10.0))
    cfg = ForageConfig(n_agents=N, n_rays=R, width=W, height=W, window_pad=PAD, vision_range=2000.0,
                       **C1_ENV)
    g, x, y, th = _c5_start(7, N, W, r)
    sw = ForageSwarm([cfg], x, y, th, radius=r, rngs=[g])
    rw = ResourceWorld(sw, [WorldConfig(**C5_WORLD)], device_rng=True)
    rw.create_resources()
    for _ in range(max(3, min(args.warmup, 20))):
        rw.step()
    torch.cuda.synchronize()
    s0, w0 = sw.sweep_counts()
    k = max(5, min(args.steps, 100))
    times = []
    for _ in range(k):
        t0 = time.perf_counter()
        rw.step()
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
    s1, w1 = sw.sweep_counts()
    rw.sync_rng()
    ms = float(np.mean(times)) * 1e3
    q25, q50, q75 = (float(v) * 1e3 for v in np.percentile(times, [25, 50, 75]))
    st = sw.get_state("overriding_mode", "exploited_patch_id")
    expl = int(((st["overriding_mode"] == 1) & (st["exploited_patch_id"] != -1)).sum())
    # algorithmic work of one agent-step without visual exclusion: a record of
    # each exploiting cue (40 lane-ops, as a pair of the flocking model), the
    # raster and counts (3 per ray), the decision and move (60)
    ops = N * (40 * expl + 3 * R + 60)
    achieved = ops / (ms * 1e-3) / 1e12
    extra = {"roofline": {"bound": "valu", "achieved": achieved, "peak": VALU_PEAK_TOPS,
                          "unit": "Tops/s", "frac": achieved / VALU_PEAK_TOPS, "traffic": None,
                          "note": "latency-bound: six small launches per step; ops counted once "
                                  "per agent-step with the exploiting cues at the end of the run"}}
    if cpu is not None:
        extra["cpu_baseline"] = cpu
    _line(args, f"foraging overlay of the large flock: N={N} agents of radius 2, R={R}, 4000x4000 "
                f"walls, 64 patches (radius 30, quality U[0.5, 1]), resource loop and Agent.update "
                f"in id order on the device",
          N / (ms * 1e-3), ms, "f64", {"replicas": 1, "agents_per_replica": N, "rays": R,
                                        "patches": 64},
          ms_per_step_median=q50, ms_per_step_iqr=[q25, q75],
          sweeps_per_step=(w1 - w0) / max(1, s1 - s0), exploiting_cues_at_end=expl,
          note="wall time per step", **extra)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--steps-f64", type=int, default=20)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-graph", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--workload", default="sweep",
                    choices=["sweep", "single", "mixed", "large", "cs", "c1", "c5overlay"],
                    help="sweep: 4096 replicas x N=50 x R=512 (default, the headline); single: "
                         "one replica N=100, R=1024, 1000x1000 torus; mixed: 2000 ragged replicas, "
                         "half foraging, half flocking; large: one flock N=8192, R=2048, "
                         "4000x4000 torus, synchronous order; cs: cooperative-signalling "
                         "perception of 1000 replicas x N=50 x R=1200; c1: the reference's CPU "
                         "foraging case (N=10, R=1200, 10 patches) on the device, with the "
                         "oracle timed on one core; c5overlay: the foraging overlay of the "
                         "large flock (N=8192, R=2048, 64 patches, 4000x4000)")
    ap.add_argument("--copy-probe", type=int, default=0, metavar="MIB",
                    help="only copy MIB MiB device-to-device 5 times (calibrates the "
                         "FETCH_SIZE / WRITE_SIZE counters) and exit")
    args = ap.parse_args()
    if args.copy_probe:
        import torch
        src = torch.ones(args.copy_probe * (1 << 20) // 4, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_probe_bytes": src.numel() * 4, "copies": 5}))
        return
    if args.gpus != 1:
        print(f"bench.py runs on one GPU: the replicas are independent and the workload "
              f"is one GPU's share; --gpus {args.gpus} is not supported", file=sys.stderr)
        sys.exit(2)

    if args.workload != "sweep":
        return other_workload(args)

    # the CPU baseline runs first, in worker processes started before this
    # process touches the GPU
    cpu = None if args.no_cpu else cpu_baseline(args.cpu_seconds)

    import torch
    from abm_amd.vf import VFSwarm

    cfgs, x, y, th = make_workload()
    n_rep = len(cfgs)
    agents = n_rep * N

    # fixed error: one step of each kernel from the same state in synchronous
    # order, where every agent sees the same (pre-step) poses in both kernels,
    # so the fields must be identical and the pose error is the float32 error
    def one_step(order, kahan=False):
        s64 = VFSwarm(cfgs, x, y, th, 0.5, radius=RADIUS, precision="f64")
        s32 = VFSwarm(cfgs, x, y, th, 0.5, radius=RADIUS, precision="f32")
        s64.step(order=order, fields=True, count=True)
        s32.step(order=order, fields=True, count=True, kahan=kahan)
        torch.cuda.synchronize()
        a64, a32 = s64.state_numpy(), s32.state_numpy()
        dx = np.abs((a32[0] - a64[0] + W / 2) % W - W / 2) / np.maximum(np.abs(a64[0]), 1.0)
        dy = np.abs((a32[1] - a64[1] + W / 2) % W - W / 2) / np.maximum(np.abs(a64[1]), 1.0)
        dth = np.abs((a32[2] - a64[2] + np.pi) % (2 * np.pi) - np.pi) / np.maximum(np.abs(a64[2]), 1.0)
        dv = np.abs(a32[3] - a64[3]) / np.maximum(np.abs(a64[3]), 1.0)
        e = np.max(np.stack([dx, dy, dth, dv]), axis=0)
        words = (R + 31) // 32
        f64b = s64.fields.cpu().numpy().reshape(-1, words)
        f32b = s32.fields.cpu().numpy().reshape(-1, words)
        same = (f64b == f32b).all(axis=1)
        pairs, rechecked, _ = s32.fallback_counts()
        one_step.near_ties = s64.near_ties()
        one_step.pairs = pairs
        return e, same, rechecked / max(pairs, 1)

    e_sync, same_sync, recheck_frac = one_step("synchronous")
    near_ties, near_pairs = one_step.near_ties, one_step.pairs
    e_seq, same_seq, _ = one_step("sequential")
    e_kahan, same_kahan, _ = one_step("synchronous", kahan=True)
    del one_step

    # timing
    sw32 = VFSwarm(cfgs, x, y, th, 0.0, radius=RADIUS, precision="f32")
    sw64 = VFSwarm(cfgs, x, y, th, 0.0, radius=RADIUS, precision="f64")
    ms32_mean, ms32_med, wall32 = time_steps(sw32, args.steps, args.warmup, not args.no_graph)
    iqr32, replays32 = getattr(time_steps, "last_iqr", None), getattr(time_steps, "last_replays", (0, 0))

    class PlainStep:   # every pair in float64: the float64 step that counts its near ties
        step = staticmethod(lambda: sw64.step(count=True))
    ms64_mean, ms64_med, wall64 = time_steps(PlainStep, args.steps_f64, min(args.warmup, 3),
                                             not args.no_graph)
    ms64g_mean = time_steps(sw64, args.steps_f64, min(args.warmup, 3), not args.no_graph)[0]
    swk = VFSwarm(cfgs, x, y, th, 0.0, radius=RADIUS, precision="f32")

    class KahanStep:
        step = staticmethod(lambda: swk.step(kahan=True))
    ms_kahan = time_steps(KahanStep, min(args.steps, 50), min(args.warmup, 10), not args.no_graph)[0]
    rate32 = agents / (ms32_mean * 1e-3)
    rate64 = agents / (ms64_mean * 1e-3)
    ops = ops_per_agent_step(N, R) * agents
    achieved = ops / (ms32_mean * 1e-3) / 1e12

    out = {
        "metric": METRIC,
        "value": rate32,
        "unit": "agent-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms32_mean,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": (f"batched VSWRM sweep: {n_rep} replicas (64x64 ALP0 x BET0 in "
                         f"[0.1,3]^2) x N={N} agents x R={R} rays, 707x707 periodic, "
                         f"reference update order, fused float32 kernel under a HIP graph"),
            "replicas": n_rep, "agents_per_replica": N, "rays": R,
        },
        "plain_f64": {"agent_steps_per_s": rate64, "ms_per_step": ms64_mean,
                      "steps": args.steps_f64,
                      "roofline_frac": ops / (ms64_mean * 1e-3) / 1e12 / VALU_PEAK_TOPS,
                      "note": ("the same lane-op count over the plain float64 kernel's time (a diagnostic "
                               "step, near-tie counts on; not what a float64 user runs); its float64 transcendentals and one wave per replica keep "
                               "VALUBusy near 58 % (rocprofv3), against about 82 % for the fused kernel")},
        "speedup_vs_plain_f64": rate32 / rate64,
        "speedup_vs_float64": ms64g_mean / ms32_mean,   # the float64 step that users get
        "float64": {"agent_steps_per_s": agents / (ms64g_mean * 1e-3), "ms_per_step": ms64g_mean,
                    "note": "the default float64 step: decisions in guarded float32, all else in float64"},
        "fixed_error": {
            "one_step_rel_err_vs_f64": float(e_sync.max()),
            "fields_bit_exact_vs_f64": bool(same_sync.all()),
            "order": "synchronous (identical per-agent views in both kernels)",
            "sequential_order_fields_identical_frac": float(same_seq.mean()),
            "sequential_order_rel_err_median": float(np.median(e_seq)),
            "sequential_order_rel_err_max_where_fields_identical":
                float(e_seq[same_seq].max()) if same_seq.any() else None,
            "f64_rechecked_pair_fraction": recheck_frac,
            "f64_near_tie_pairs": near_ties,
            "f64_near_tie_note": (f"pairs of the float64 step (of {near_pairs}) whose bin or "
                                  f"half-width decision lies within 1e-12 of its tie, where device "
                                  f"and host libm may round to opposite sides"),
        },
        "kahan_sums": {
            "one_step_rel_err_vs_f64": float(e_kahan.max()),
            "fields_bit_exact_vs_f64": bool(same_kahan.all()),
            "ms_per_step": ms_kahan,
            "time_ratio_vs_default": ms_kahan / ms32_mean,
            "note": "ABM_KAHAN_SUMS: Kahan-compensated ray sums per lane, group sums in float64 "
                    "(the default: nibble-table sums and a float32 DPP tree)",
        },
        "pair_ray_evals_per_s": agents * (N - 1) * R / (ms32_mean * 1e-3),
        "ms_per_step_median": ms32_med,
        "ms_per_step_iqr": iqr32,
        "graph_replays": {"replays": replays32[0], "steps_per_replay": replays32[1]},
        "wall_ms_per_step": wall32,
        "roofline": {
            "bound": "valu",
            "achieved": achieved,
            "peak": VALU_PEAK_TOPS,
            "unit": "Tops/s",
            "frac": achieved / VALU_PEAK_TOPS,
            "traffic": traffic_bytes(),
            "ops_per_launch": ops,
            "note": "achieved counts the op model's lane-ops (40 per pair, 17 per ray, 20 per "
                    "agent: 10,684 per agent-step here), not what the bit-packed kernel issues; "
                    "issue_frac is the issued VALU lane slots (profiled VALU wave instructions "
                    "per agent-step x 64) over the same peak",
        },
    }
    vpa = valu_instructions_per_agent_step()
    if vpa is not None:
        out["roofline"]["valu_wave_instructions_per_agent_step"] = vpa
        out["roofline"]["issue_frac"] = vpa * 64 * agents / (ms32_mean * 1e-3) / 1e12 / VALU_PEAK_TOPS
    if cpu is not None:
        out["cpu_baseline"] = cpu
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
