"""Benchmark: trajectories/s to tf on one GPU at <= 1e-6 rel L2 error vs FP64, batched vs plain.

Headline workload: a mixed batch of independent trajectories, half of each family
(--count per family, default 4096, 8192 in all), seeded:
  ks   Kuramoto-Sivashinsky u_t = -u_xx - u_xxxx - u u_x on [0, D): n ~ U{256, 512, 1024,
       2048, 4096} (rfft), D ~ U[22, 200], u0 = sum_{k<=8} a_k cos(2 pi k x / D + theta_k),
       a_k ~ N(0, 0.1^2), theta_k ~ U[0, 2 pi); IF34, epsilon 1e-5, tf 100
  nls  cubic NLS u_t = (i/2) u_xx + i |u|^2 u on [-64, 64): n ~ U{1024, 2048, 4096, 8192} (fft),
       1-3 sech solitons with amplitudes U[1, 2.5], speeds U[-2, 2], positions U[-40, 40],
       random phases; ETD35, epsilon 1e-6, tf 20
A "step" is the whole batch integrated t0 -> tf (both families' plans launched together
on two streams), inputs resident in HBM.  The learned step-size proposer is trained on the
device from the solver's own accept/reject records (separate seeds) before anything is
timed.

Variants (FP64 coefficient generation, error norm and dt control on the device in all):
  f64            FP64 throughout (the parity path)
  mixed          FP64 state, propagators exp(f h L) and FFTs; FP32 NL arrays and psi
                 coefficients
  f32            FP32 state, stages and FFTs
  f32+learned    f32 with the learned proposer choosing the step after each accept
  mixed+learned  mixed with the learned proposer
Each variant's error is the rel L2 distance at tf to the FP64 batch, per trajectory (max
and median per family).  The FP64 step-sequence floor (FP64 with safety_f 0.79 instead of
0.8) is measured beside it: the chaotic KS family and the multi-soliton NLS collisions
move far beyond 1e-6 under any change of the step sequence.  A variant passes the gate on
a family when its max and median errors are <= max(1e-6, the floor's max / median).  The
headline value is the fastest variant that passes on both families; K timed steps of it
follow W warm-up steps.

Also in the line:
  * plain_fp64: the reference's API, one drop-in solver evolve per trajectory on the GPU
    (FP64), timed on a sample of each (family, n) and weighted by the batch's size mix;
  * roofline: the dominant kernel (the n = 8192 NLS bucket) of the headline variant run
    alone, algorithmic bytes per launch / launch time from HIP events on its stream;
  * single: the single-instance workloads (KS n = 1024 IF34 tf 50; two-soliton NLS
    n = 8192 ETD35 tf 20 in FP64, FP32 and mixed) on the GPU drop-in and on one CPU core;
  * workloads: the KS ensemble (4096 trajectories, IF34 and ETD35, tf 100), the 2-D
    Allen-Cahn batch (64 x 512^2, ETD35, tf 10) and a radial NLS batch (2048 trajectories,
    Hankel nr = 100, ETD35), one timed pass per precision;
  * cpu_baseline: the NumPy FP64 oracle on a stratified sample of the headline batch,
    one trajectory per host core.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--count C] [--no-cpu]
                       [--variants f64,mixed,f32,f32+learned[,mixed+learned]]
                       [--workloads single,ks,ac2d,radial] [--only roofline|batch|ks|ac2d|radial]
                       [--variant V] [--copy-mib X]
"""
import argparse
import json
import multiprocessing as mp
import os
import platform
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

# Hardware queues per process, read when the HIP runtime starts.  The batch runs nine
# size buckets on private streams beside the two family streams; with HIP's default
# of 4 queues, streams share a queue and a kernel waits behind every packet queued
# before it there (other buckets, the joins), so buckets that could overlap run one
# after another.  Measured on the mixed batch: 4 or 8 queues 5.7 s, 16 or 32 queues
# 4.75 s per step.
os.environ["GPU_MAX_HW_QUEUES"] = "16"

METRIC = "trajectories/s to tf at ≤1e-6 rel L2 err vs FP64 (batched vs plain); % HBM peak"
HBM_PEAK_GBS = 8000.0
GATE = 1e-6

FAMILIES = {  # name: (method, epsilon, tf, seed)
    "ks": ("IF34", 1e-5, 100.0, 5001),
    "nls": ("ETD35", 1e-6, 20.0, 5002),
}
KS_SIZES = (256, 512, 1024, 2048, 4096)
NLS_SIZES = (1024, 2048, 4096, 8192)

# the learned proposer's policy in the "+learned" variants: the reference controller's
# proposal, shrunk where the network predicts its rejection and grown ahead of it on a
# geometric grid of ratio 2^(1/8) where the network predicts a larger accepted step; the
# network runs after every (16 x 512 / T)-th accepted step (T: the workgroup size; a
# batch-1 inference costs ~0.1 ms beside the streaming stages, every 4th accept cost more
# than the steps it saved)
PROPOSER = {"policy": "grow", "margin": 0.02, "keep": (0.0, float(np.log(2.0) / 8.0)), "period": 16}

# precision id, state element bytes, NL element bytes
MODES = {"f64": ("F64", 16, 16), "mixed": ("MIXED", 16, 8), "f32": ("F32", 8, 8)}

# ---------------------------------------------------------------------------
# byte model: algorithmic HBM bytes of one attempt (the stage formulas' reads of u
# and NL arrays, writes of NL arrays and the candidate, one lin_op read per stage;
# FFT work stays in LDS, coefficient arrays are not credited)
# ---------------------------------------------------------------------------
# method: (u reads, NL reads, NL writes, candidate writes, stages, NL1 = nl(u) after an accept)
COUNTS = {
    "ETD35": (6, 19, 5, 1, 6, True),   # etd35.py:320-344
    "IF34": (4, 7, 4, 1, 4, False),    # if34.py:120-130
}


def attempt_bytes(method, m, e_u, e_nl, e_L=8):
    u_r, nl_r, nl_w, c_w, s, _ = COUNTS[method]
    return m * ((u_r + c_w) * e_u + (nl_r + nl_w) * e_nl + s * e_L)


def accept_bytes(method, m, e_u, e_nl):
    return m * (e_u + e_nl) if COUNTS[method][5] else 0


def alg_bytes(method, modes, stats, mode):
    _, e_u, e_nl = MODES[mode]
    return sum(s["attempts"] * attempt_bytes(method, m, e_u, e_nl) + s["steps"] * accept_bytes(method, m, e_u, e_nl)
               for s, m in zip(stats, modes))


# HBM bytes per attempt of the n = 8192 NLS ETD35 bucket (the roofline launch) measured
# with rocprofv3 FETCH_SIZE / WRITE_SIZE, each scaled by the counter's reading of a 1 GiB
# device copy in the same run; per mode
TRAFFIC_PER_ATTEMPT_N8192 = {"f64": 6.785e6, "mixed": 4.719e6, "f32": 3.062e6}


def progress(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def sig(v, n=4):
    return float(f"{v:.{n}g}") if isinstance(v, (float, np.floating)) else v


def summarize(d):
    if isinstance(d, dict):
        return {k: summarize(v) for k, v in d.items()}
    if isinstance(d, (list, tuple)):
        return [summarize(v) for v in d]
    return sig(d)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def family_inputs(name, count, seed=None):
    from rkstiff_amd.workloads import ks_ensemble, nls_ensemble
    gen = ks_ensemble if name == "ks" else nls_ensemble
    return gen(count, FAMILIES[name][3] if seed is None else seed)


def nls_two_soliton(n=8192):
    dx = 128.0 / n
    x = np.arange(-64.0, 64.0, dx)
    kx = 2 * np.pi * np.fft.fftfreq(n, d=dx)
    u0 = 2.0 / np.cosh(2.0 * (x + 10.0)) * np.exp(1j * x) + 1.5 / np.cosh(1.5 * (x - 10.0)) * np.exp(-0.5j * x)
    return kx, -0.5j * kx**2, np.fft.fft(u0)


def ks_readme(n=1024):
    dx = 32 * np.pi / n
    x = np.arange(0.0, 32 * np.pi, dx)
    kx = 2 * np.pi * np.fft.rfftfreq(n, d=dx)
    return kx, kx**2 * (1 - kx**2), np.fft.rfft(np.cos(x / 16) * (1 + np.sin(x / 16)))


# ---------------------------------------------------------------------------
# GPU plans
# ---------------------------------------------------------------------------
class FamilyRun:
    """One family's trajectories in one plan (one precision mode, optional proposer)."""

    def __init__(self, name, ens, mode, safety=0.8, net=None, tune=True, only_n=None, spec=None):
        import torch
        from rkstiff_amd import _lib
        from rkstiff_amd.autotune import tune_launch
        from rkstiff_amd.config import SolverConfig
        from rkstiff_amd.engine import Plan
        self.name, self.mode = name, mode
        self.method, eps, self.tf, _ = FAMILIES[name] if spec is None else spec
        if only_n is not None:
            ens = [e for e in ens if e[0] == only_n]
        self.ens = ens
        descs = [nl.descriptor(torch.as_tensor(L)) for (_, _, L, nl, _) in ens]
        self.plan = Plan(self.method, ens[0][3], getattr(_lib, MODES[mode][0]), SolverConfig(epsilon=eps, safety_f=safety),
                         None, descs)
        if net is not None:
            self.plan.set_proposer(net, margin=PROPOSER["margin"], keep=PROPOSER["keep"], policy=PROPOSER["policy"],
                                   period=PROPOSER["period"])
        dt = self.plan.dtype
        self.u0 = [torch.as_tensor(e[4]).to(dt).cuda() for e in ens]
        self.uf = [torch.empty_like(u) for u in self.u0]
        n = len(ens)
        self.t0s, self.tfs, self.hs = [0.0] * n, [self.tf] * n, [self.tf / 100.0] * n
        self.tuned = tune_launch(self.plan, self.u0, 0.0, self.tf / 20.0, self.tf / 2000.0) if tune else None

    def launch(self):
        self.plan.evolve(self.u0, self.uf, self.t0s, self.tfs, self.hs)

    def stats(self):
        return self.plan.stats()

    def alg_bytes(self):
        return alg_bytes(self.method, self.plan.modes, self.stats(), self.mode)

    def launch_shape(self):
        la = self.plan.launch
        if self.tuned is None or la is None:
            return None
        return {"concurrent_buckets": la["concurrent"], "wg_per_cu": la["wg_per_cu"], "fft_tile": self.plan.tiles()}


def tune_batch(runs, streams, whole=False):
    """The FFT tiles of the families' plans chosen on joint launches, each family on its
    stream as in the timed launches (after each plan's own tuning): pilots to tf/20, or
    (whole) single launches over the whole interval, the launches that decide which
    bucket ends last."""
    from rkstiff_amd.autotune import tune_together
    if whole:
        return tune_together([(r.plan, r.u0, 0.0, r.tf, r.tf / 100.0, s) for r, s in zip(runs, streams)],
                             reps=1, warm=False, uniform=True)
    return tune_together([(r.plan, r.u0, 0.0, r.tf / 20.0, r.tf / 2000.0, s) for r, s in zip(runs, streams)])


def run_together(runs, streams):
    """Launch every family's plan on its own stream; wall time until all are done."""
    import torch
    torch.cuda.synchronize()
    t = time.perf_counter()
    for r, s in zip(runs, streams):
        with torch.cuda.stream(s):
            r.launch()
    torch.cuda.synchronize()
    return time.perf_counter() - t


def rel_errors(a, ref):
    import torch
    return np.array([float(torch.linalg.norm(x.to(torch.complex128) - r) / torch.linalg.norm(r)) for x, r in zip(a, ref)])


def err_summary(e):
    return {"max": float(e.max()), "median": float(np.median(e))}


# ---------------------------------------------------------------------------
# learned proposer: records from the solver's own runs, trained on the device
# ---------------------------------------------------------------------------
def train_proposer(records, steps):
    import torch
    from rkstiff_amd.batch import BatchSolver
    from rkstiff_amd.config import SolverConfig
    from rkstiff_amd.learned import DtProposer, training_set
    datas = []
    for name, (method, eps, tf, seed) in FAMILIES.items():
        ens = family_inputs(name, 48 if name == "ks" else 96, seed + 100)
        s = BatchSolver(method, [(torch.as_tensor(L), nl) for (_, _, L, nl, _) in ens], precision="f32",
                        config=SolverConfig(epsilon=eps))
        s.record(6000)
        s.evolve([torch.as_tensor(e[4]).to(s.dtype).cuda() for e in ens], 0.0, tf)
        datas.append(training_set(*s.records(), s.plan.cfg))
        progress(f"proposer: {name} training records {datas[-1].shape[0]}")
    data = torch.cat(datas)
    g = torch.Generator().manual_seed(0)
    data = data[torch.randperm(data.shape[0], generator=g)[:records].to(data.device)].contiguous()
    net = DtProposer.for_data(data, seed=0)
    torch.cuda.synchronize()
    t = time.perf_counter()
    hist = net.train(data, steps=steps, batch=1024, lr=1e-3, loss="pinball", tau=0.2)
    torch.cuda.synchronize()
    sec = time.perf_counter() - t
    macs = 96 * 256 + 2 * 256 * 256 + 256
    tflops = 3 * 2 * 1024 * macs * steps / sec / 1e12
    info = {"records": int(data.shape[0]), "steps": steps, "batch": 1024, "loss": "pinball tau 0.2",
            "loss_first": float(hist[:10].mean()), "loss_last": float(hist[-50:].mean()), "seconds": sec,
            "mfma": {"achieved": tflops, "peak": 2500.0, "unit": "TFLOP/s", "frac": tflops / 2500.0,
                     "what": "BF16 GEMMs of training incl. launch gaps (wall)"}}
    return net, info


# ---------------------------------------------------------------------------
# plain FP64 drop-in (the reference's API, one trajectory at a time)
# ---------------------------------------------------------------------------
def plain_seconds(name, e):
    """Seconds of one drop-in evolve t0 -> tf of trajectory e (FP64 state on the GPU)."""
    import torch
    import rkstiff_amd
    from rkstiff_amd.config import SolverConfig
    method, eps, tf, _ = FAMILIES[name]
    n, kx, L, nl, u0 = e
    solver = getattr(rkstiff_amd, method)(torch.as_tensor(L), nl, config=SolverConfig(epsilon=eps))
    u = torch.as_tensor(u0, dtype=torch.complex128).cuda()
    solver.evolve(u, 0.0, tf / 50.0, store_data=False)  # builds the plan
    torch.cuda.synchronize()
    t = time.perf_counter()
    solver.evolve(u, 0.0, tf, store_data=False)
    torch.cuda.synchronize()
    return time.perf_counter() - t


def plain_batch_rate(ens_by_fam):
    """Drop-in trajectories/s over the batch: one sampled trajectory per (family, n), each
    size's time weighted by how many trajectories of that size the batch holds."""
    total_t, total_n, per = 0.0, 0, {}
    for name, ens in ens_by_fam.items():
        sizes = sorted({e[0] for e in ens})
        for n in sizes:
            e = next(x for x in ens if x[0] == n)
            sec = plain_seconds(name, e)
            cnt = sum(1 for x in ens if x[0] == n)
            per[f"{name}_n{n}"] = {"s_per_trajectory": sec, "count_in_batch": cnt}
            total_t += sec * cnt
            total_n += cnt
    return total_n / total_t, per


# ---------------------------------------------------------------------------
# CPU baseline: the NumPy FP64 oracle (test infrastructure) on host cores
# ---------------------------------------------------------------------------
def _cpu_one(args):
    name, seed, idx = args
    os.environ.setdefault("OMP_NUM_THREADS", "1")
    from oracle import problems, solvers
    method, eps, tf, _ = FAMILIES[name]
    ens = family_inputs(name, idx + 1, seed)
    n, kx, L, _nl, u0 = ens[idx]
    nl = problems.rfft_advect_nl(kx, -1.0) if name == "ks" else problems.nls_nl(1.0)
    drv = solvers.make_solver(method, L, nl, solvers.SolverConfig(epsilon=eps))
    t0 = time.perf_counter()
    drv.evolve(u0, t0=0.0, tf=tf, store_data=False)
    return name, n, time.perf_counter() - t0


def _cpu_single(args):
    which = args
    os.environ.setdefault("OMP_NUM_THREADS", "1")
    from oracle import problems, solvers
    if which == "ks1024":
        kx, L, u0 = ks_readme()
        drv = solvers.make_solver("IF34", L, problems.rfft_advect_nl(kx, -1.0), solvers.SolverConfig(epsilon=1e-4))
        tf = 50.0
    else:
        kx, L, u0 = nls_two_soliton()
        drv = solvers.make_solver("ETD35", L, problems.nls_nl(1.0), solvers.SolverConfig(epsilon=1e-6))
        tf = 20.0
    t0 = time.perf_counter()
    drv.evolve(u0, t0=0.0, tf=tf, store_data=False)
    return time.perf_counter() - t0


def host_cores():
    try:
        avail = len(os.sched_getaffinity(0))
    except AttributeError:
        avail = os.cpu_count() or 1
    # the GPU box gives one GPU's job 16 host cores, whatever the machine has
    return min(avail, 16), avail


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def cpu_baseline(ens_by_fam, per_size):
    for k in ("OMP_NUM_THREADS", "OPENBLAS_NUM_THREADS", "MKL_NUM_THREADS"):
        os.environ[k] = "1"
    workers, avail = host_cores()
    tasks = []
    for name, ens in ens_by_fam.items():
        seed = FAMILIES[name][3]
        for n in sorted({e[0] for e in ens}):
            idxs = [i for i, e in enumerate(ens) if e[0] == n][:per_size]
            tasks += [(name, seed, i) for i in idxs]
    ctx = mp.get_context("spawn")
    with ctx.Pool(workers) as pool:
        t0 = time.perf_counter()
        res = pool.map(_cpu_one, tasks, chunksize=1)
        wall = time.perf_counter() - t0
    per = {}
    for name, n, sec in res:
        per.setdefault(f"{name}_n{n}", []).append(sec)
    return {"value": len(tasks) / wall, "unit": "trajectories/s", "cores": workers, "kind": "port",
            "sample": f"{len(tasks)} trajectories of the mixed batch ({per_size} per family and grid size, the "
                      f"batch's size mix), one per core on {workers} of {avail} available cores "
                      f"(os.cpu_count() {os.cpu_count()}), NumPy FP64 oracle, wall {wall:.1f} s",
            "cpu_model": cpu_model(), "numpy": np.__version__,
            "single_core_s_per_trajectory": {k: float(np.median(v)) for k, v in per.items()}}


# ---------------------------------------------------------------------------
# the headline: variants, gate, timed steps, roofline
# ---------------------------------------------------------------------------
def variant_parts(v):
    mode, _, extra = v.partition("+")
    return mode, extra == "learned"


def headline(args, ens_by_fam, net):
    import torch
    streams = [torch.cuda.Stream() for _ in FAMILIES]
    n_all = sum(len(e) for e in ens_by_fam.values())
    out = {"variants": {}}
    progress("f64 reference and step-sequence floor")
    ref = {name: FamilyRun(name, ens, "f64") for name, ens in ens_by_fam.items()}
    tune_batch(list(ref.values()), streams)
    wall = run_together(list(ref.values()), streams)
    out["variants"]["f64"] = {"traj_per_s": n_all / wall, "seconds": wall}
    ref_u = {k: [u.clone() for u in r.uf] for k, r in ref.items()}
    launch = {"f64": {k: r.launch_shape() for k, r in ref.items()}}
    ok = {"f64": all(s["status"] == 0 for r in ref.values() for s in r.stats())}
    counts = {"f64": {k: _counts(r.stats()) for k, r in ref.items()}}
    del ref
    floors = {}
    fl = {name: FamilyRun(name, ens, "f64", safety=0.79, tune=False) for name, ens in ens_by_fam.items()}
    run_together(list(fl.values()), streams)
    for k, r in fl.items():
        floors[k] = err_summary(rel_errors(r.uf, ref_u[k]))
    del fl
    out["f64_step_sequence_floor"] = {**floors, "what": "FP64 with safety_f 0.79 vs 0.8"}
    errs = {"f64": {k: {"max": 0.0, "median": 0.0} for k in FAMILIES}}
    for v in args.variants:
        if v == "f64":
            continue
        mode, learned = variant_parts(v)
        if learned and net is None:
            continue
        progress(f"variant {v}")
        runs = {name: FamilyRun(name, ens, mode, net=net if learned else None) for name, ens in ens_by_fam.items()}
        tune_batch(list(runs.values()), streams)
        wall = run_together(list(runs.values()), streams)
        out["variants"][v] = {"traj_per_s": n_all / wall, "seconds": wall}
        errs[v] = {k: err_summary(rel_errors(r.uf, ref_u[k])) for k, r in runs.items()}
        ok[v] = all(s["status"] == 0 for r in runs.values() for s in r.stats())
        launch[v] = {k: r.launch_shape() for k, r in runs.items()}
        counts[v] = {k: _counts(r.stats()) for k, r in runs.items()}
        progress(f"variant {v}: {n_all / wall:.1f} trajectories/s")
        del runs
    passes = {}
    for v, e in errs.items():
        fam_ok = {}
        for k in FAMILIES:
            fam_ok[k] = (e[k]["max"] <= max(GATE, floors[k]["max"]) and e[k]["median"] <= max(GATE, floors[k]["median"]))
        passes[v] = ok[v] and all(fam_ok.values())
        out["variants"][v].update({"rel_l2_vs_fp64": e, "passes_gate": passes[v], "all_ok": ok[v],
                                   "launch": launch[v], "counts": counts[v]})
    eligible = [v for v in out["variants"] if passes.get(v)]
    best = max(eligible, key=lambda v: out["variants"][v]["traj_per_s"])
    out["headline_variant"] = best
    # timed region: W warm-up steps, then K steps of the headline variant
    mode, learned = variant_parts(best)
    progress(f"timed steps of {best}")
    runs = {name: FamilyRun(name, ens, mode, net=net if learned else None) for name, ens in ens_by_fam.items()}
    rl = list(runs.values())
    joint = tune_batch(rl, streams, whole=True)
    progress(f"timed variant: tiles {joint['tiles']} from {len(joint['trials'])} whole-interval trials")
    for _ in range(args.warmup):
        run_together(rl, streams)
    torch.cuda.synchronize()
    walls = []
    for i in range(args.steps):
        walls.append(run_together(rl, streams))
        if (i + 1) % 5 == 0:
            progress(f"timed step {i + 1}/{args.steps}: {walls[-1]:.3f} s")
    out["timed"] = {"walls_s": walls, "value": n_all * len(walls) / sum(walls), "ms_per_step": 1e3 * sum(walls) / len(walls)}
    out["timed"]["whole_batch_alg_GBs"] = sum(r.alg_bytes() for r in rl) / (sum(walls) / len(walls)) / 1e9
    out["timed"]["counts"] = {k: _counts(r.stats()) for k, r in runs.items()}
    del runs, rl
    return out, best


def _counts(st):
    out = {k: int(sum(x[k] for x in st)) for k in ("attempts", "rejects", "steps", "coef_updates")}
    a = np.array([x["attempts"] for x in st], dtype=np.float64)
    out["attempts_per_trajectory"] = {"median": float(np.median(a)), "p99": float(np.percentile(a, 99)),
                                      "max": float(a.max())}
    return out


def roofline(ens_by_fam, variant, net, reps=3):
    """The headline variant's n = 8192 NLS bucket alone: one kernel launch per evolve, timed
    with HIP events on the stream it is launched on."""
    import torch
    mode, learned = variant_parts(variant)
    progress(f"roofline: n = 8192 bucket of the nls family, {variant}")
    r = FamilyRun("nls", ens_by_fam["nls"], mode, net=net if learned else None, only_n=8192)
    progress("roofline: tuned")
    stream = torch.cuda.current_stream()
    r.launch()  # warm
    torch.cuda.synchronize()
    ms = []
    for i in range(reps):
        progress(f"roofline: launch {i + 1}/{reps}")
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        r.launch()
        e1.record(stream)
        e1.synchronize()
        ms.append(e0.elapsed_time(e1))
    st = r.stats()
    att = sum(s["attempts"] for s in st)
    alg = r.alg_bytes()
    k_ms = float(np.mean(ms))
    ach = alg / (k_ms * 1e-3) / 1e9
    traffic = TRAFFIC_PER_ATTEMPT_N8192.get(mode)
    longest = max(s["attempts"] for s in st)
    return {"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(ach / HBM_PEAK_GBS, 4), "traffic": None if traffic is None else sig(traffic * att),
            "kernel": f"rks_kernel n=8192 cubic ETD35 ({mode}{', proposer' if learned else ''})",
            "trajectories": len(r.ens), "attempts": att, "alg_bytes_per_launch": alg, "kernel_ms": k_ms,
            # the launch ends with its longest trajectory (started first): its attempts
            # and the launch time per attempt of it
            "longest_trajectory_attempts": longest, "ms_per_attempt_of_longest": k_ms / longest}


# ---------------------------------------------------------------------------
# single-instance workloads and the other batches
# ---------------------------------------------------------------------------
def single_workloads():
    import torch
    import rkstiff_amd
    from rkstiff_amd.batch import BatchSolver
    from rkstiff_amd.config import SolverConfig
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    out = {}
    kx, L, u0 = ks_readme()
    s = rkstiff_amd.IF34(torch.as_tensor(L), AdvectiveNL(torch.as_tensor(kx), -1.0), config=SolverConfig(epsilon=1e-4))
    u = torch.as_tensor(u0).cuda()
    s.evolve(u, 0.0, 1.0, store_data=False)
    torch.cuda.synchronize()
    t = time.perf_counter()
    s.evolve(u, 0.0, 50.0, store_freq=20)
    torch.cuda.synchronize()
    out["ks1024_if34_tf50"] = {"gpu_dropin_fp64_s": time.perf_counter() - t, "snapshots": len(s.t)}
    kx, L, u0 = nls_two_soliton()
    res = {}
    for prec, dt in (("f64", torch.complex128), ("f32", torch.complex64)):
        s = rkstiff_amd.ETD35(torch.as_tensor(L), CubicNL(8192, 1.0), config=SolverConfig(epsilon=1e-6))
        u = torch.as_tensor(u0).to(dt).cuda()
        s.evolve(u, 0.0, 0.5, store_data=False)
        torch.cuda.synchronize()
        t = time.perf_counter()
        res[prec] = s.evolve(u, 0.0, 20.0, store_data=False)
        torch.cuda.synchronize()
        out.setdefault("nls8192_etd35_tf20", {})[f"gpu_dropin_{prec}_s"] = time.perf_counter() - t
    bs = BatchSolver("ETD35", [(torch.as_tensor(L), CubicNL(8192, 1.0))], precision="mixed",
                     config=SolverConfig(epsilon=1e-6))
    um = torch.as_tensor(u0).cuda()
    bs.evolve([um], 0.0, 0.5)
    torch.cuda.synchronize()
    t = time.perf_counter()
    res["mixed"] = bs.evolve([um], 0.0, 20.0)[0]
    torch.cuda.synchronize()
    o = out["nls8192_etd35_tf20"]
    o["gpu_batch1_mixed_s"] = time.perf_counter() - t
    o["rel_l2_vs_fp64"] = {k: float(rel_errors([res[k]], [res["f64"]])[0]) for k in ("f32", "mixed")}
    return out


def ks_workload(count):
    import torch
    from rkstiff_amd.workloads import ks_ensemble
    ens = ks_ensemble(count, 2024)
    out = {}
    for method in ("IF34", "ETD35"):
        res, fin = {}, {}
        for mode in ("f64", "mixed", "f32"):
            r = FamilyRun("ks_ensemble", ens, mode, spec=(method, 1e-5, 100.0, 2024))
            tune_batch([r], [torch.cuda.current_stream()])
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            r.launch()
            e1.record()
            e1.synchronize()
            sec = e0.elapsed_time(e1) * 1e-3
            res[mode] = {"traj_per_s": count / sec, "alg_GBs": r.alg_bytes() / sec / 1e9, "launch": r.launch_shape(),
                         "attempts_mean": float(np.mean([s["attempts"] for s in r.stats()]))}
            fin[mode] = [u.clone() for u in r.uf]
            del r
            progress(f"ks ensemble {method} {mode}: {count / sec:.1f} trajectories/s")
        for mode in ("mixed", "f32"):
            res[mode]["rel_l2_vs_fp64"] = err_summary(rel_errors(fin[mode], fin["f64"]))
        out[method] = res
    return {"count": count, "sizes": list(KS_SIZES), "tf": 100.0, "epsilon": 1e-5, "unit": "trajectories/s",
            "results": out}


def ac_workload(batch):
    import torch
    from rkstiff_amd.batch import BatchSolver
    from rkstiff_amd.config import SolverConfig
    from rkstiff_amd.nonlinear import allen_cahn_ops
    n = 512
    rng = np.random.default_rng(7)
    ky = np.fft.fftfreq(n, d=1.0 / n)
    kxr = np.fft.rfftfreq(n, d=1.0 / n)
    mask = np.sqrt(kxr[None, :] ** 2 + ky[:, None] ** 2) > 32.0
    u0s = []
    for _ in range(batch):
        uh = np.fft.rfft2(rng.uniform(-0.05, 0.05, (n, n)))
        uh[mask] = 0.0
        u0s.append(uh.reshape(-1))
    L, nl = allen_cahn_ops(n)
    res, fin = {}, {}
    for mode in ("f64", "mixed", "f32"):
        bs = BatchSolver("ETD35", [(L, nl)] * batch, precision=mode, config=SolverConfig(epsilon=1e-5))
        u0 = [torch.as_tensor(u).to(bs.dtype).cuda() for u in u0s]
        bs.autotune(u0, 0.0, 0.5)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        fin[mode] = bs.evolve(u0, 0.0, 10.0, sync=False)
        e1.record()
        e1.synchronize()
        sec = e0.elapsed_time(e1) * 1e-3
        st = bs.stats()
        _, e_u, e_nl = MODES[mode]
        alg = sum(s["attempts"] * attempt_bytes("ETD35", m, e_u, e_nl, e_L=4 if mode == "f32" else 8)
                  + s["steps"] * accept_bytes("ETD35", m, e_u, e_nl) for s, m in zip(st, bs.modes))
        res[mode] = {"traj_per_s": batch / sec, "alg_GBs": alg / sec / 1e9,
                     "attempts_mean": float(np.mean([s["attempts"] for s in st]))}
        progress(f"allen-cahn 2-D {mode}: {batch / sec:.1f} trajectories/s")
    for mode in ("mixed", "f32"):
        res[mode]["rel_l2_vs_fp64"] = err_summary(rel_errors(fin[mode], fin["f64"]))
    return {"count": batch, "grid": [n, n], "method": "ETD35", "tf": 10.0, "epsilon": 1e-5,
            "unit": "trajectories/s", "launches": "hipGraph-replayed attempt sequence", "results": res}


def radial_workload(count):
    """Radial NLS (demos/nls.ipynb cells 6-12: i u_t = -(1/2) lap u - gamma |u|^2 u in the
    order-zero Hankel domain, nr = 100 on [0, 5]): ``count`` Gaussian beams around the
    demo's (amplitude U[1.8, 2.0], width U[0.9, 1.1], gamma 2: self-focusing, ~100-200
    attempts each), ETD35, eps 1e-5, tf 0.8, batched on the
    stepping kernel (FP64 and MIXED) against the plain per-instance FP64 drop-in on a
    sample of 8."""
    import torch
    import rkstiff_amd
    from rkstiff_amd.batch import BatchSolver
    from rkstiff_amd.config import SolverConfig
    from rkstiff_amd.transforms import HankelTransform
    ht = HankelTransform(nr=100, rmax=5.0)
    r = ht.r.cpu().numpy()
    rng = np.random.default_rng(11)
    u0s = []
    for _ in range(count):
        a, w = rng.uniform(1.8, 2.0), rng.uniform(0.9, 1.1)
        u0s.append(ht.ht(torch.as_tensor(a * np.exp(-(r / w) ** 2) + 0j).cuda()))
    L, nl, tf = -1j * ht.kr**2, ht.cubic_nl(2.0), 0.8
    res, fin = {}, {}
    for mode in ("f64", "mixed"):
        bs = BatchSolver("ETD35", [(L, nl)] * count, precision=mode, config=SolverConfig(epsilon=1e-5))
        u0 = [u.to(bs.dtype) for u in u0s]
        bs.evolve(u0, 0.0, tf / 10)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        fin[mode] = bs.evolve(u0, 0.0, tf, sync=False)
        e1.record()
        e1.synchronize()
        sec = e0.elapsed_time(e1) * 1e-3
        res[mode] = {"traj_per_s": count / sec,
                     "attempts_mean": float(np.mean([s["attempts"] for s in bs.stats()]))}
        progress(f"radial NLS {mode}: {count / sec:.1f} trajectories/s")
    res["mixed"]["rel_l2_vs_fp64"] = err_summary(rel_errors(fin["mixed"], fin["f64"]))
    solver = rkstiff_amd.ETD35(L, nl, config=SolverConfig(epsilon=1e-5))
    solver.evolve(u0s[0], 0.0, tf / 10, store_data=False)
    torch.cuda.synchronize()
    t = time.perf_counter()
    for u in u0s[:8]:
        solver.evolve(u, 0.0, tf, store_data=False)
    torch.cuda.synchronize()
    plain = 8 / (time.perf_counter() - t)
    return {"count": count, "nr": 100, "rmax": 5.0, "method": "ETD35", "tf": tf, "epsilon": 1e-5,
            "unit": "trajectories/s", "results": res, "plain_fp64_dropin": plain,
            "batched_f64_over_plain": res["f64"]["traj_per_s"] / plain}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--count", type=int, default=4096, help="trajectories per family")
    ap.add_argument("--variants", default="f64,mixed,f32,f32+learned")
    ap.add_argument("--workloads", default="single,ks,ac2d,radial")
    ap.add_argument("--ks-count", type=int, default=4096)
    ap.add_argument("--ac-batch", type=int, default=64)
    ap.add_argument("--records", type=int, default=200000)
    ap.add_argument("--train-steps", type=int, default=2000)
    ap.add_argument("--proposer-period", type=int, default=PROPOSER["period"],
                    help="the network runs after every (period x 512 / T)-th accepted step")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-per-size", type=int, default=3)
    ap.add_argument("--only", default="", help="'roofline': only the dominant kernel pass; 'batch': only the "
                                               "mixed batch in --variant; 'ks' / 'ac2d': only that workload (profiling)")
    ap.add_argument("--roofline-variant", "--variant", dest="roofline_variant", default="f64")
    ap.add_argument("--copy-mib", type=int, default=0, help="device copy of this size first (counter scale)")
    args = ap.parse_args()
    PROPOSER["period"] = args.proposer_period
    if args.gpus != 1:
        print(json.dumps({"error": "this build measures one GPU; trajectories are independent, "
                                   "so N GPUs would each run their own share of them"}))
        sys.exit(2)
    args.variants = [v for v in args.variants.split(",") if v]
    if "f64" not in args.variants:
        args.variants.insert(0, "f64")

    import logging
    import torch
    # the autotuner's pilot evolves report on stderr (progress of long profiled runs)
    logging.basicConfig(level=logging.WARNING, stream=sys.stderr, format="[bench] %(message)s")
    logging.getLogger("rkstiff_amd.autotune").setLevel(logging.INFO)
    torch.cuda.init()
    if args.copy_mib > 0:
        src = torch.empty(args.copy_mib * 2**18, dtype=torch.float32, device="cuda").fill_(1.0)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": src.numel() * 4, "copy_bytes_written": dst.numel() * 4}), flush=True)
        del src, dst

    ens_by_fam = {name: family_inputs(name, args.count) for name in FAMILIES}
    need_net = (variant_parts(args.roofline_variant)[1] if args.only in ("roofline", "batch")
                else any(variant_parts(v)[1] for v in args.variants))
    net, train_info = (None, None)
    if args.only == "roofline":
        if need_net:
            net, train_info = train_proposer(args.records, args.train_steps)
        rf = roofline(ens_by_fam, args.roofline_variant, net)
        print(json.dumps({"roofline": rf}), flush=True)
        return
    if args.only == "batch":  # the mixed batch in one variant, tuned, launched --steps times (profiling)
        if need_net:
            net, train_info = train_proposer(args.records, args.train_steps)
        streams = [torch.cuda.Stream() for _ in FAMILIES]
        runs = [FamilyRun(name, ens, variant_parts(args.roofline_variant)[0],
                          net=net if variant_parts(args.roofline_variant)[1] else None)
                for name, ens in ens_by_fam.items()]
        joint = tune_batch(runs, streams, whole=True)
        progress(f"joint tiles {joint['tiles']} from {len(joint['trials'])} whole-interval trials")
        for tr in joint["trials"]:
            progress(f"  trial {tr['tiles']}: {tr['seconds']:.3f} s")
        walls = []
        for i in range(args.steps):
            walls.append(run_together(runs, streams))
            progress(f"batch launch {i + 1}/{args.steps}: {walls[-1]:.3f} s")
        per_n = {}
        for r in runs:
            st = r.stats()
            for n in sorted(set(r.plan.modes)):
                sel = [(x, m) for x, m in zip(st, r.plan.modes) if m == n]
                per_n[f"{r.name}_m{n}"] = {"trajectories": len(sel), "attempts": sum(x["attempts"] for x, _ in sel),
                                           "alg_bytes": alg_bytes(r.method, [m for _, m in sel], [x for x, _ in sel],
                                                                  r.mode)}
        print(json.dumps({"batch": args.roofline_variant, "walls_s": walls,
                          "launch": {r.name: r.launch_shape() for r in runs},
                          "counts": {r.name: _counts(r.stats()) for r in runs}, "per_bucket": per_n}), flush=True)
        return
    if args.only in ("ks", "ac2d", "radial"):  # one secondary workload alone (profiling)
        out = (ks_workload(args.ks_count) if args.only == "ks" else
               ac_workload(args.ac_batch) if args.only == "ac2d" else radial_workload(2048))
        print(json.dumps(summarize(out)), flush=True)
        return
    if need_net:
        net, train_info = train_proposer(args.records, args.train_steps)
    res, best = headline(args, ens_by_fam, net)
    progress("roofline pass")
    rf = roofline(ens_by_fam, best, net)
    progress("plain FP64 drop-in sample")
    plain_rate, plain_per = plain_batch_rate(ens_by_fam)
    wl = args.workloads.split(",")
    workloads = {}
    if "single" in wl:
        progress("single-instance workloads")
        workloads["single"] = single_workloads()
    if "ks" in wl:
        workloads["ks_ensemble"] = ks_workload(args.ks_count)
    if "ac2d" in wl:
        workloads["allen_cahn_2d"] = ac_workload(args.ac_batch)
    if "radial" in wl:
        workloads["radial_nls"] = radial_workload(2048)
    mode, learned = variant_parts(best)
    value = res["timed"]["value"]
    line = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "trajectories/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(res["timed"]["ms_per_step"], 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32" if mode == "f32" else "f64",
        "data": "synthetic",
        "config": {"workload": f"mixed_batch_{args.count}ks_if34_tf100_{args.count}nls_etd35_tf20",
                   "families": {k: {"method": v[0], "epsilon": v[1], "tf": v[2],
                                    "n": list(KS_SIZES if k == "ks" else NLS_SIZES), "count": args.count}
                                for k, v in FAMILIES.items()},
                   "batch": 2 * args.count, "variant": best,
                   "precision": {"f64": "f64 throughout", "mixed": "f64 state, propagators and FFTs; "
                                 "f32 NL arrays and psi coefficients; f64 norm and dt control",
                                 "f32": "f32 stages and FFTs; f64 coefficients, norm, dt control"}[mode]
                   + ("; learned step-size proposer" if learned else ""),
                   "parallelism": "1 GPU, one workgroup per trajectory, persistent kernels, two families on two streams"},
        "roofline": rf,
        "accuracy": {"rel_l2_vs_fp64": res["variants"][best]["rel_l2_vs_fp64"],
                     "fp64_step_sequence_floor": res["f64_step_sequence_floor"], "gate": GATE,
                     "rule": "per family: max and median <= max(gate, floor max / median)"},
        "plain_fp64": {"value": plain_rate, "unit": "trajectories/s", "per_size": plain_per,
                       "what": "drop-in solver classes, FP64, one evolve per trajectory"},
        "batched_over_plain": value / plain_rate,
        "variants": res["variants"],
        "timed": res["timed"],
        "proposer_training": train_info,
        "proposer_policy": {k: (list(v) if isinstance(v, tuple) else v) for k, v in PROPOSER.items()},
        "workloads": workloads,
    }
    if not args.no_cpu:
        progress("cpu baseline")
        line["cpu_baseline"] = cpu_baseline(ens_by_fam, args.cpu_per_size)
        ctx = mp.get_context("spawn")
        with ctx.Pool(2) as pool:
            t_ks, t_nls = pool.map(_cpu_single, ["ks1024", "nls8192"])
        if "single" in workloads:
            workloads["single"]["ks1024_if34_tf50"]["cpu_oracle_1core_s"] = t_ks
            workloads["single"]["nls8192_etd35_tf20"]["cpu_oracle_1core_s"] = t_nls
    line = {k: summarize(v) if k not in ("metric", "unit", "data", "dtype", "scaling") else v for k, v in line.items()}
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
