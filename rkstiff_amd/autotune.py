"""Launch-shape autotuner for the persistent stepping kernels.

A plan groups its trajectories in size buckets, one persistent-kernel launch
per bucket.  Three launch choices change throughput, and results by rounding
at most (the tile):

* whether the buckets run one after another on the caller's stream or
  overlap on private streams.  In a mixed-size ensemble a bucket's last
  long trajectories otherwise leave most CUs idle before the next bucket
  starts;
* how many workgroups of each bucket stay resident per CU (fewer resident
  trajectories share a CU's caches and LDS bandwidth with fewer others);
* the FFT tile of each bucket where a second one exists (n = 512 .. 4096):
  twice the threads per trajectory, half the modes per thread in the stage
  passes and transforms.  A bucket starts on the tile that the library
  chooses for it (-1, ``Plan.tiles`` says which).

``tune_launch`` times short pilot evolves of the plan's own trajectories and
keeps the fastest shape.  Finally each bucket's trajectories are ordered by
the attempts they took in a pilot over the whole interval, most first, so
the longest trajectories start first and a bucket's tail stays short
(longest-processing-time-first; trajectories of one bucket differ mainly in
their step counts).  The per-bucket choices (another tile than the library's,
then half and a quarter of the resident workgroups) are timed on pilots in which only
that bucket's trajectories move (the others get tf = t0, which leaves them
untouched), so one bucket's choice is not lost in the noise of the others;
a choice that wins there is kept only if the whole ensemble, buckets
overlapping, is not slower with it.  Then concurrent (the plan default) and
sequential buckets are compared on the whole ensemble, and the tuned shape
is kept only if the whole ensemble is faster with it than with the default
shape.  A change is kept only when
it is faster by more than ``min_gain``; every timing is the fastest of
``reps`` pilots after a warm-up pilot.  The shape is applied to the plan and
returned with the timings of every trial.
"""
import itertools
import logging
import time

import numpy as np
import torch


_log = logging.getLogger("rkstiff_amd.autotune")


def _timed(plan, u0, uf, t0s, tfs, hs, reps):
    _log.info("pilot evolves of %d trajectories", plan.ninst)
    plan.evolve(u0, uf, t0s, tfs, hs)  # warm
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(max(1, reps)):
        t = time.perf_counter()
        plan.evolve(u0, uf, t0s, tfs, hs)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


def _bucket_log2(plan, n):
    """The size bucket of an instance of n points: log2 n, or for the Hankel kind the
    size class 2^l >= n, l >= 4 (rks_host.hip hankel_log2)."""
    from . import _lib
    if plan.nl_kind == _lib.NL_HANKEL_CUBIC:
        return max(4, (int(n) - 1).bit_length())
    return int(n).bit_length() - 1


def _other_tile(tile):
    """The tile tried against ``tile``: the second one, or the base tile against that."""
    return 0 if tile == 1 else 1


def tune_launch(plan, u0, t0, tf, h, reps=2, min_gain=0.02):
    """Tune ``plan``'s launch shape on pilot evolves over [t0, tf] from ``u0``.

    u0: list of device state tensors (the plan's dtype), one per trajectory;
    t0/tf/h: scalars or per-trajectory sequences (h: first step).
    Returns {"concurrent", "wg_per_cu", "tile", "seconds", "trials", "buckets"}; the first
    three are what ``Plan.set_launch`` takes (tile -1: the library's choice).
    """
    n = plan.ninst
    t0s = np.broadcast_to(np.asarray(t0, dtype=np.float64), (n,)).tolist()
    tfs = np.broadcast_to(np.asarray(tf, dtype=np.float64), (n,)).tolist()
    hs = np.broadcast_to(np.asarray(h, dtype=np.float64), (n,)).tolist()
    uf = [torch.empty_like(u) for u in u0]
    buckets = plan.buckets()
    trials = []
    if not buckets:
        # the 2-D engine: a fixed kernel sequence, nothing to choose
        sec = _timed(plan, u0, uf, t0s, tfs, hs, reps)
        return {"concurrent": None, "wg_per_cu": [], "tile": [], "seconds": sec,
                "trials": [{"concurrent": None, "wg_per_cu": [], "tile": [], "seconds": sec}], "buckets": []}
    inst_l2 = [_bucket_log2(plan, x) for x in plan.ns]

    def trial(conc, wg, ti, bucket=None):
        plan.set_launch(conc, wg, ti)
        if bucket is None:
            sec = _timed(plan, u0, uf, t0s, tfs, hs, reps)
        else:
            l2 = buckets[bucket][0]
            only = [tfs[i] if inst_l2[i] == l2 else t0s[i] for i in range(n)]
            sec = _timed(plan, u0, uf, t0s, only, hs, reps)
        trials.append({"concurrent": conc, "wg_per_cu": list(wg), "tile": list(ti), "bucket": bucket,
                       "seconds": sec})
        return sec

    nb = len(buckets)
    wg0, ti0 = [0] * nb, [-1] * nb
    default = trial(True, wg0, ti0)  # the plan's default shape
    own = plan.tiles()
    best_wg, best_ti, whole = list(wg0), list(ti0), default

    def consider(b, base, wg, ti):
        """Keep (wg, ti) if bucket b alone gains min_gain and the whole ensemble is not slower."""
        nonlocal whole
        sec = trial(True, wg, ti, b if nb > 1 else None)
        if not sec < base * (1.0 - min_gain):
            return None
        if nb > 1:
            w = trial(True, wg, ti)
            if w > whole:
                return None
            whole = w
        else:
            whole = sec
        return sec

    for b, (_l2, _cnt, _mx, ntile) in enumerate(buckets):
        # this bucket alone: tile, then the resident-workgroup limit of the chosen tile
        base = trial(True, best_wg, best_ti, b) if nb > 1 else default
        if ntile > 1:
            ti = list(best_ti)
            ti[b] = _other_tile(own[b])
            sec = consider(b, base, best_wg, ti)
            if sec is not None:
                base, best_ti = sec, ti
        plan.set_launch(True, best_wg, best_ti)
        if plan.tiles()[b] == 0:
            mx = plan.buckets()[b][2]
            for v in sorted({mx // 2, mx // 4} - {0, mx}, reverse=True):
                wg = list(best_wg)
                wg[b] = v
                sec = consider(b, base, wg, best_ti)
                if sec is not None:
                    base, best_wg = sec, wg
    best_conc, best = True, whole
    if nb > 1:
        sec = trial(False, best_wg, best_ti)
        if sec < best * (1.0 - min_gain):
            best, best_conc = sec, False
        if not best < default:
            best, best_conc, best_wg, best_ti = default, True, list(wg0), list(ti0)
    plan.set_launch(best_conc, best_wg, best_ti)
    # longest first: the attempts of a pilot over the whole ensemble estimate each
    # trajectory's cost
    plan.evolve(u0, uf, t0s, tfs, hs)
    attempts = [s["attempts"] for s in plan.stats()]
    plan.set_priority(attempts)
    return {"concurrent": best_conc, "wg_per_cu": best_wg, "tile": best_ti, "seconds": best, "trials": trials,
            "buckets": [{"log2n": l2, "count": c, "max_wg_per_cu": m, "tiles": t} for l2, c, m, t in buckets]}


def _timed_together(jobs, reps, warm=True):
    """Fastest of ``reps`` of every job's evolve launched together, each plan on its own
    stream (after a warm-up launch when ``warm``)."""
    def run():
        torch.cuda.synchronize()
        t = time.perf_counter()
        for plan, u0, uf, t0s, tfs, hs, stream in jobs:
            with torch.cuda.stream(stream):
                plan.evolve(u0, uf, t0s, tfs, hs)
        torch.cuda.synchronize()
        return time.perf_counter() - t
    _log.info("joint evolves of %d plans", len(jobs))
    if warm:
        run()
    return min(run() for _ in range(max(1, reps)))


def tune_together(jobs, reps=2, min_gain=0.02, warm=True, uniform=False):
    """Tune the FFT tiles of several plans that run at the same time.

    jobs: list of (plan, u0, t0, tf, h, stream): each plan's trial interval and first step
    (scalars or per-trajectory sequences) and the stream it is launched on.  Call after
    ``tune_launch`` on each plan.  A bucket's best tile alone is not its best tile beside
    other plans' buckets: the overlapped launch ends with its longest bucket, whose
    trajectories may gain more from twice the threads each (shorter attempts) than from
    more of them resident.  Which bucket ends last depends on the whole interval, so the
    trials may be whole evolves (then ``warm=False, reps=1``: every trial is one launch of
    all plans).  The buckets with a second tile are flipped in turn, largest (trajectories
    x n) first over all plans, and a flip is kept when the joint launch is faster by more
    than ``min_gain``.  With ``uniform`` the flips start from the best combination of
    each plan's own tuning, the library's own choice, the second tile on every bucket that has
    one, and the first tile everywhere (single flips miss combinations that only pay together: on the
    mixed batch the KS family's second tiles gain most when the NLS family's buckets
    keep the first).  Resident-workgroup
    limits, bucket concurrency and trajectory order stay as tuned.  Returns {"tiles":
    per-plan tiles as ``Plan.set_launch`` takes them, "seconds": the best joint launch, "trials": [...]}.
    """
    runs = []
    for plan, u0, t0, tf, h, stream in jobs:
        n = plan.ninst
        bc = lambda v: np.broadcast_to(np.asarray(v, dtype=np.float64), (n,)).tolist()
        runs.append((plan, u0, [torch.empty_like(u) for u in u0], bc(t0), bc(tf), bc(h), stream))
    shapes = []
    for plan, *_ in runs:
        nb = len(plan.buckets())
        la = plan.launch or {}
        shapes.append({"concurrent": la.get("concurrent", True),
                       "wg": list(la.get("wg_per_cu") or [0] * nb),
                       "tile": list(la.get("tile") or [-1] * nb)})

    def apply():
        for (plan, *_), sh in zip(runs, shapes):
            if plan.buckets():
                plan.set_launch(sh["concurrent"], sh["wg"], sh["tile"])

    def effective(plan, tile):
        """The tiles that ``tile`` stands for (every launch below sets its own shape first)."""
        if plan.buckets():
            plan.set_launch(True, None, tile)
        return plan.tiles()

    apply()
    best = _timed_together(runs, reps, warm)
    trials = [{"tiles": [list(sh["tile"]) for sh in shapes], "seconds": best}]
    if uniform:
        # every combination of (own tuning, the library's choice, second tile everywhere, first
        # tile everywhere) over the plans, each shape once (at most three plans; more: one plan
        # at a time)
        opts = []
        for j, (plan, *_) in enumerate(runs):
            nt = [b[3] for b in plan.buckets()]
            o, seen = [], []
            for cand in (list(shapes[j]["tile"]), [-1] * len(nt), [1 if t > 1 else 0 for t in nt], [0] * len(nt)):
                runs_on = effective(plan, cand)
                if runs_on not in seen:
                    o.append(cand)
                    seen.append(runs_on)
            opts.append(o)
        combos = list(itertools.product(*opts)) if len(runs) <= 3 else \
            [tuple(o[k] if i == j else o[0] for i, o in enumerate(opts)) for j in range(len(opts))
             for k in range(1, len(opts[j]))]
        keep = [list(sh["tile"]) for sh in shapes]
        for combo in combos:
            if [list(c) for c in combo] == keep or all(list(c) == o[0] for c, o in zip(combo, opts)):
                continue
            for sh, c in zip(shapes, combo):
                sh["tile"] = list(c)
            apply()
            sec = _timed_together(runs, reps, warm)
            trials.append({"tiles": [list(sh["tile"]) for sh in shapes], "seconds": sec})
            if sec < best * (1.0 - min_gain):
                best, keep = sec, [list(c) for c in combo]
        for sh, c in zip(shapes, keep):
            sh["tile"] = list(c)
        apply()
    flips = [(cnt << l2, j, b) for j, (plan, *_) in enumerate(runs)
             for b, (l2, cnt, _mx, ntile) in enumerate(plan.buckets()) if ntile > 1]
    for _, j, b in sorted(flips, reverse=True):
        old = shapes[j]["tile"][b]
        shapes[j]["tile"][b] = _other_tile(runs[j][0].tiles()[b])
        apply()
        sec = _timed_together(runs, reps, warm)
        trials.append({"tiles": [list(sh["tile"]) for sh in shapes], "seconds": sec})
        if sec < best * (1.0 - min_gain):
            best = sec
        else:
            shapes[j]["tile"][b] = old
    apply()
    return {"tiles": [list(sh["tile"]) for sh in shapes], "seconds": best, "trials": trials}
