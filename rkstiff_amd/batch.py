"""Batched ensembles: thousands of independent trajectories in one launch.

``BatchSolver`` integrates a list of trajectories that share a method and a
built-in nonlinearity kind but may differ in grid size, lin_op, wavenumbers,
initial state, time span and step size.  Each trajectory keeps its own
adaptive dt, accept flag and status; one persistent-kernel launch per grid
size bucket (instances grouped by n, largest first, pulled from an atomic work
queue) integrates all of them.  This is the throughput path; the reference's
API (one solver object per trajectory) is the drop-in in ``solvers``.

Precision:
  "f64"    FP64 everywhere (matches the reference to rounding)
  "f32"    FP32 state, stages, FFTs and coefficients (FP64 coefficient
           generation, error norm and dt control)
  "mixed"  FP64 state, propagators exp(f h L) and FFTs; FP32 NL arrays and
           the remaining coefficients (FP32 storage halves their HBM bytes;
           the FP64 propagators and FFTs keep the error at the FP64 level of
           the step-sequence sensitivity)
"""
import numpy as np
import torch

from . import _lib
from .config import SolverConfig
from .engine import Plan

PRECISIONS = {"f64": _lib.F64, "f32": _lib.F32, "mixed": _lib.MIXED}


class BatchSolver:
    """Evolve many trajectories of one method/nonlinearity kind together."""

    def __init__(self, method, problems, precision="f64", config=None, etd_config=None,
                 max_loops=50, max_s=4.0, min_s=0.25):
        if method not in _lib.METHOD_IDS:
            raise ValueError(f"unknown method {method}")
        if precision not in PRECISIONS:
            raise ValueError(f"precision must be one of {sorted(PRECISIONS)}")
        if not problems:
            raise ValueError("no problems")
        kinds = {p[1].kind for p in problems}
        if len(kinds) != 1:
            raise ValueError("all problems of a batch must share one nonlinearity kind")
        self.method = method
        self.precision = precision
        self.config = config if config is not None else SolverConfig()
        nl0 = problems[0][1]
        descs = []
        for L, nl in problems:
            if nl.modes() != (L.shape[0] if hasattr(L, "shape") else len(L)):
                raise ValueError("lin_op and nonlinear term have different numbers of modes")
            descs.append(nl.descriptor(L))
        self.plan = Plan(method, nl0, PRECISIONS[precision], self.config, etd_config, descs,
                         max_loops, max_s, min_s)
        self.modes = self.plan.modes
        self.dtype = self.plan.dtype
        self._stats = None

    @property
    def adaptive(self):
        return bool(_lib.tableau(self.method).adaptive)

    def evolve(self, u0, t0, tf, h=None, sync=True):
        """u0: list of device tensors; t0/tf/h: scalars or per-trajectory lists.

        h is h_init for adaptive methods (default (tf - t0)/100, as evolve) and
        the constant step for constant-step methods.  Returns the list of
        states at tf (new tensors).
        """
        n = len(u0)
        if n != self.plan.ninst:
            raise ValueError(f"expected {self.plan.ninst} initial states, got {n}")
        t0s = np.broadcast_to(np.asarray(t0, dtype=np.float64), (n,)).tolist()
        tfs = np.broadcast_to(np.asarray(tf, dtype=np.float64), (n,)).tolist()
        if h is None:
            if not self.adaptive:
                raise ValueError("constant-step methods need h")
            hs = [(b - a) / 100.0 for a, b in zip(t0s, tfs)]
        else:
            hs = np.broadcast_to(np.asarray(h, dtype=np.float64), (n,)).tolist()
        if not self.adaptive:
            for a, b, hh in zip(t0s, tfs, hs):
                if a + hh > b:
                    raise ValueError("Step size h must be <= (tf - t0); reduce h or extend tf.")
        # per trajectory, this loop and the plan's are what a large ensemble spends on the host:
        # 2048 states cost 5.0 ms before the launch with a conversion of each, 3.2 ms without
        dtype = self.dtype
        u0 = [u if u.dtype is dtype and u.is_contiguous() else u.to(dtype).contiguous() for u in u0]
        uf = [torch.empty_like(u) for u in u0]
        self.plan.set_storage(0, 0, 0)
        self.plan.evolve(u0, uf, t0s, tfs, hs)
        # counters of this evolve: read now, or (sync=False) at the next stats() call
        self._stats = self.plan.stats() if sync else None
        return uf

    def autotune(self, u0, t0, tf_probe, h=None, reps=2):
        """Pick the launch shape (rkstiff_amd.autotune) on pilot evolves t0 -> tf_probe."""
        from .autotune import tune_launch
        u0 = [u.to(self.dtype).contiguous() for u in u0]
        if h is None:
            h = (np.asarray(tf_probe, dtype=np.float64) - np.asarray(t0, dtype=np.float64)) / 100.0
        self.plan.set_storage(0, 0, 0)
        return tune_launch(self.plan, u0, t0, tf_probe, h, reps=reps)

    # -- learned step-size proposer (rkstiff_amd.learned) ----------------------
    def record(self, cap):
        """Keep up to ``cap`` training records per trajectory during the next evolves."""
        self.plan.set_records(cap)

    def records(self):
        """(records (ninst, cap, 68) device tensor, records per trajectory)."""
        return self.plan.read_records()

    def set_proposer(self, net, margin=0.0, keep=None, policy="propose", period=1):
        """Set the step after accepted steps with ``net`` (a DtProposer); None restores the
        reference's controller.  The network runs after every (``period`` 512 / T)-th
        accepted step, T the trajectory's workgroup size (the reference's proposal stands
        after the others).  With d = y - margin (y: the
        network output) and h_ref the reference controller's proposal:

        "propose"  keep h (no coefficient regeneration) when keep[0] <= d < keep[1], else
                   take h exp(d); the default band [0, ln incr_f) mirrors the reference
                   keeping h while 1 <= s <= incr_f.
        "guard"    h_ref, unless d < ln(h_ref / h) + keep[0] (the network predicts its
                   rejection): then take h exp(d) ahead of it.  Default keep[0] = 0.
        "grow"     as "guard", and when d >= ln(h_ref / h) + g with g = keep[1] > 0, grow
                   ahead of the reference to h_ref e^(j g), j = floor((d - ln(h_ref / h)) / g):
                   steps on a geometric grid, so few coefficient regenerations.
                   Default keep = (0, ln 2 / 8).
        """
        if keep is None:
            keep = (0.0, float(np.log(2.0) / 8.0)) if policy == "grow" else (0.0, float(np.log(self.config.incr_f)))
        self.plan.set_proposer(net, margin, keep, policy, period)

    def stats(self):
        """Per-trajectory counters: tc, steps, attempts, rejects, status, ..."""
        if self._stats is None:
            self._stats = self.plan.stats()
        return self._stats

    def failures(self):
        """Indices of trajectories that stopped with MAXLOOPS / MINSTEP."""
        return [i for i, s in enumerate(self.stats()) if s["status"] not in (_lib.RKS_OK,)]
