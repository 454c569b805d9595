"""Dense (non-diagonal) strategies on the device for a batch of small systems.

The reference's dense strategies (etd35.py:498-720, etd34.py:307-436,
etd4.py:178-308, etd5.py:264-482, if34.py:202-254, if4.py:125-199) keep
matrix coefficients: exponentials of f h L (scipy's expm) and psi functions
by the contour mean h (1/N) sum_m r_m psi_r(r_m) (r_m I - f h L)^-1, combined
per method; stages are matrix-vector products.  ``coefficients`` computes
every coefficient matrix of B systems in one set of launches
(rks_dense_coeffs: Pade-13 scaling and squaring, Gauss-Jordan inverses, the
recipes), and ``combine`` forms one stage sum for all of them
(rks_dense_combine).  The drop-in solvers use both with B = 1.
"""
import ctypes

import torch

from . import _lib
from .config import ETDConfig


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def coefficients(method, L, h, etd_config=None):
    """(B, ncoef, n, n) complex128 coefficient matrices (tableau order) of ``method`` at
    z_b = h_b L_b.  L: (B, n, n) or (n, n) complex128 device tensor; h: float or B floats."""
    lib = _lib.load()
    if method not in _lib.METHOD_IDS:
        raise ValueError(f"unknown method {method}")
    etd = etd_config if etd_config is not None else ETDConfig()
    L = L.to(torch.complex128)
    if L.dim() == 2:
        L = L.unsqueeze(0)
    if L.dim() != 3 or L.shape[1] != L.shape[2]:
        raise ValueError("L must be (B, n, n)")
    if not L.is_cuda:
        raise TypeError("L must be a device tensor")
    L = L.contiguous()
    B, n = L.shape[0], L.shape[1]
    hs = [float(h)] * B if not hasattr(h, "__len__") else [float(x) for x in h]
    if len(hs) != B:
        raise ValueError("one h per system")
    ncoef = _lib.tableau(method).ncoef
    out = torch.empty((B, ncoef, n, n), dtype=torch.complex128, device=L.device)
    harr = (ctypes.c_double * B)(*hs)
    mid, points = _lib.METHOD_IDS[method], int(etd.contour_points)
    # work memory from torch's stream-ordered allocator: nothing to wait for before it is reused
    nbytes = ctypes.c_size_t()
    _lib.check(lib.rks_dense_ws_bytes(mid, n, B, points, ctypes.byref(nbytes)))
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device=L.device)
    _lib.check(lib.rks_dense_coeffs_ws(mid, n, B, ctypes.c_void_p(L.data_ptr()), harr, points,
                                       float(etd.contour_radius), ctypes.c_void_p(out.data_ptr()),
                                       ctypes.c_void_p(ws.data_ptr()), ws.numel(), _stream()))
    return out


def combine(terms, out):
    """out[b] = sum of alpha * mat[b] (x[b] + s2 x2[b]) over ``terms``, a list of
    (mat or None, x, x2 or None, s2, alpha) with complex128 device tensors shaped
    (B, n, n) / (B, n); out: (B, n) complex128, distinct from every x."""
    lib = _lib.load()
    if not 1 <= len(terms) <= _lib.DENSE_MAX_TERMS:
        raise ValueError(f"1 to {_lib.DENSE_MAX_TERMS} terms")
    B, n = out.shape
    arr = (_lib.DenseTerm * len(terms))()
    keep = []
    for k, (mat, x, x2, s2, alpha) in enumerate(terms):
        for v in (x, x2):
            if v is not None and (v.dtype != torch.complex128 or not v.is_contiguous() or v.numel() != B * n):
                raise ValueError("term vectors must be contiguous complex128 (B, n)")
        if mat is not None and (mat.dtype != torch.complex128 or not mat.is_contiguous() or mat.numel() != B * n * n):
            raise ValueError("term matrices must be contiguous complex128 (B, n, n)")
        keep.append((mat, x, x2))
        arr[k].mat = mat.data_ptr() if mat is not None else None
        arr[k].x = x.data_ptr()
        arr[k].x2 = x2.data_ptr() if x2 is not None else None
        arr[k].s2 = float(s2)
        arr[k].alpha = float(alpha)
    _lib.check(lib.rks_dense_combine(n, B, arr, len(terms), ctypes.c_void_p(out.data_ptr()), _stream()))
    return out
