"""Products with a 64-wide inner side over edge-sized rows on ``ictc_hip_gates_*`` (fp32 operands in
three bf16 parts on the matrix cores): the radial network's last layer ``h W^T`` (reference
``mace_ictc/models/pure_cartesian_ictd_fix.py:1545-1553``), its input adjoint ``g W`` and its
weight adjoint ``g^T h``.  ``product`` recognises the three forms in ``a @ b``; ``linear.mm`` asks
it first and keeps its library routes for every other shape.

The lines between the routes (MI355X, us per call in a replayed graph, the library's time in brackets):

* forward from 2,048 rows and 6 M results: a block has its rows to load and split before its first
  product, so that a small launch takes 6 us whatever its size: 6.0 (2.7) at 2,048 x 128, 6.9 (5.8) at 5,500 x
  352, 7.0 (6.2) at 3,500 x 704, 6.9 (5.7) at 20,000 x 128.  Between 3.5 and 6 M the two are close alone, 10.3 (11.1)
  at 16,000 x 288, 10.0 (8.9) at 40,000 x 128, but between other kernels the library is ahead (that size with its radial
  kernels and adjoints 48.6, 44.5); from the line on 9.8 (10.3) at 16,000 x 384, 10.0 (12.3) at 2,048 x 2,944, 16.9 (18.0) at
  28,000 x 352, 288 (408) at 105,634 x 2,944;
* input adjoint from 50,000 rows: a block takes 128 rows and a fixed 1.1 us per 32 columns, so fewer
  rows leave CUs idle: 105 (88) at 8,192 x 2,944, 120 (108) at 32,768 x 2,944, 176 (225) at 50,000 x 2,944, 40 (40) at
  65,000 x 512, 81 (94) at 105,634 x 704, 311 (373) at 105,634 x 2,944.  A second round of blocks begins above
  131,072 rows and costs 36 us at 2,944 columns, less than the lead: 365 (466) at 131,072, 401 (480) at 131,200,
  418 (481) at 140,000, 599 (714) at 211,000; 59 (60) at 131,200 x 352, 28 (28) at 140,000 x 128;
* both of these from rows of whole 64-byte lines: the kernels stream the [E, N] rows past the caches, which the lines
  that two rows share do not bear.  At 105,000 rows forward 34 (28) at 132 columns, 44 (36) at 200, 54 (45) at 264, 114
  (84) at 552, but 22 (26) at 144, 27 (32) at 176, 52 (60) at 400, 66 (75) at 528; input adjoint 44 (42) at 264, 50 (46) at
  300, 83 (74) at 552, but 44 (45) at 352, 57 (58) at 480;
* weight adjoint from 4,096 rows, or 2,048 from 640 columns: 15 (11) at 2,048 x 128, 15 (12) at 2,048 x 512, 17 (16)
  at 4,000 x 512; 16 (18) at 2,048 x 704, 17 (33) at 8,000 x 128, 22 (23) at 8,000 x 704, 19 (25) at 16,000 x 128,
  156 (216) at 105,634 x 1,408.
"""
from __future__ import annotations

from typing import Optional

import torch

from ... import _lib

WIDTH = 64
MIN_OUTER = 128            # narrower outer sides stay on the library (its 64 x 64 products take one tile)
FORWARD_ROWS = 2048
FORWARD_RESULTS = 6_000_000
INPUT_GRAD_ROWS = 50000
WEIGHT_GRAD_ROWS = 2048
WEIGHT_GRAD_NARROW = 640   # narrower outer sides ...
WEIGHT_GRAD_NARROW_ROWS = 4096   # ... from these rows
LINE = 16                  # floats of a 64-byte line
MAX_OUTER = 1 << 20
MAX_ROW_STRIDE = 1 << 22


def _rows(t: torch.Tensor, width: int) -> bool:
    """t [R, width] read row by row: unit column stride, rows that do not overlap."""
    return t.stride(1) == 1 and width <= t.stride(0) <= MAX_ROW_STRIDE


def _lines(t: torch.Tensor) -> bool:
    """Rows that start on a 64-byte line."""
    return t.stride(0) % LINE == 0 and t.data_ptr() % (4 * LINE) == 0


def _hidden(t: torch.Tensor) -> bool:
    return t.stride(1) == 1 and t.stride(0) == WIDTH and t.data_ptr() % 16 == 0


def _weight(t: torch.Tensor) -> bool:
    """t [outer, 64] within the kernels' 32-bit byte offsets."""
    sn, sk = t.stride()
    return 0 <= sn <= 1 << 28 and 0 <= sk <= 1 << 22 and (t.shape[0] - 1) * sn + (WIDTH - 1) * sk < 1 << 29


def _forward(hidden: torch.Tensor, weight: torch.Tensor, out: Optional[torch.Tensor]) -> torch.Tensor:
    edges, width = hidden.shape[0], weight.shape[0]
    if out is None:
        out = torch.empty(edges, width, device=hidden.device, dtype=torch.float32)
    _lib.check(_lib.lib().ictc_hip_gates_forward(
        hidden.data_ptr(), weight.data_ptr(), weight.stride(0), weight.stride(1), out.data_ptr(), out.stride(0), edges,
        width, _lib.stream_of(hidden.device)), "ictc_hip_gates_forward")
    return out


def _input_grad(grad: torch.Tensor, weight: torch.Tensor, out: Optional[torch.Tensor]) -> torch.Tensor:
    edges, width = grad.shape
    if out is None:
        out = torch.empty(edges, WIDTH, device=grad.device, dtype=torch.float32)
    _lib.check(_lib.lib().ictc_hip_gates_input_grad(
        grad.data_ptr(), grad.stride(0), weight.data_ptr(), weight.stride(0), weight.stride(1), out.data_ptr(), edges,
        width, _lib.stream_of(grad.device)), "ictc_hip_gates_input_grad")
    return out


def _weight_grad(grad: torch.Tensor, hidden: torch.Tensor, transposed: bool) -> torch.Tensor:
    """g^T h [N, 64], or its transpose [64, N]."""
    edges, width = grad.shape
    lib, dev = _lib.lib(), grad.device
    floats = int(lib.ictc_hip_gates_weight_grad_workspace(edges, width))
    if floats < 0:
        _lib.check(-floats, "ictc_hip_gates_weight_grad_workspace")
    ws = torch.empty(max(floats, 1), device=dev, dtype=torch.float32)
    out = torch.empty((WIDTH, width) if transposed else (width, WIDTH), device=dev, dtype=torch.float32)
    strides = (1, width) if transposed else (WIDTH, 1)
    _lib.check(lib.ictc_hip_gates_weight_grad(
        grad.data_ptr(), grad.stride(0), hidden.data_ptr(), ws.data_ptr(), floats, out.data_ptr(), *strides, edges,
        width, _lib.stream_of(dev)), "ictc_hip_gates_weight_grad")
    return out


def product(a: torch.Tensor, b: torch.Tensor, out: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """a [M, K] @ b [K, N] when it is one of the three forms at a size they are the faster route
    for; None otherwise.  out: a caller's row-major result (the first two forms; a row slice of a
    wider matrix for the first)."""
    m, k = a.shape
    n = b.shape[1]
    outer = m if n == WIDTH else n
    # sizes first: a small call's products end here
    forward = k == WIDTH and m >= FORWARD_ROWS and m * n >= FORWARD_RESULTS and MIN_OUTER <= n <= MAX_OUTER
    input_grad = n == WIDTH and m >= INPUT_GRAD_ROWS and MIN_OUTER <= k <= MAX_OUTER and k % 4 == 0
    weight_grad = (k >= WEIGHT_GRAD_ROWS and (n == WIDTH or m == WIDTH) and out is None
                   and MIN_OUTER <= outer <= MAX_OUTER
                   and (k >= WEIGHT_GRAD_NARROW_ROWS or outer >= WEIGHT_GRAD_NARROW))
    if not (forward or input_grad or weight_grad) or not a.is_cuda or a.device != b.device:
        return None
    if a.dtype != torch.float32 or b.dtype != torch.float32:
        return None
    if (forward and _hidden(a) and _weight(b.t())
            and (n % LINE == 0 if out is None else _rows(out, n) and _lines(out))):
        return _forward(a, b.t(), out)
    if (input_grad and _rows(a, k) and _lines(a) and _weight(b)
            and (out is None or (out.stride(0) == WIDTH and out.stride(1) == 1))):
        return _input_grad(a, b, out)
    if weight_grad and n == WIDTH and _rows(a.t(), m) and b.stride(1) == 1 and b.stride(0) == WIDTH:
        return _weight_grad(a.t(), b, False)
    if weight_grad and m == WIDTH and _rows(b, n) and a.stride(0) == 1 and a.stride(1) == WIDTH:
        return _weight_grad(b, a.t(), True)
    return None
