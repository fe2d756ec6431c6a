"""Whole solves of small problems through ``fs_small_solve`` / ``fs_small_grad``.

On small clouds a loss is bound by launches and by the host: some 240 launches and 1.9 ms for a
debiased loss and gradient of 256 x 256 x 16 when every norm, log weight, bounding box and plane
conversion is a PyTorch operation and every step two launches per problem.  Here the xy problem,
the two self problems of a debiased loss and every item of a batch advance together, one launch
per step, and what stands around the steps is two launches in front and one behind; the
gradient of the whole (debiased) loss is one launch.

The functions here decide whether a call is such a problem (``loss_problem``, ``solver_problem``),
run it (``solve``) and differentiate it (``_SmallLoss``, same conventions as ``_autograd``).
"""
from __future__ import annotations

import ctypes
import os
import threading
from types import SimpleNamespace
from typing import Optional

import torch

from flash_sinkhorn_amd import _graphs, _lib
from flash_sinkhorn_amd.kernels._common import epsilon_schedule, max_diameter

_P, _I64, _D, _F, _I = (ctypes.c_void_p, ctypes.c_int64, ctypes.c_double, ctypes.c_float,
                        ctypes.c_int)
_DTYPES = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}

MAX_ROWS = 65536
WIDE_D = 128  # from here on the products of the clouds are kept (fs_dense.hpp), at most this many:
MAX_KEPT = 1 << 28
MAX_D = 16384  # rows that the kernels take at all
KEEP_PRODUCTS = os.environ.get("FLASH_SINKHORN_KEEP_PRODUCTS", "1") != "0"  # (keeps_products)
_TABLE = 511  # entries of a schedule the device keeps
# Most workspace of a batch: planes, value operands and vectors of every item, until the backward pass
# (0.9 MB for a debiased item of 2,048 x 3).  Item by item there is next to nothing to hold.
MAX_BATCH_BYTES = 16 << 30
MAX_GRAPH_BYTES = 32 << 20  # of a batch's workspace, where its run is kept as a graph


class Problem(ctypes.Structure):
    """``fs_small_problem``."""
    _fields_ = [("x", _P), ("y", _P), ("a", _P), ("b", _P), ("eps_list", _P),
                ("n", _I64), ("m", _I64), ("d", _I64), ("items", _I64),
                ("blur", _D), ("scaling", _D),
                ("cost_scale", _F), ("eps", _F), ("rho_x", _F), ("rho_y", _F), ("threshold", _F),
                ("dtype", _I), ("normalize", _I), ("self_terms", _I), ("want_values", _I),
                ("sched", _I), ("entries", _I), ("cut", _I), ("extrapolate", _I),
                ("check_every", _I), ("alternating", _I)]


class Declined(Exception):
    """The schedule has more entries than the device keeps, or the workspace of a batch more bytes
    than are right to hold: the general path takes the call, item by item."""


_words = threading.local()


def _host_words(items: int) -> torch.Tensor:
    """Pinned ints in which a call finds the lengths of its schedules; one buffer per thread (the
    call that uses it returns only after the device has written it)."""
    buf = getattr(_words, "buf", None)
    if buf is None or buf.numel() < 4 * items:
        buf = _words.buf = torch.empty(max(256, 4 * items), dtype=torch.int32, pin_memory=True)
    return buf


_SIDES = ("f", "g", "xx", "yy")


class Solved:
    """A solve that has been enqueued: what it read, its workspace (planes, log weights, potentials in
    the form the gradient kernel reads) where a gradient may be asked for, the loss per item, and the
    standard potentials: of a loss in one buffer, for its own backward pass, of a solver every
    one a tensor of its own, for the caller."""
    __slots__ = ("form", "x", "y", "a", "b", "ws", "loss", "pots", "own", "entries")

    def problem(self) -> Problem:
        p = Problem.from_buffer_copy(self.form)
        p.x, p.y, p.a, p.b = self.x.data_ptr(), self.y.data_ptr(), _lib.ptr(self.a), _lib.ptr(self.b)
        return p

    def tensors(self):
        """What a backward pass needs, in the order ``restored`` takes it."""
        return self.x, self.y, self.a, self.b, self.ws, self.pots

    @classmethod
    def restored(cls, form: Problem, tensors) -> "Solved":
        s = cls()
        s.form, s.loss, s.own, s.entries = form, None, None, None
        s.x, s.y, s.a, s.b, s.ws, s.pots = tensors
        return s

    def potentials(self, which: str):
        """("f" | "g" | "xx" | "yy") -> (of the cost, of the gradient): of a loss [items, rows] each,
        of a solver as the caller gets them (None: not asked for)."""
        if self.own is not None:
            return self.own[which]
        p = self.form
        n, m, k = p.n * p.items, p.m * p.items, _SIDES.index(which)
        at = [0, 2 * n, 2 * (n + m), 2 * (2 * n + m)][k]
        size = n if k % 2 == 0 else m
        rows = p.n if k % 2 == 0 else p.m
        return tuple(self.pots[at + i * size:at + (i + 1) * size].view(p.items, rows) for i in (0, 1))


def _size_ok(n: int, m: int, d: int, fixed: bool, self_terms: int, stops: bool,
             items: int = 1, steps: int = 0) -> bool:
    """Whether a problem of this size is faster here than on the general path, launch by launch.
    ``steps``: averaged steps at a fixed eps (0: of no matter, the problem is not large).

    d > 128: while the kept products stay below 1 GiB; reading them beats forming them at every such
    width (8,192 x 1,536: 0.07 against 0.5 ms a step).

    d <= 64 (``pair_sweep_kernel`` from 2e7 logits per step on): everywhere but for few steps at a fixed eps
    on two clouds of 24,000 rows and more.  The general path runs the first steps faster, these
    kernels the others, so the line is a number of steps that grows with the logits of one: 12 per 1e9 of
    them less 4 on 33 .. 64 columns, 5 less 5 on fewer.  Loss and gradient here / there, ms, N(0, I) at eps
    0.01 and 0.1, eight clusters at 0.01, 64 columns, after 8 | 20 | 100 steps:
      40,000: 6.9 / 6.3, 9.2 / 7.6, 8.1 / 7.6 | 8.0 / 8.3, 12.1 / 11.0, 9.6 / 10.1 | 15.6 / 21.3, 30.8 / 34.4, 17.2 / 26.4
      50,000: 10.3 / 8.9, 13.3 / 10.7, 12.0 / 10.9 | 11.7 / 11.1, 17.8 / 15.1, 13.7 / 13.6 | 21.0 / 26.3, 42.5 / 44.1, 23.8 / 33.4
      65,000: 16.3 / 12.9, 21.3 / 15.8, 19.1 / 16.0 | 18.0 / 15.5, 27.9 / 21.3, 21.7 / 19.6 | 30.9 / 33.7, 63.4 / 59.6, 35.6 / 42.7
    and 12 columns:
      50,000: 6.1 / 5.6, 7.3 / 10.3, 5.9 / 5.7 | 8.9 / 8.1, 12.0 / 16.8, 7.4 / 8.4 | 24.0 / 25.1, 42.6 / 60.1, 16.2 / 26.4
      65,000: 9.6 / 7.9, 11.7 / 15.7, 9.1 / 7.9 | 13.9 / 11.0, 19.5 / 26.1, 11.1 / 11.4 | 36.5 / 32.4, 71.9 / 95.6, 23.2 / 32.8
    and 40 columns, whose planes are 48 wide here and 64 there, so that the line is too high for 33 .. 48 of them (it stands where
    64 columns have it):
      32,000: 3.1 / 4.5, 4.8 / 5.8, 3.9 / 5.7 | 4.1 / 6.1, 8.2 / 9.0, 4.7 / 8.1 | 10.1 / 17.0, 30.0 / 30.6, 10.1 / 24.1
      40,000: 4.6 / 5.5, 7.3 / 7.5, 5.8 / 7.0 | 5.9 / 7.4, 9.9 / 11.5, 6.9 / 9.7 | 14.5 / 19.7, 29.0 / 38.1, 14.2 / 27.7
      50,000: 6.6 / 7.8, 10.4 / 10.7, 8.5 / 10.0 | 8.2 / 10.0, 14.4 / 15.7, 9.8 / 13.1 | 18.8 / 24.6, 40.2 / 50.0, 19.1 / 34.4
      65,000: 10.8 / 11.2, 17.1 / 15.2, 13.5 / 14.4 | 13.1 / 13.9, 23.2 / 21.9, 15.4 / 18.5 | 28.2 / 31.3, 61.3 / 67.4, 27.7 / 46.1
    With self problems these kernels were faster in all of 160 settings from 26,000 to 60,000 rows (60,000 x 64, 10
    steps: 18.5 / 20.0, 45,000: 10.7 / 12.7), and so they are on schedules (60,000 x 64: 20.6 / 26.3).

    d <= 128, or early stopping on a schedule: the small kernels, which go over the logits once per
    side: up to 2e7 logits at fixed eps (3,000 x 128: 1.05 against 1.54 ms; 4,500: 2.8 against 2.4),
    6e7 on a schedule (6,500 x 128: 1.54 against 1.94 ms; 9,000: 3.1 against 2.8).
    """
    if not (0 < n <= MAX_ROWS and 0 < m <= MAX_ROWS and 0 < d <= MAX_D):
        return False
    if d > WIDE_D:
        return not self_terms and items * n * m <= MAX_KEPT
    if d > 64 or (stops and not fixed):
        logits = (n * m if self_terms < 2 else 0) + ((n * n + m * m) // 2 if self_terms else 0)
        return logits <= (20_000_000 if fixed else 60_000_000)
    if d <= 8 or not fixed or self_terms or not steps or min(n, m) < 24000:
        return True
    logits = n * m / 1e9
    return steps >= (12 * logits - 4 if d > 32 else 5 * logits - 5)


def _operands_ok(allow_tf32: bool) -> bool:
    return allow_tf32 or _lib.STRICT_OPERANDS == "fp16x2"


def held(*values: Optional[float]) -> bool:
    """Whether fp32 holds every one of these (None: not given) as a positive normal number.  The
    library reads zero and less as "none" (a strict marginal, no early stopping), so a relaxation of
    zero, a negative one or one that rounds to zero would be another problem: the general path
    takes such values, or refuses them."""
    for v in values:
        if v is not None and not 1.1754944e-38 <= v <= 3.4028234e38:
            return False
    return True


def _rho(rho: Optional[float]) -> float:
    return 0.0 if rho is None else float(rho)


def solve(x, y, a, b, *, items: int, blur: float = 0.0, scaling: float = 0.0, eps: float = 0.0,
          entries: int = 0, cut: int = 0, eps_list=None, cost_scale: float, rho_x, rho_y,
          normalize: bool, self_terms: int, want_values: bool, extrapolate: bool,
          want_loss: bool, threshold: Optional[float] = None, check_every: int = 1,
          alternating: bool = False, prelast: bool = False, keep: bool = False) -> Solved:
    """Enqueue one run of small problems: contiguous x [items, n, d] and y [items, m, d] of one dtype,
    weights as contiguous fp32 or None.  ``eps_list`` (host floats), ``eps`` with ``entries``, or
    a schedule by diameter, in that order.  Without ``want_loss``: the potentials, with ``prelast``
    also those before the extrapolation.  ``keep``: the workspace stays with the result also without
    ``want_values``."""
    n, d = x.shape[-2:]
    m = y.shape[-2]
    sched = 2 if eps_list is not None else (0 if eps > 0.0 else 1)
    table = None
    if sched == 2:
        entries = len(eps_list)
        if entries > _TABLE:
            raise Declined
        table = (ctypes.c_float * entries)(*eps_list)

    form = Problem(
        None, None, None, None, None, n, m, d, items, blur, scaling, cost_scale, eps, _rho(rho_x),
        _rho(rho_y), threshold or 0.0, _DTYPES[x.dtype], int(normalize), int(self_terms),
        int(want_values), sched, entries, cut, int(extrapolate), int(check_every),
        int(alternating))

    rows = (n + m) * items * (4 if self_terms else 2)
    # potentials for the caller: (side, kind) of every tensor
    own = () if want_loss else tuple(
        (side, kind) for side in ((2, 3) if self_terms == 2 else (0, 1, 2, 3) if self_terms else (0, 1))
        for kind in range(1 + bool(prelast)))

    p = Problem.from_buffer_copy(form)
    p.x, p.y = x.data_ptr(), y.data_ptr()
    if table is not None:
        p.eps_list = ctypes.addressof(table)
    L = _lib.lib()
    nbytes = L.fs_small_workspace_bytes(ctypes.byref(p))
    if items > 1 and nbytes > MAX_BATCH_BYTES:
        raise Declined
    kept = L.fs_small_products_bytes(ctypes.byref(p)) if d > 16 else 0  # (none at narrower rows)

    def enqueue(x, y, a, b):  # (of these clouds, or of a graph's copies)
        p.x, p.y, p.a, p.b = x.data_ptr(), y.data_ptr(), _lib.ptr(a), _lib.ptr(b)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
        # (tensors of their own: a caller may change or keep the loss and every potential)
        if want_loss:
            pots = (torch.empty(rows, dtype=torch.float32, device=x.device),)
            loss = torch.empty(x.shape[:-2], dtype=torch.float32, device=x.device)
        else:
            pots = tuple(torch.empty(x.shape[:-2] + (m if side & 1 else n,), dtype=torch.float32,
                                     device=x.device) for side, _ in own)
            loss = None
        words = _host_words(items).data_ptr() if sched == 1 or threshold else None
        # (of the solve alone: what follows it reads the workspace)
        products = torch.empty(kept, dtype=torch.uint8, device=x.device) if kept else None
        rc = L.fs_small_solve_products(
            ctypes.byref(p), ws.data_ptr(), ws.numel(), _lib.ptr(products), kept, words, _lib.ptr(loss),
            pots[0].data_ptr() if want_loss else None, _lib.stream_of(x))
        if rc > 0:
            if rc == 1:
                raise ValueError("diameter must be > 0.")
            if rc == 2:
                raise ValueError("the diameter of the clouds is not a number.")
            raise Declined
        _lib.check(rc, "fs_small_solve")
        if own:
            where = (_P * 8)()
            for (side, kind), t in zip(own, pots):
                where[2 * side + kind] = t.data_ptr()
            _lib.check(L.fs_small_potentials(ctypes.byref(p), ws.data_ptr(), ws.numel(), where,
                                             _lib.stream_of(x)), "fs_small_potentials")
        return pots + ((loss,) if want_loss else ()) + ((ws,) if want_values or keep else ())

    # (a graph keeps its products; of a batch it counts all items, and the workspace that a replay
    # may copy)
    if (sched == 0 and not threshold and not keep and _graphs.eligible(items * n, m, entries, x.device)
            and (d <= WIDE_D or items * n * m <= 1 << 22) and kept <= MAX_GRAPH_BYTES
            and (items == 1 or nbytes <= MAX_GRAPH_BYTES)):
        # a fixed sequence of kernels on fixed shapes: replayed (1.9 instead of 3 us per launch)
        key = ("self pair" if self_terms else "alternating" if alternating else "symmetric",
               int(self_terms), x.device.index, x.dtype, x.shape, y.shape,
               eps, entries, cost_scale, _rho(rho_x), _rho(rho_y), a is None, b is None, normalize,
               want_values, extrapolate, want_loss, own)
        out = _graphs.run(key, enqueue, [x, y, a, b])
    else:
        out = enqueue(x, y, a, b)
    s = Solved()
    s.form, s.x, s.y, s.a, s.b = form, x, y, a, b
    s.ws = out[-1] if want_values or keep else None
    s.pots, s.loss = out[:2] if want_loss else (None, None)
    s.own = None
    if own:
        got = dict(zip(own, out))
        s.own = {_SIDES[side]: (got[side, 0], got.get((side, 1))) for side, kind in own if kind == 0}
    s.entries = entries
    if threshold:  # averaged steps of the first problem
        word = int(_host_words(items)[0])
        if word >= 0 and word & 1:
            s.entries = (word // 2 + 1) * int(check_every)
        elif sched == 1:
            s.entries = None  # the words have been used for the checks
    elif sched == 1:
        s.entries = int(_host_words(items)[0])
    return s


def points(x, y):
    """The clouds as ``solve`` takes them: contiguous, of one type it reads (fp32 otherwise)."""
    if x.dtype not in _DTYPES or y.dtype is not x.dtype:
        x, y = x.float(), y.float()
    return x.detach().contiguous(), y.detach().contiguous()


def pair_problem(x, y, a, b, allow_tf32: bool, fixed: bool, self_terms: int = 0,
                 stops: bool = False, any_size: bool = False) -> bool:
    """Whether clouds and weights (any of which may need a gradient) are ones ``solve`` takes."""
    return (x.is_cuda and y.is_cuda and x.ndim == 2 and y.ndim == 2 and a.ndim == 1 and b.ndim == 1
            and x.shape[1] == y.shape[1]
            and (0 < x.shape[1] <= WIDE_D and max(x.shape[0], y.shape[0]) <= MAX_ROWS if any_size else
                 _size_ok(x.shape[0], y.shape[0], x.shape[1], fixed, self_terms, stops)
                 # (a solver called by itself on two large clouds takes the same kernels, to the last bit,
                 # whether it is asked for ``solve_info`` or not)
                 and (x.shape[1] <= 8 or min(x.shape[0], y.shape[0]) < 24000))
            and x.shape[0] > 0 and y.shape[0] > 0
            and a.shape[0] == x.shape[0] and b.shape[0] == y.shape[0]
            and x.is_floating_point() and y.is_floating_point() and _operands_ok(allow_tf32)
            and x.device == y.device == a.device == b.device)


def solver_problem(x, y, a, b, allow_tf32: bool, fixed: bool, stops: bool,
                   any_size: bool = False) -> bool:
    """Whether ``sinkhorn_flashstyle_symmetric`` may hand its clouds and weights to ``solve``.  One cloud
    against itself, with wide rows or on more than a few thousand points, stays with the general
    path: one half-update per step instead of two, and f equal to g to the bit."""
    if not any_size and x.data_ptr() == y.data_ptr() and a.data_ptr() == b.data_ptr() and x.shape == y.shape \
            and (x.shape[1] > WIDE_D or x.shape[0] ** 2 >= 20_000_000):
        return False
    return pair_problem(x, y, a, b, allow_tf32, fixed, 0, stops, any_size) and not (
        torch.is_grad_enabled()
        and (x.requires_grad or y.requires_grad or a.requires_grad or b.requires_grad))


def alternating_problem(x, y, a, b, allow_tf32: bool) -> bool:
    """Whether ``sinkhorn_flashstyle_alternating`` may hand its clouds and weights to ``solve``: a
    half-update is one launch of the small kernels, the streaming kernels' two.  Up to 1.4e8 logits, 6.5e7 on 33 .. 64
    columns, 3.6e7 on more; 40 iterations here / there, us a half-update: 8,000 x 3 16 / 23, 24 columns 21 / 26, 9,000 x 16
    33 / 30, 11,000 x 32 48 / 42, 12,000 x 16 42 / 39; 6,206 x 5,067 x 37 18 / 26, 8,000 x 40 27 / 33, x 60 33 / 35, 9,000 x 40
    50 / 47; 5,000 x 80 26 / 39, 6,000 x 80 35 / 42, x 128 40 / 44.  (The last third of the range on up to 32 columns has been the
    streaming kernels' since what stands in front of their loop is one launch: 10 % of a solve there.)"""
    n, m, d = x.shape[0], y.shape[0], x.shape[-1]
    return (solver_problem(x, y, a, b, allow_tf32, True, False, any_size=True)
            and n * m <= (140_000_000 if d <= 32 else 65_000_000 if d <= 64 else 36_000_000))


class Products:
    """The inner products that a solve of wide rows has kept, for the gradient in x and the Hessian-vector
    product behind it.  ``tensors`` are what an autograd node saves (the points as the solve read them and
    its workspace), ``restored`` makes it of them again."""
    __slots__ = ("form", "x", "y", "ws")

    def __init__(self, form: Problem, x, y, ws):
        self.form, self.x, self.y, self.ws = form, x, y, ws

    def tensors(self):
        return self.x, self.y, self.ws

    def problem(self) -> Problem:
        p = Problem.from_buffer_copy(self.form)
        p.x, p.y = self.x.data_ptr(), self.y.data_ptr()
        return p

    def gradient(self, grad_out):
        """The gradient in x times the scalar ``grad_out``, fp32 [n, d]."""
        p, L = self.problem(), _lib.lib()
        scratch = torch.empty(L.fs_dense_grad_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8,
                              device=self.x.device)
        gx = torch.empty(self.x.shape, dtype=torch.float32, device=self.x.device)
        gs = grad_out.detach().to(dtype=torch.float32).reshape(1).contiguous()
        _lib.check(L.fs_dense_grad(ctypes.byref(p), self.ws.data_ptr(), self.ws.numel(), gs.data_ptr(),
                                   gx.data_ptr(), scratch.data_ptr(), scratch.numel(),
                                   _lib.stream_of(self.x)), "fs_dense_grad")
        return gx


def _room(device, nbytes: int) -> bool:
    """Whether half of the card stays free with ``nbytes`` more of it held (what PyTorch's allocator
    has idle counts as free).  While a graph is captured its pool is the caller's: not asked."""
    if torch.cuda.is_current_stream_capturing():
        return True
    free, total = torch.cuda.mem_get_info(device)
    if free - nbytes < total // 2:
        free += torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device)
    return free - nbytes >= total // 2


def keeps_products(x, y) -> bool:
    """Whether a loss keeps the products of its solve for what follows it: of wide rows, where forming them
    again takes longer than a step (up to 2^22 of them a solve is a replayed graph, whose
    workspace is the next call's).

    They stay below 1 GiB, but until the loss's graph is freed, and a program may hold hundreds of losses:
    where less than half of the card would be left, or with FLASH_SINKHORN_KEEP_PRODUCTS=0, the
    gradient forms them again (8,192 x 1,536: 1.65 ms for 0.70) and nothing is held."""
    return (KEEP_PRODUCTS and x.is_cuda and x.ndim == 2 and WIDE_D < x.shape[1] <= MAX_D and x.dtype in _DTYPES
            and y.dtype is x.dtype and 1 << 22 < x.shape[0] * y.shape[0] <= MAX_KEPT
            and _room(x.device, 4 * (x.shape[0] * y.shape[0] + (x.shape[0] + y.shape[0]) * x.shape[1])))


def _weights(w, lead, count, device, normalize):
    """(fp32 contiguous weights of shape lead + (count,) or None, does ``solve`` normalise them);
    False where the general path has to complain."""
    if w is None:
        return None, False
    if not torch.is_tensor(w) or not w.is_floating_point() or w.device != device:
        return False, False
    if w.shape == lead + (count, 1):
        w = w[..., 0]
    if w.shape != lead + (count,):
        return False, False
    w = w.float()
    if normalize and w.requires_grad and torch.is_grad_enabled():  # the division is part of the graph
        w = w / w.sum(dim=-1, keepdim=True).clamp(min=1e-40)
        normalize = False
    return w.contiguous(), normalize


def loss_problem(loss, args, label_x, label_y):
    """(x, y, a, b, normalize) when a ``SamplesLoss`` call is a small problem, else None.  Calls that
    are not (or not valid) are left to the general path, its checks and its messages."""
    if loss.backend != "symmetric" or loss.eps_list is not None:
        return None
    if loss.threshold is not None and (loss.inner_iterations <= 0
                                       or torch.cuda.is_current_stream_capturing()):
        return None
    if loss.diameter is not None or not _operands_ok(loss.allow_tf32):
        return None
    if label_x is not None and label_y is not None and loss.label_cost_matrix is not None \
            and loss.lambda_y != 0.0:
        return None
    if loss.threshold is not None and not loss.threshold > 0.0:
        return None
    if not held(loss.rho_x, loss.rho_y, loss.threshold, loss.cost_scale):
        return None
    if loss.debias and loss.rho_x != loss.rho_y and not loss.potentials:
        return None
    if loss.use_epsilon_scaling:
        if not (loss.blur > 0.0 and held(loss.blur ** 2) and 0.0 < loss.scaling < 1.0) \
                or (loss.n_iters or 1) <= 0:
            return None
    elif loss.eps is None or loss.n_iters is None or not held(loss.eps) or loss.n_iters <= 0:
        return None
    if len(args) == 2:
        (x, y), a, b = args, None, None
    elif len(args) == 4:
        a, x, b, y = args
    else:
        return None
    if not torch.is_tensor(x) or not torch.is_tensor(y) or not x.is_floating_point() \
            or not y.is_floating_point() or not x.is_cuda or y.device != x.device:
        return None
    if x.ndim not in (2, 3) or y.ndim != x.ndim or x.shape[-1] != y.shape[-1] \
            or x.shape[:-2] != y.shape[:-2]:
        return None
    if not _size_ok(x.shape[-2], y.shape[-2], x.shape[-1], not loss.use_epsilon_scaling,
                    int(loss.debias and not loss.potentials), loss.threshold is not None,
                    x.shape[0] if x.ndim == 3 else 1, 0 if loss.use_epsilon_scaling else loss.n_iters):
        return None
    if x.shape[-1] > WIDE_D and (loss.use_epsilon_scaling or not loss.potentials):
        return None  # (by the solver alone: neither cost, gradients nor diameters are built for it)
    lead = x.shape[:-2]
    if lead and not 0 < lead[0] <= 65535:
        return None
    if not (loss.normalize or loss.potentials) and any(
            torch.is_tensor(w) and w.dtype is torch.float64 for w in (a, b)):
        return None  # (such a loss is summed and returned in their type)
    a, norm_a = _weights(a, lead, x.shape[-2], x.device, loss.normalize)
    b, norm_b = _weights(b, lead, y.shape[-2], x.device, loss.normalize)
    if a is False or b is False:
        return None
    if a is not None and b is not None and norm_a != norm_b:  # one of them needs a gradient
        a = a if norm_b else a / a.sum(dim=-1, keepdim=True).clamp(min=1e-40)
        b = b if norm_a else b / b.sum(dim=-1, keepdim=True).clamp(min=1e-40)
        norm_a = norm_b = False
    return x, y, a, b, norm_a or norm_b


def _solve_for(loss, x, y, a, b, normalize, **kw) -> Solved:
    sched = (dict(blur=loss.blur, scaling=loss.scaling, cut=loss.n_iters or 0)
             if loss.use_epsilon_scaling else dict(eps=loss.eps, entries=loss.n_iters))
    return solve(*points(x, y), None if a is None else a.detach(), None if b is None else b.detach(),
                 items=x.shape[0] if x.ndim == 3 else 1, cost_scale=loss.cost_scale,
                 rho_x=loss.rho_x, rho_y=loss.rho_y, normalize=normalize,
                 extrapolate=loss.last_extrapolation, threshold=loss.threshold,
                 check_every=loss.inner_iterations, **sched, **kw)


def potentials(loss, x, y, a, b, normalize):
    s = _solve_for(loss, x, y, a, b, normalize, self_terms=0, want_values=False, want_loss=False)
    return s.potentials("f")[0], s.potentials("g")[0]


def _gradients(s: Solved, grad_out, want_x: bool, want_y: bool):
    p, L = s.problem(), _lib.lib()
    gx = torch.empty(s.x.shape, dtype=torch.float32, device=s.x.device) if want_x else None
    gy = torch.empty(s.y.shape, dtype=torch.float32, device=s.x.device) if want_y else None
    gs = grad_out.float().contiguous()
    _lib.check(L.fs_small_grad(ctypes.byref(p), s.ws.data_ptr(), s.ws.numel(), gs.data_ptr(),
                               _lib.ptr(gx), _lib.ptr(gy), _lib.stream_of(s.x)), "fs_small_grad")
    return gx, gy


class _SmallGrad(torch.autograd.Function):
    """The gradients, differentiable once more in x (``_autograd._SinkhornGradFn``)."""

    @staticmethod
    def forward(ctx, x, y, grad_out, solved, config, want_x, want_y):
        gx, gy = _gradients(solved, grad_out, want_x, want_y)
        ctx.save_for_backward(x, y, grad_out, *solved.tensors())
        ctx.form, ctx.config = solved.form, config
        return gx, gy

    @staticmethod
    def backward(ctx, grad_grad_x, grad_grad_y):
        x, y, grad_out = ctx.saved_tensors[:3]
        from flash_sinkhorn_amd.hvp import hvp_x_sqeuclid_from_potentials
        cfg, s = ctx.config, Solved.restored(ctx.form, ctx.saved_tensors[3:])
        if grad_grad_y is not None or s.form.self_terms:
            raise NotImplementedError("Double backward w.r.t y is not implemented yet.")
        if grad_grad_x is None:
            return (None,) * 7
        items, f, g = s.form.items, s.potentials("f")[1], s.potentials("g")[1]
        outs = []
        with torch.no_grad():
            gs = grad_out.reshape(-1)
            for i in range(items):
                xi, yi, v = (t if t.ndim == 2 else t[i] for t in (x, y, grad_grad_x))
                weights = tuple(_item_weights(w, rows, i, s.form.normalize)
                                for w, rows in ((s.a, s.form.n), (s.b, s.form.m)))
                hvp, _ = hvp_x_sqeuclid_from_potentials(
                    xi, yi, f[i], g[i], v, eps=_last_eps(cfg, xi, yi), rho_x=cfg.rho_x, rho_y=cfg.rho_y,
                    cost_scale=cfg.cost_scale, tau2=cfg.hvp_tau2, max_cg_iter=cfg.hvp_max_cg_iter,
                    cg_rtol=cfg.hvp_cg_rtol, cg_atol=cfg.hvp_cg_atol,
                    cg_stabilise_every=cfg.hvp_cg_stabilise_every,
                    preconditioner=cfg.hvp_preconditioner, precond_terms=cfg.hvp_precond_terms,
                    use_preconditioner=cfg.hvp_use_preconditioner,
                    allow_tf32=False,  # second order needs full fp32 operands
                    use_exp2=cfg.use_exp2, _weights=weights, _scale=gs[i])
                outs.append(hvp)
        return (outs[0] if x.ndim == 2 else torch.stack(outs),) + (None,) * 6


def _last_eps(cfg, x, y) -> float:
    if not cfg.use_epsilon_scaling:
        return float(cfg.eps)
    if cfg.n_iters is None:
        return cfg.blur ** 2
    return epsilon_schedule(max_diameter(x, y), cfg.blur, cfg.scaling)[: cfg.n_iters][-1]


def _item_weights(w, rows, i, normalize):
    if w is None:
        return None
    w = w.reshape(-1, rows)[i]
    return w / w.sum().clamp(min=1e-40) if normalize else w


def _differentiate(form: Problem, config: dict, grad_out, tensors, need):
    """Gradients of a loss in x, y and its weights from what its node has saved: x and y, then
    ``Solved.tensors``."""
    x, y, *solved = tensors
    s = Solved.restored(form, solved)
    gx = gy = ga = gb = None
    if need[0] or need[1]:
        if x.dtype not in _DTYPES:  # (as the gradient of the general path)
            raise ValueError(f"Unsupported dtype for x/y: {x.dtype}")
        if torch.is_grad_enabled():  # create_graph
            gx, gy = _SmallGrad.apply(x, y, grad_out, s, SimpleNamespace(**config), need[0], need[1])
        else:
            gx, gy = _gradients(s, grad_out, need[0], need[1])
    scale = grad_out if x.ndim == 2 else grad_out[:, None]
    if need[2]:
        f = s.potentials("f")[0] - s.potentials("xx")[0] if form.self_terms else s.potentials("f")[0]
        ga = scale * (f if x.ndim == 3 else f[0])
    if need[3]:
        g = s.potentials("g")[0] - s.potentials("yy")[0] if form.self_terms else s.potentials("g")[0]
        gb = scale * (g if x.ndim == 3 else g[0])
    return gx, gy, ga, gb


class _SmallLoss(torch.autograd.Function):
    """Cost of every item, debiased or not, from one run; scalar for a single problem.  For what only a Function
    serves or refuses (tangents, any call inside a transform of functorch, subclasses); the others have a native
    node (``loss``)."""

    @staticmethod
    def forward(ctx, x, y, a, b, loss, normalize):
        need = ctx.needs_input_grad
        s = _solve_for(loss, x, y, a, b, normalize, self_terms=int(loss.debias),
                       want_values=need[0] or need[1], want_loss=True)
        ctx.save_for_backward(x, y, *s.tensors())
        # (the settings as they are now, for a second backward pass)
        ctx.form, ctx.config = s.form, dict(vars(loss))
        return s.loss

    @staticmethod
    def backward(ctx, grad_out):
        return _differentiate(ctx.form, ctx.config, grad_out, ctx.saved_tensors, ctx.needs_input_grad) + (None, None)


class _Ask:
    """What a native node calls for a gradient that it does not form itself."""
    __slots__ = ("form", "config")

    def __init__(self, form, config):
        self.form, self.config = form, config

    def __call__(self, grad_out, tensors, need):
        return _differentiate(self.form, self.config, grad_out, tensors, need)

    def node(self, tensors, shape, given):
        """A tensor whose node is a Function's with the same gradient, of stand-ins for x, y and the weights: compiled
        autograd records such a node as a call."""
        with torch.enable_grad():
            return _LateLoss.apply(self, tensors, shape, *given)


class _LateLoss(torch.autograd.Function):
    """See ``_Ask.node``."""

    @staticmethod
    def forward(ctx, ask, tensors, shape, x, y, a, b):
        ctx.ask = ask
        ctx.save_for_backward(*tensors)
        return tensors[2].new_empty(shape, dtype=torch.float32)

    @staticmethod
    def backward(ctx, grad_out):
        return (None, None, None) + tuple(ctx.ask(grad_out, ctx.saved_tensors, ctx.needs_input_grad[3:]))


_NATIVE = None


def _native():
    """The module with the native node, and the address of the gradient it calls."""
    global _NATIVE
    if _NATIVE is None:
        _NATIVE = _lib.native(), ctypes.cast(_lib.lib().fs_small_grad, _P).value
    return _NATIVE


def loss(module, x, y, a, b, normalize):
    given = [x, y, a, b]
    native, grad = _native()
    if torch._C._are_functorch_transforms_active() or not native.ordinary(given):
        return _SmallLoss.apply(x, y, a, b, module, normalize)
    need = [torch.is_grad_enabled() and t is not None and t.requires_grad for t in given]
    s = _solve_for(module, x, y, a, b, normalize, self_terms=int(module.debias),
                   want_values=need[0] or need[1], want_loss=True)
    if True not in need:
        return s.loss
    # (the settings as they are now, for a second backward pass)
    return native.attach(s.loss, a, b, [x, y, *s.tensors()], ctypes.addressof(s.form), ctypes.sizeof(s.form), grad,
                         _Ask(s.form, dict(vars(module))))
