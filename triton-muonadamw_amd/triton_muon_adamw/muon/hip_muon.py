"""Muon branch on the gfx950 kernels.

Drop-in for the reference's ``TritonMuon`` (muon/triton_muon.py:375-456) and its
launchers ``solve_ns_kernel_{1,2,3}`` (:95-117, :191-212, :281-310),
``newton_shultz_step`` (:313-325) and ``muon_step`` (:327-372).

``HipMuon.step()`` groups the matrices that have a gradient by
``(min(R,C), max(R,C))`` and runs each group as batched launches of
``mamw_muon_step`` (at most 32 matrices and a bounded workspace per call):
prep (momentum, Nesterov, bf16, transpose, sum of squares), norm, scale
(``X / ||X||`` in bf16 and its transpose), then per Newton-Schulz iteration a
Gram, a polynomial and an update GEMM, the last of which writes the
parameters.  The reference runs about 30 launches per matrix; here a group of
up to 32 matrices costs ``3 + 3*ns_steps`` launches.  Few small matrices, of
any shapes, go out together on the direct path instead (``direct_pays``,
``direct_set_pays``): ``2 + 3*ns_steps`` launches for up to 64 of them.
Small steps (``HipMuon.concurrent_flops_limit``) run the shape groups
concurrently on side streams forked from and joined back into the caller's
current stream; the results are the same bits as in order.

Semantics kept from the reference: the constructor signature and defaults,
``AssertionError`` for an unknown ``adjust_lr_fn`` (:392-393) and for a
non-2-D parameter at step time (:96-97), momentum buffers shaped like the
parameter (:407-412), ``grad is None`` skipped (:420-421), zero-filling
``zero_grad`` (:450-456), and weight decay with the unscaled ``lr`` (:370).
The numerics follow torch.optim.Muon (the reference's own correctness oracle):
see ``include/muonadamw_amd.h``.  Differences from the reference, each
matching torch: ``match_rms_adamw`` scales by ``0.2*sqrt(max(R,C))`` (the
reference raises ``TypeError``, :428) and ``ns_steps=0`` applies the
normalised momentum (the reference still runs one iteration, :360).
"""

from __future__ import annotations

import ctypes
import functools
import math
import os
from collections.abc import Iterable
from typing import Literal

import torch
import torch.nn as nn
from torch.autograd import forward_ad

from .. import _lib

_ADJUST_FNS = ["original", "match_rms_adamw", "spectral_unclamped"]


def scaled_lr(lr: float, adjust_lr_fn: str, rows: int, cols: int) -> float:
    """Shape-dependent Muon learning rate (triton_muon.py:424-431; torch/optim/_muon.py:73-84)."""
    if adjust_lr_fn == "original":
        return lr * math.sqrt(max(1, rows / cols))
    if adjust_lr_fn == "match_rms_adamw":
        return lr * (0.2 * math.sqrt(max(rows, cols)))
    return lr * math.sqrt(rows / cols)


def _check_matrix(t: torch.Tensor, name: str, dtype=torch.float32, bf16_ok: bool = False) -> None:
    _lib.require_gpu_tensor(t, name)
    if t.dtype != dtype and not (bf16_ok and t.dtype == torch.bfloat16):
        raise TypeError(f"{name} must be {dtype}{' or torch.bfloat16' if bf16_ok else ''} (got {t.dtype})")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


def _workspace_bytes(batch: int, rows: int, cols: int, ns_steps: int) -> int:
    n = ctypes.c_size_t()
    _lib.check(_lib.load().mamw_muon_workspace_bytes(batch, rows, cols, ns_steps, ctypes.byref(n)),
               "mamw_muon_workspace_bytes")
    return n.value


def _direct_workspace_bytes(arr, count: int, ns_steps: int) -> int:
    n = ctypes.c_size_t()
    _lib.check(_lib.load().mamw_muon_direct_workspace_bytes(arr, count, ns_steps, ctypes.byref(n)),
               "mamw_muon_direct_workspace_bytes")
    return n.value


# ---------------------------------------------------------------------------
# Which kernels a launch group takes: the LDS-staged tiles (mamw_muon_step) or
# the direct path (mamw_muon_direct_step, one wavefront per 32- or 64-wide
# tile), the same bits either way.  Both times are estimated in microseconds
# per step (five iterations) with constants fitted to 460 measured pairs on one
# MI355X (16 <= m <= 4096, n up to 16 m, 1 to 32 matrices), before the direct
# stores were written through and the staged last rounds split, which the
# staged estimate has a term for.  Against 130 pairs of the kernels as they are
# now: rms error 9% staged, 11% direct; the choice lost over 6% (at most 27%) in
# 12 of them, each a staged launch that the direct path would have beaten.
# Measured on both sides (staged / direct): 512 x 2048 one matrix 195 / 96, two
# 198 / 109, eight 240 / 219, sixteen 339 / 372; 768 x 3072 one 268 / 143, eight
# 443 / 512; 2048 x 2048 one 347 / 307, four 782 / 1036.

def _staged_product_us(tile: int, tiles: int, k: int, cus: int, split: bool, sym: bool = False,
                       large: bool = False) -> float:
    """One staged product: whole rounds of its grid (one 256-wide or two
    128-wide workgroups per CU; a 128-wide workgroup alone on its CU is
    faster), a k step of 64 at 1.33, 0.88 or 0.50 us, and 3.5 us a launch.
    ``split``: k-blocked operands (a step's; those of the standalone products
    are row-major), whose last round of few 256-wide tiles runs as 128-wide
    ones; how few, by ``sym`` and ``large`` (m >= 2048) (launch_gemm)."""
    if tile == 256:
        full, rest = divmod(tiles, cus)
        if split and 0 < rest <= 64:
            last = 0.50
        elif split and 0 < rest <= 128 and (sym if full else large):
            last = 0.88
        else:
            last = 1.33 if rest else 0.0
        rounds = full * 1.33 + last
    else:
        full, rest = divmod(tiles, 2 * cus)
        rounds = full * 0.88 + (0.0 if rest == 0 else 0.50 if rest <= cus else 0.88)
    return rounds * (k / 64) + 3.5


def _direct_product_us(t64: int, t32: int, k: int, nbytes64: float, nbytes32: float) -> float:
    """One direct product of ``t64`` 64-wide (or ``t32`` 32-wide) tiles: 3.1 us,
    0.14 us (0.035 us) per k step of 64 of its longest reduction ``k``, and the
    operand bytes of all tiles at 26 TB/s (L2)."""
    wide = t64 >= 384  # kDirectWideTiles
    return 3.1 + (k / 64) * (0.14 if wide else 0.035) + (nbytes64 if wide else nbytes32) / 26e6


def _staged_us(m: int, n: int, count: int, cus: int) -> float:
    """A step of ``count`` m x n matrices on the staged path."""
    tile = gemm_tile(m, n, count)
    mp, np_ = _rup(m, tile), _rup(n, tile)
    utile = 256 if (tile == 128 and m >= 1024 and mp % 256 == 0 and np_ % 256 == 0) else tile
    tm = mp // tile
    sym = count * tm * (tm + 1) // 2
    large = mp >= 2048
    return (5 * (_staged_product_us(tile, sym, np_, cus, True, True, large)
                 + _staged_product_us(tile, sym, mp, cus, True, True, large)
                 + _staged_product_us(utile, count * (mp // utile) * (np_ // utile), mp, cus, True, False, large))
            + 8e-6 * count * mp * np_ + 12)


def _direct_us(groups) -> float:
    """A step on the direct path, one launch of all ``groups`` (m, n, count)."""
    pads = [(_rup(m, 64), _rup(n, 64), count) for m, n, count in groups]

    def product(tiles, k):  # tiles(mp, np, tile edge), k(mp, np)
        t64, t32 = (sum(c * tiles(mp, np_, t) for mp, np_, c in pads) for t in (64, 32))
        b64, b32 = (sum(c * tiles(mp, np_, t) * 4.0 * t * k(mp, np_) for mp, np_, c in pads) for t in (64, 32))
        return _direct_product_us(t64, t32, max(k(mp, np_) for mp, np_, _ in pads), b64, b32)

    sym = lambda mp, np_, t: (mp // t) * (mp // t + 1) // 2  # noqa: E731
    upd = lambda mp, np_, t: (mp // t) * (np_ // t)  # noqa: E731
    return (5 * (product(sym, lambda mp, np_: np_) + product(sym, lambda mp, np_: mp)
                 + product(upd, lambda mp, np_: mp)) + 7.6e-6 * sum(c * mp * np_ for mp, np_, c in pads) + 12)


def _direct_fits(m: int, n: int, ns_steps: int) -> bool:
    """The direct path's limits for one m x n (or n x m) matrix."""
    return (ns_steps >= 1 and _rup(m, 64) * _rup(n, 64) <= 1 << 26 and _rup(m, 128) * _rup(n, 128) <= 1 << 26)


@functools.lru_cache(maxsize=4096)
def direct_pays(rows: int, cols: int, count: int, cus: int, ns_steps: int) -> bool:
    """Whether a group of ``count`` rows x cols matrices, run by itself, takes
    the direct path: where its estimate is a tenth below the staged path's (the
    estimates' error is as large, and the direct path's workspace is larger by
    X)."""
    m, n = min(rows, cols), max(rows, cols)
    return (_direct_fits(m, n, ns_steps)
            and _direct_us(((m, n, count),)) < 0.9 * _staged_us(m, n, count, cus))


@functools.lru_cache(maxsize=1024)
def direct_set_pays(groups: tuple, cus: int, ns_steps: int, launches: int = 0) -> bool:
    """Whether shape classes that may run beside each other (``groups``: a
    tuple of (m, n, count)) go out as direct launches of all of them
    (``launches`` of them; 0: as many as MUON_DIRECT_MAX matrices each make),
    instead of staged groups on their own streams: all or none, since a staged class fills the GPU and a direct one
    beside it costs more than its staged form would (1024-2048-4096-4096-1024
    MLP: 1748 us all staged, 2031 with its three smaller classes direct).
    Staged classes on streams take about 1.15 times their longest class, 0.6
    of their sum, or 95 us of host time each, whichever is most."""
    if not all(_direct_fits(m, n, ns_steps) for m, n, _ in groups):
        return False
    staged = [_staged_us(m, n, count, cus) for m, n, count in groups]
    launches = max(launches, -(-sum(count for _, _, count in groups) // _lib.MUON_DIRECT_MAX))
    direct = _direct_us(groups) + (launches - 1) * 60
    return direct < 0.9 * max(1.15 * max(staged), 0.6 * sum(staged), 95.0 * len(groups))


# ---------------------------------------------------------------------------
# Standalone launchers (bf16 matrices).  The kernels need dimensions padded to
# multiples of 128 (reduction length: 64); inputs that are not are copied into
# zero-padded buffers, which leaves every product unchanged.

def _padded(x: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    if x.shape == (rows, cols) and x.is_contiguous():
        return x
    out = torch.zeros((rows, cols), dtype=x.dtype, device=x.device)
    out[: x.shape[0], : x.shape[1]] = x
    return out


def _rup(x: int, to: int) -> int:
    return (x + to - 1) // to * to


def _check_bf16_2d(x: torch.Tensor, name: str) -> None:
    if x.ndim != 2:
        raise AssertionError("Muon only supports 2D tensors")
    _lib.require_gpu_tensor(x, name)
    if x.dtype != torch.bfloat16:
        raise TypeError(f"{name} must be bfloat16 (got {x.dtype})")


_PLAIN = (torch.Tensor, nn.Parameter)  # no attributes or copies of their own
_NS_GRAM, _NS_POLY, _NS_UPDATE, _NS_STEP = range(4)  # MAMW_NS_*


@functools.lru_cache(maxsize=4096)
def ns_direct_pays(op: int, m: int, n: int, cus: int) -> bool:
    """Whether a standalone product takes the direct path: the estimates of its
    products (those of the steps above; here a last round is never split), and
    what each path does around them: packing (5 us) there; the copy into
    ``out``, for the update and the iteration a transpose, and padding here.
    Measured staged / direct, us: Gram of 1024 x 4096 41 / 23, 1531 x 3001 52 /
    31, 2304 x 4096 80 / 47, 2560 x 8192 140 / 99, 4096 x 4096 89 / 123;
    polynomial of 1024 17 / 12, 2304 58 / 33, 2560 67 / 38, 3072 73 / 56, 4096
    92 / 123; update of 768 x 3001 39 / 21, 2048 x 2048 59 / 34, 2048 x 8192 89 /
    103; iteration of 512 x 512 35 / 17, 1024 x 4096 82 / 41, 2304 x 4096 203 /
    131, 4096 x 4096 292 / 393."""
    if max(_rup(m, 64) * _rup(n, 64), _rup(m, 64) ** 2) > 1 << 26:
        return False
    mp, np_ = _rup(m, 128), _rup(n, 128)
    tile = 256 if mp >= 2048 and mp % 256 == 0 else 128  # the products see padded matrices
    utile = tile if np_ % 256 == 0 else 128
    sym = (mp // tile) * (mp // tile + 1) // 2
    d, e = _rup(m, 64), _rup(n, 64)
    r, r2 = d // 64, d // 32
    s64, s32 = r * (r + 1) // 2, r2 * (r2 + 1) // 2
    u64, u32 = r * (e // 64), r2 * (e // 32)
    products = {
        _NS_GRAM: (_staged_product_us(tile, sym, np_, cus, False),
                   _direct_product_us(s64, s32, e, s64 * 256.0 * e, s32 * 128.0 * e)),
        _NS_POLY: (_staged_product_us(tile, sym, mp, cus, False),
                   _direct_product_us(s64, s32, d, s64 * 256.0 * d, s32 * 128.0 * d)),
        _NS_UPDATE: (_staged_product_us(utile, (mp // utile) * (np_ // utile), mp, cus, False),
                     _direct_product_us(u64, u32, d, u64 * 256.0 * d, u32 * 128.0 * d)),
    }
    staged = direct = 5.0
    for k in (_NS_GRAM, _NS_POLY, _NS_UPDATE) if op == _NS_STEP else (op,):
        staged, direct = staged + products[k][0], direct + products[k][1]
    if op >= _NS_UPDATE:
        staged += 4 + 1.5e-6 * mp * np_
    return direct < 0.95 * staged


def _ns_direct(op: int, X: torch.Tensor, S, out: torch.Tensor, a: float, b: float, c: float) -> bool:
    """The product on the direct path, straight into ``out``; False where it
    stays with the padded, staged one: inputs or an output that are not plain
    contiguous bf16 matrices of the right shape on one device (copies there
    handle any strides, types, subclasses and broadcasts, and refuse what
    autograd must refuse), an output with a forward-mode tangent (which the
    copy clears), 16-byte misaligned inputs (which it refuses unless it pads
    them), and sizes where it is the faster one."""
    if type(X) not in _PLAIN or type(out) not in _PLAIN or S is not None and type(S) not in _PLAIN:
        return False
    if forward_ad._current_level >= 0 and forward_ad.unpack_dual(out).tangent is not None:
        return False
    m, n = X.shape
    shape = (m, m) if op in (_NS_GRAM, _NS_POLY) else (m, n)
    if (m < 1 or n < 1 or out.dtype != torch.bfloat16 or out.shape != shape or out.device != X.device
            or not out.is_contiguous() or out.requires_grad or out.is_inference()):
        return False
    for t in (X,) if S is None else (X, S):
        if not t.is_contiguous() or t.data_ptr() % 16 or t.device != X.device:
            return False
    if S is not None and S.shape != (m, m) or op == _NS_POLY and n != m:
        return False
    dev = X.device
    if not ns_direct_pays(op, m, n, torch.cuda.get_device_properties(dev).multi_processor_count):
        return False
    lib = _lib.load()
    nbytes = ctypes.c_size_t()
    _lib.check(lib.mamw_ns_direct_workspace_bytes(m, n, ctypes.byref(nbytes)), "mamw_ns_direct_workspace_bytes")
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device=dev)
    with _lib.device_guard(dev):
        st = lib.mamw_ns_direct(op, X.data_ptr(), S.data_ptr() if S is not None else None, out.data_ptr(), m, n, a, b,
                                c, ws.data_ptr(), nbytes.value, _lib.raw_stream(dev))
    _lib.check(st, "mamw_ns_direct")
    torch.autograd.graph.increment_version(out)  # written in place, as copy_ records
    return True


def solve_ns_kernel_1(matrix: torch.Tensor, out: torch.Tensor) -> None:
    """out = matrix @ matrix.T for a bf16 m x k matrix (triton_muon.py:95-117)."""
    _check_bf16_2d(matrix, "matrix")
    if _ns_direct(_NS_GRAM, matrix, None, out, 0.0, 0.0, 0.0):
        return
    m, k = matrix.shape
    mp, kp = _rup(m, 128), _rup(k, 64)
    X = _padded(matrix, mp, kp)
    A = torch.empty((mp, mp), dtype=torch.bfloat16, device=matrix.device)
    lib = _lib.load()
    with torch.cuda.device(matrix.device):
        st = lib.mamw_ns_gram(X.data_ptr(), A.data_ptr(), 1, mp, kp, _lib.stream_handle(matrix.device))
    _lib.check(st, "mamw_ns_gram")
    out.copy_(A[:m, :m])


def solve_ns_kernel_2(matrix: torch.Tensor, b: float, c: float, out: torch.Tensor) -> None:
    """out = b*A + c*(A @ A.T) for a symmetric bf16 m x m matrix A (triton_muon.py:191-212)."""
    _check_bf16_2d(matrix, "matrix")
    if _ns_direct(_NS_POLY, matrix, None, out, 0.0, b, c):
        return
    m = matrix.shape[0]
    mp = _rup(m, 128)
    A = _padded(matrix, mp, mp)
    B = torch.empty((mp, mp), dtype=torch.bfloat16, device=matrix.device)
    lib = _lib.load()
    with torch.cuda.device(matrix.device):
        st = lib.mamw_ns_poly(A.data_ptr(), B.data_ptr(), 1, mp, b, c, _lib.stream_handle(matrix.device))
    _lib.check(st, "mamw_ns_poly")
    out.copy_(B[:m, :m])


def _transpose(x: torch.Tensor) -> torch.Tensor:
    r, c = x.shape
    t = torch.empty((c, r), dtype=x.dtype, device=x.device)
    with torch.cuda.device(x.device):
        st = _lib.load().mamw_transpose_bf16(x.data_ptr(), t.data_ptr(), 1, r, c,
                                             _lib.stream_handle(x.device))
    _lib.check(st, "mamw_transpose_bf16")
    return t


def solve_ns_kernel_3(X: torch.Tensor, out_2: torch.Tensor, a: float, out: torch.Tensor) -> None:
    """out = a*X + out_2 @ X for bf16 X (m x n) and symmetric out_2 (m x m) (triton_muon.py:281-310)."""
    _check_bf16_2d(X, "X")
    _check_bf16_2d(out_2, "out_2")
    if _ns_direct(_NS_UPDATE, X, out_2, out, a, 0.0, 0.0):
        return
    m, n = X.shape
    mp, np_ = _rup(m, 128), _rup(n, 128)
    Xp = _padded(X, mp, np_)
    Bp = _padded(out_2, mp, mp)
    XT = _transpose(Xp)
    O = torch.empty((mp, np_), dtype=torch.bfloat16, device=X.device)
    lib = _lib.load()
    with torch.cuda.device(X.device):
        st = lib.mamw_ns_update(Bp.data_ptr(), Xp.data_ptr(), XT.data_ptr(), O.data_ptr(), None, 1, mp, np_,
                                a, _lib.stream_handle(X.device))
    _lib.check(st, "mamw_ns_update")
    out.copy_(O[:m, :n])


def newton_shultz_step(X: torch.Tensor, a: float, b: float, c: float, out: torch.Tensor) -> None:
    """One Newton-Schulz iteration out = a*X + (b*A + c*A@A) @ X, A = X @ X.T (triton_muon.py:313-325)."""
    _check_bf16_2d(X, "X")
    if _ns_direct(_NS_STEP, X, None, out, a, b, c):
        return
    m, n = X.shape
    mp, np_ = _rup(m, 128), _rup(n, 128)
    dev = X.device
    Xp = _padded(X, mp, np_)
    XT = _transpose(Xp)
    A = torch.empty((mp, mp), dtype=torch.bfloat16, device=dev)
    B = torch.empty((mp, mp), dtype=torch.bfloat16, device=dev)
    O = torch.empty((mp, np_), dtype=torch.bfloat16, device=dev)
    lib = _lib.load()
    with torch.cuda.device(dev):
        s = _lib.stream_handle(dev)
        _lib.check(lib.mamw_ns_gram(Xp.data_ptr(), A.data_ptr(), 1, mp, np_, s), "mamw_ns_gram")
        _lib.check(lib.mamw_ns_poly(A.data_ptr(), B.data_ptr(), 1, mp, b, c, s), "mamw_ns_poly")
        _lib.check(lib.mamw_ns_update(B.data_ptr(), Xp.data_ptr(), XT.data_ptr(), O.data_ptr(), None, 1, mp,
                                      np_, a, s), "mamw_ns_update")
    out.copy_(O[:m, :n])


def muon_step(weights: torch.Tensor, grad: torch.Tensor, momentum: torch.Tensor, beta: float, a: float,
              b: float, c: float, lr: float, scaled_lr: float, weight_decay: float, steps: int, eps: float,
              nesterov: bool, out: torch.Tensor | None = None) -> None:
    """One Muon update of one matrix in place (triton_muon.py:327-372).

    ``out`` (optional, fp32, shaped like ``weights``) receives the
    orthogonalised update, as the reference's ``out`` buffer does (:368).
    """
    if weights.ndim != 2:
        raise AssertionError("Muon only supports 2D tensors")
    for t, name in ((weights, "weights"), (grad, "grad"), (momentum, "momentum")):
        _check_matrix(t, name)
        if t.shape != weights.shape or t.device != weights.device:
            raise ValueError(f"{name} must match the weights' shape and device")
    if out is not None:
        _check_matrix(out, "out")
        if out.shape != weights.shape or out.device != weights.device:
            raise ValueError("out must match the weights' shape and device")
    R, C = weights.shape
    arr = (_lib.MuonMatrix * 1)()
    arr[0] = _lib.MuonMatrix(weights.data_ptr(), grad.data_ptr(), momentum.data_ptr(),
                             out.data_ptr() if out is not None else None, R, C, scaled_lr, 0)
    lib = _lib.load()
    cus = torch.cuda.get_device_properties(weights.device).multi_processor_count
    direct = direct_pays(R, C, 1, cus, steps)
    nbytes = _direct_workspace_bytes(arr, 1, steps) if direct else _workspace_bytes(1, R, C, steps)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=weights.device)
    args = (arr, 1, lr, weight_decay, beta, int(bool(nesterov)), a, b, c, steps, eps, ws.data_ptr(), nbytes)
    with _lib.device_guard(weights.device):
        s = _lib.raw_stream(weights.device)
        st = lib.mamw_muon_direct_step(*args, None, None, s) if direct else lib.mamw_muon_step(*args, s)
    _lib.check(st, "mamw_muon_step")


def gemm_tile(m: int, n: int, batch: int) -> int:
    """The library's GEMM tile edge for a launch group (``mamw_plan.cpp``
    ``choose_tile``): 256 from m = 2048; from m = 1024 for batches of 8 or
    more when the 256 padding adds at most 1/16 to the 128 padding; else 128."""
    if m >= 2048:
        return 256
    rup = lambda x, t: -(-x // t) * t  # noqa: E731
    if m >= 1024 and batch >= 8 and rup(m, 256) * rup(n, 256) * 16 <= rup(m, 128) * rup(n, 128) * 17:
        return 256
    return 128


def group_sizes(count: int, cap: int, m: int, n: int, cus: int) -> list[int]:
    """Sizes of the launch groups for ``count`` matrices of one shape class
    (``m = min(R, C)``, ``n = max(R, C)``), each at most ``cap``.

    Every group runs its Gram, polynomial and update GEMMs as one grid each,
    and a grid whose workgroups do not fill whole rounds of the GPU's CU slots
    leaves CUs idle in its last round.  The cost of a group of k matrices is
    modelled as each product's rounds times its reduction length (Gram: n,
    polynomial and update: m) times the relative time of one k step of its
    tile (a 256 x 256 step, one workgroup per CU, counts 1.4 steps of the
    128 x 128 tile, two workgroups per CU), plus a quarter round of each
    product per group for its launches.  The cheapest split into groups of any
    sizes wins (ties: fewer groups), found by dynamic programming over the
    number of matrices covered.  Tiles follow the library's choice for the
    group's size (``gemm_tile``), and a group on the 128 tile takes 256 x 256
    updates from m = 1024 when both padded edges are multiples of 256.

    The model counts whole rounds; a last round of few 256-wide tiles costs
    less, since it runs as 128-wide ones (launch_gemm).  Measured for 64 of
    1024 x 4096: [24, 24, 16], its choice, 5842 us; [32, 32], whose 320
    symmetric tiles are split after a round, 6006.
    """
    if count <= 0:
        return []
    cap = max(1, min(cap, count))
    step = {128: 1.0, 256: 1.4}

    def cost(k: int) -> float:
        tile = gemm_tile(m, n, k)
        mp, np_ = -(-m // tile) * tile, -(-n // tile) * tile
        utile = 256 if (tile == 128 and m >= 1024 and mp % 256 == 0 and np_ % 256 == 0) else tile
        tm = mp // tile
        sym, upd = tm * (tm + 1) // 2, (mp // utile) * (np_ // utile)
        rounds = lambda tiles, t: -(-tiles * k // (cus * (1 if t == 256 else 2)))  # noqa: E731
        return (rounds(sym, tile) * step[tile] * (n + m) + rounds(upd, utile) * step[utile] * m
                + 0.25 * (step[tile] * (n + m) + step[utile] * m))

    # best[c]: (cost, number of groups, sizes) of the cheapest split of c matrices
    best: list = [(0.0, 0, [])] + [None] * count
    for c in range(1, count + 1):
        for k in range(1, min(cap, c) + 1):
            pc, pg, ps = best[c - k]
            cand = (pc + cost(k), pg + 1, ps + [k])
            cur = best[c]
            if cur is None or cand[0] < cur[0] - 1e-9 or (abs(cand[0] - cur[0]) <= 1e-9 and cand[1] < cur[1]):
                best[c] = cand
    return sorted(best[count][2], reverse=True)


def _launch_rounds(tiles: int, tile: int, k: int, cus: int) -> float:
    """Time of one GEMM launch in k steps of a 256-wide tile: whole rounds of
    the grid (two 128-wide workgroups per CU, a quarter of the work each); a
    last round that runs split (launch_gemm) counts whole here."""
    slots = cus * (2 if tile == 128 else 1)
    return math.ceil(tiles / slots) * (k / 64) * (1.0 if tile == 256 else 0.5)


def _class_time(calls, key, steps: int, cus: int) -> float:
    """Estimated Newton-Schulz time of one shape class (its launch groups one
    after another): a launch whose grid fills a fraction of the GPU still
    takes a round, which is what makes a class of small grids slow for its
    flops."""
    t = 0.0
    for c in calls:
        if (c.device, c.group) != key:
            continue
        tile = gemm_tile(c.m, c.n_, c.n)
        mp, np_ = -(-c.m // tile) * tile, -(-c.n_ // tile) * tile
        tm = mp // tile
        sym = c.n * tm * (tm + 1) // 2  # Gram and polynomial tiles (lower triangle)
        utile = 256 if (tile == 128 and c.m >= 1024 and mp % 256 == 0 and np_ % 256 == 0) else tile
        upd = c.n * (mp // utile) * (np_ // utile)
        t += steps * (_launch_rounds(sym, tile, np_, cus) + _launch_rounds(sym, tile, mp, cus)
                      + _launch_rounds(upd, utile, mp, cus))
    return t


def _lanes(calls, steps: int, cus: dict) -> tuple[dict, dict]:
    """Streams of concurrent shape classes, per device, and each class's
    estimated time (_class_time).  The longest class runs on the caller's
    stream (None); the others, longest first, each on the least loaded of
    L - 1 side streams of the library's own (_lib.side_streams), where a side
    stream's classes run one after another.  L is the fewest lanes (2 to 4)
    whose side streams all finish within the caller's class; more concurrent
    streams than that only contend.  Measured: config 3 (the 4096 x 14336
    class against four smaller ones) 4.91 ms with two lanes against 5.01 with
    one side stream per class; GPT-2 1.80 against 1.81; the reference's hybrid
    MLP (four batch-1 classes whose grids mostly underfill the GPU) needs
    three."""
    lanes: dict = {}
    times: dict = {}
    for dev in dict.fromkeys(c.device for c in calls):
        keys = list(dict.fromkeys((c.device, c.group) for c in calls if c.device == dev))
        for k in keys:
            times[k] = _class_time(calls, k, steps, cus[dev])
        keys.sort(key=lambda k: times[k], reverse=True)
        lanes[keys[0]] = None
        rest = keys[1:]
        if not rest:
            continue
        n_side, pick = _lane_split([times[k] for k in keys])
        streams = _lib.side_streams(dev, n_side)
        for k, i in zip(rest, pick):
            lanes[k] = streams[i]
    return lanes, times


def _lane_split(times: list[float]) -> tuple[int, list[int]]:
    """The side-stream split of _lanes for class times sorted longest first:
    the first class stays on the caller's stream; returns the number of side
    streams (1 to 3) and, for each later class, the side stream it joins (the
    least loaded so far).  The fewest side streams whose loads all fit within
    the first class's time; three when none does."""
    rest = times[1:]
    for n_side in range(1, min(3, len(rest)) + 1):
        load = [0.0] * n_side
        pick = []
        for t in rest:
            i = min(range(n_side), key=lambda j: load[j])
            load[i] += t
            pick.append(i)
        if max(load) <= times[0]:
            break
    return n_side, pick


class _Call:
    """One launch group (matrices of one shape class)."""

    __slots__ = ("device", "arr", "n", "ws_bytes", "m", "n_", "group", "direct")

    def __init__(self, device, arr, n, ws_bytes, m, n_, group, direct=False):
        self.device, self.arr, self.n, self.ws_bytes, self.m, self.n_ = device, arr, n, ws_bytes, m, n_
        self.group = group  # index of the shape class (device, m, n)
        self.direct = direct  # mamw_muon_direct_step (else mamw_muon_step)


class _Launch:
    """One library call: a launch group, or several direct-path groups together."""

    __slots__ = ("device", "arr", "n", "direct", "lane", "ws_key")

    def __init__(self, device, arr, n, direct, lane, ws_key):
        self.device, self.arr, self.n, self.direct, self.lane, self.ws_key = device, arr, n, direct, lane, ws_key


def _disjoint(calls) -> bool:
    """Whether no memory that one matrix of ``calls`` writes (parameter,
    momentum) is read or written by another: one launch may run them at once."""
    spans = []
    for c in calls:
        for e in c.arr:
            ne = e.rows * e.cols
            spans.append((e.param, e.param + ne * (2 if e.flags & _lib.BF16_PARAM else 4), True))
            spans.append((e.momentum, e.momentum + ne * 4, True))
            spans.append((e.grad, e.grad + ne * (2 if e.flags & _lib.BF16_GRAD else 4), False))
    spans.sort()
    end_any = end_write = 0
    for lo, hi, write in spans:
        if lo < (end_any if write else end_write):
            return False
        end_any = max(end_any, hi)
        if write:
            end_write = max(end_write, hi)
    return True


def _entries(calls):
    """The matrices of ``calls`` as one array."""
    return (_lib.MuonMatrix * sum(c.n for c in calls))(*[e for c in calls for e in c.arr])


def _merge(calls, ns_steps: int = 1, limit: int | None = None) -> list[list]:
    """Direct-path ``calls`` as the runs that go out as one launch each: in
    order, at most MUON_DIRECT_MAX matrices and ``limit`` bytes of workspace,
    no memory in common.  (A class's later groups may hold a parameter of an
    earlier one again.)"""
    def fits(run):
        n = sum(c.n for c in run)
        return (n <= _lib.MUON_DIRECT_MAX and _disjoint(run)
                and (limit is None or _direct_workspace_bytes(_entries(run), n, ns_steps) <= limit))

    runs: list[list] = []
    for c in calls:
        last = runs[-1] if runs else None
        if last is not None and fits(last + [c]):
            last.append(c)
        else:
            runs.append([c])
    return runs


class HipMuon:
    """Muon over a list of 2-D parameters, batched by shape on gfx950."""

    # Workspace per launch is capped at this many bytes, except that one matrix
    # takes what the staged path needs for it (None: 1/20 of the device's
    # memory, at most 16 GiB; on a 288 GB MI355X 14.4 GB, which
    # lets the 4096 x 14336 Llama-8B matrices run in groups of 32 whose
    # symmetric grids fill whole rounds of the 256 CUs: 3 ms per step faster
    # than groups of 20).  Within the cap, group_sizes() picks the split; a
    # group whose direct workspace is over it stays staged.
    workspace_limit_bytes: int | None = None
    # A step whose Newton-Schulz work (sum of ns_steps*(3 m^2 n + m^3)) is at
    # most this many flops runs its shape classes concurrently (lanes from
    # _lanes, one workspace per class): their launches are too small to fill
    # the GPU one after another (measured: GPT-2 Muon step -10%, config-3
    # -17%).  Larger steps run the classes in order, which keeps each class's
    # operands in the L2 and memory-side cache.  Measured on the first L
    # layers of the Llama-8B set, concurrent against in order: L = 1 (1.4e13)
    # 13.19 vs 14.10 ms, L = 2 (3.0e13) 26.46 vs 26.73, L = 4 (5.9e13) 52.72 vs
    # 52.10, L = 8 (1.2e14) 105.9 vs 102.9, all 32 layers 405 vs 391.
    concurrent_flops_limit = 4e13

    def __init__(
        self,
        params: Iterable[nn.Parameter] | list[nn.Parameter],
        lr: float = 1e-3,
        weight_decay: float = 0.1,
        coeffs: tuple[float, float, float] = (3.445, -4.775, 2.0315),
        nesterov: bool = True,
        beta: float = 0.95,
        ns_steps: int = 5,
        eps: float = 1e-7,
        adjust_lr_fn: Literal["original", "match_rms_adamw", "spectral_unclamped"] = "original",
    ):
        if adjust_lr_fn not in _ADJUST_FNS:
            raise AssertionError(f"Invalid adjust_lr_fn: {adjust_lr_fn}")
        self.model_params = list(params)
        self.a = coeffs[0]
        self.b = coeffs[1]
        self.c = coeffs[2]
        self.is_nesterov = nesterov
        self.beta = beta
        self.lr = lr
        self.adjust_lr_fn = adjust_lr_fn
        self.weight_decay = weight_decay
        self.steps = ns_steps
        self.eps = eps
        self.momentum = {}
        for param in self.model_params:
            self._momentum(param)
        self._plan_key = None
        self._plan_lr = lr
        self._calls: list[_Call] = []
        self._launches: list[_Launch] = []
        self._ws: dict = {}  # device (launches in order) or (device, shape class) (own streams) -> workspace
        self._ws_home: dict = {}  # same keys -> handle of the stream the workspace's memory belongs to
        self._concurrent = False
        # (device, shape class) -> side stream, or None: the caller's stream (of a staged class)
        self._lanes: dict = {}

    def _momentum(self, param: nn.Parameter) -> torch.Tensor:
        """The momentum buffer of ``param``, created (zero) on first use: at
        construction, or for a parameter that joined ``model_params`` later
        (a parameter list loaded in the reference's state format).  fp32 also
        for bf16 parameters (the reference uses the parameter's dtype,
        :407-412)."""
        buf = self.momentum.get(param)
        if buf is None:
            buf = self.momentum[param] = torch.zeros_like(param, device=param.device, dtype=torch.float32)
        return buf

    def _workspace_limit(self, device: torch.device) -> int:
        if self.workspace_limit_bytes is not None:
            return self.workspace_limit_bytes
        return min(16 << 30, torch.cuda.get_device_properties(device).total_memory // 20)

    def _build_calls(self, active: list[nn.Parameter]) -> None:
        groups: dict[tuple, list[nn.Parameter]] = {}
        for p in active:
            if p.ndim != 2:
                raise AssertionError("Muon only supports 2D tensors")
            g = p.grad
            _check_matrix(p, "param", bf16_ok=True)
            _check_matrix(g, "param.grad", bf16_ok=True)
            if g.shape != p.shape or g.device != p.device:
                raise ValueError("param.grad must match the parameter's shape and device")
            _check_matrix(self._momentum(p), "momentum")
            if self.momentum[p].shape != p.shape:
                raise ValueError(f"momentum buffer of shape {tuple(self.momentum[p].shape)} for a parameter of "
                                 f"shape {tuple(p.shape)}")
            R, C = p.shape
            groups.setdefault((p.device, min(R, C), max(R, C)), []).append(p)
        calls = []
        flops = sum(self.steps * (3.0 * m * m * n + float(m) ** 3) * len(pl) for (_, m, n), pl in groups.items())
        concurrent = len(groups) > 1 and flops <= self.concurrent_flops_limit
        limits = {dev: self._workspace_limit(dev) for dev, _, _ in groups}
        for gi, ((dev, m, n), plist) in enumerate(groups.items()):
            one = _workspace_bytes(1, m, n, self.steps)
            cap = max(1, min(_lib.MUON_MAX_BATCH, limits[dev] // max(one, 1)))
            cus = torch.cuda.get_device_properties(dev).multi_processor_count
            sizes = iter(group_sizes(len(plist), cap, m, n, cus))
            per = next(sizes)
            chunks, cur, seen = [], [], set()
            for p in plist:  # a parameter listed twice goes to a later launch (launches are ordered)
                if len(cur) == per or id(p) in seen:
                    chunks.append(cur)
                    cur, seen = [], set()
                    per = next(sizes, per)
                cur.append(p)
                seen.add(id(p))
            chunks.append(cur)
            for chunk in chunks:
                arr = (_lib.MuonMatrix * len(chunk))()
                for i, p in enumerate(chunk):
                    R, C = p.shape
                    flags = (_lib.dtype_flag(p, _lib.BF16_PARAM, "param")
                             | _lib.dtype_flag(p.grad, _lib.BF16_GRAD, "param.grad"))
                    arr[i] = _lib.MuonMatrix(p.data_ptr(), p.grad.data_ptr(), self.momentum[p].data_ptr(), None,
                                             R, C, scaled_lr(self.lr, self.adjust_lr_fn, R, C), flags)
                calls.append(_Call(dev, arr, len(chunk), 0, m, n, gi))
        # The kernels: all of a device's concurrent classes direct or none (then
        # as few launches as hold them), a class that runs by itself as it
        # pays.  Concurrent classes longest first (a class's own launches keep
        # their order: stable sort), the staged ones on streams.
        def fits(c):
            return (_direct_fits(c.m, c.n_, self.steps)
                    and _direct_workspace_bytes(c.arr, c.n, self.steps) <= limits[c.device])

        cus = {dev: torch.cuda.get_device_properties(dev).multi_processor_count for dev in limits}
        if concurrent:
            times = {key: _class_time(calls, key, self.steps, cus[key[0]]) for key in {(c.device, c.group) for c in calls}}
            calls.sort(key=lambda c: -times[(c.device, c.group)])
        runs: list[list[_Call]] = []
        for dev in limits:
            mine = [c for c in calls if c.device == dev]
            if concurrent:
                classes = tuple((c.m, c.n_, c.n) for c in mine)
                direct = direct_set_pays(classes, cus[dev], self.steps) and all(fits(c) for c in mine)
                if direct:
                    merged = _merge(mine, self.steps, limits[dev])
                    direct = direct_set_pays(classes, cus[dev], self.steps, len(merged))
                for c in mine:
                    c.direct = direct
                runs += merged if direct else [[c] for c in mine]
            else:
                for c in mine:
                    c.direct = direct_pays(c.m, c.n_, c.n, cus[dev], self.steps) and fits(c)
                runs += [[c] for c in mine]
        for c in calls:
            c.ws_bytes = (_direct_workspace_bytes(c.arr, c.n, self.steps) if c.direct
                          else _workspace_bytes(c.n, c.m, c.n_, self.steps))
        self._lanes = _lanes([c for c in calls if not c.direct], self.steps, cus)[0] if concurrent else {}
        launches, need = [], {}
        for run in runs:
            dev = run[0].device
            arr, n, wsb, lane, key = run[0].arr, run[0].n, run[0].ws_bytes, None, dev
            if concurrent and not run[0].direct:
                lane, key = self._lanes[(dev, run[0].group)], (dev, run[0].group)
            if len(run) > 1:
                arr, at = _entries(run), 0
                for c in run:  # the groups' entries are those of the launch
                    c.arr = (_lib.MuonMatrix * c.n).from_buffer(arr, at * ctypes.sizeof(_lib.MuonMatrix))
                    at += c.n
                n = at
                wsb = _direct_workspace_bytes(arr, n, self.steps)
            need[key] = max(need.get(key, 0), wsb)
            launches.append(_Launch(dev, arr, n, run[0].direct, lane, key))
        for key in [k for k in self._ws if k not in need]:
            del self._ws[key]
            self._ws_home.pop(key, None)
        for key, nbytes in need.items():
            ws = self._ws.get(key)
            if ws is None or ws.numel() < nbytes:
                self._ws[key] = None
                dev = key[0] if isinstance(key, tuple) else key
                self._ws[key] = torch.empty(nbytes, dtype=torch.uint8, device=dev)
                self._ws_home[key] = _lib.raw_stream(dev)
        self._calls = calls
        self._launches = launches
        self._concurrent = concurrent

    @torch.no_grad()
    def step(self):
        """Optimizer step for the Muon optimizer."""
        self._run(self._plan(), None, None)

    @torch.no_grad()
    def _step_amp(self, grad_scale: torch.Tensor | None, found_inf: torch.Tensor | None) -> None:
        """One step driven by ``torch.amp.GradScaler`` with its tensors left on the
        device: gradients divided by ``grad_scale``; where ``found_inf`` is
        non-zero the momentum and the parameters are left untouched (no host
        synchronisation).  Gradients are read, not rewritten."""
        self._run(self._plan(), grad_scale, found_inf)

    def _plan(self) -> list[nn.Parameter]:
        """The parameters that have a gradient, with the launch plan checked
        (rebuilt when any of them changed): argument errors raise here, before
        anything of the step is queued."""
        active, layouts = _lib.layout(self.model_params)
        if not active:
            return active
        key = (self.adjust_lr_fn, self.steps, layouts)
        if key != self._plan_key:
            _lib.check_not_capturing("Muon")
            self._plan_key = None
            self._build_calls(active)
            self._plan_key = key
            self._plan_lr = self.lr
        elif self.lr != self._plan_lr:  # a schedule moved lr: refresh the per-matrix scaled lr only
            for call in self._calls:
                for i in range(call.n):
                    e = call.arr[i]
                    e.scaled_lr = scaled_lr(self.lr, self.adjust_lr_fn, e.rows, e.cols)
            self._plan_lr = self.lr
        return active

    def _run(self, active: list[nn.Parameter], grad_scale: torch.Tensor | None,
             found_inf: torch.Tensor | None) -> None:
        """Queue the step over ``active`` (planned by :meth:`_plan`)."""
        if not active:
            return
        lib = _lib.load()
        nest = int(bool(self.is_nesterov))

        amp = grad_scale is not None or found_inf is not None
        amp_ptrs: dict = {}  # device -> (grad_scale, found_inf) on that device, made before any fork
        if amp:
            for call in self._launches:
                if call.device not in amp_ptrs:
                    amp_ptrs[call.device] = tuple(
                        t.to(call.device, torch.float32, non_blocking=True) if t is not None else None
                        for t in (grad_scale, found_inf))

        def launch(call, ws, stream_handle):
            args = (call.arr, call.n, self.lr, self.weight_decay, self.beta, nest, self.a, self.b, self.c, self.steps,
                    self.eps, ws.data_ptr(), ws.numel())
            gs, fi = amp_ptrs[call.device] if amp else (None, None)
            scaler = (gs.data_ptr() if gs is not None else None, fi.data_ptr() if fi is not None else None)
            with _lib.device_guard(call.device):
                if call.direct:
                    st = lib.mamw_muon_direct_step(*args, *scaler, stream_handle)
                elif not amp:
                    st = lib.mamw_muon_step(*args, stream_handle)
                else:
                    st = lib.mamw_muon_step_amp(*args, *scaler, stream_handle)
            _lib.check(st, "mamw_muon_step")

        if not self._concurrent:
            for call in self._launches:
                handle = _lib.raw_stream(call.device)
                launch(call, self._workspace(call.ws_key, call.device, handle), handle)
            return
        # Concurrent shape classes (lanes from _lanes): the largest on the
        # caller's current stream, the others on side streams.  Every side
        # stream waits for the caller's stream before anything of this step is
        # queued there, runs its classes' launches in order, and the caller's
        # stream waits for all of them at the end, so the step stays ordered
        # with the caller's work on its stream.
        side = {}
        for call in self._launches:
            s = call.lane
            if s is not None and (call.device, id(s)) not in side:
                side[(call.device, id(s))] = s
                s.wait_stream(torch.cuda.current_stream(call.device))
                for t in amp_ptrs.get(call.device, ()):  # the scaler may drop its tensors after step()
                    if t is not None:
                        t.record_stream(s)
        for call in self._launches:
            s = call.lane
            handle = _lib.raw_stream(call.device) if s is None else s.cuda_stream
            launch(call, self._workspace(call.ws_key, call.device, handle, s), handle)
        for (dev, _), s in side.items():
            torch.cuda.current_stream(dev).wait_stream(s)

    def _workspace(self, key, device: torch.device, handle: int, stream=None) -> torch.Tensor:
        """The workspace ``key`` for a launch on ``stream`` (the current one by
        default; ``handle`` its handle): recorded there unless its memory
        belongs to that stream, the one current when the plan was built."""
        ws = self._ws[key]
        if handle != self._ws_home[key]:
            ws.record_stream(torch.cuda.current_stream(device) if stream is None else stream)
        return ws

    def zero_grad(self, set_to_none: bool = False):
        """Resets gradients back to zero (the reference's behaviour), or to None
        with ``set_to_none=True`` (torch.optim's)."""
        for param in self.model_params:
            if param.grad is not None:
                if set_to_none:
                    param.grad = None
                else:
                    param.grad.zero_()

    def state_dict(self) -> dict:
        """Optimizer state in ``torch.optim.Muon``'s format: ``state[i]`` holds the
        ``momentum_buffer`` of parameter ``i`` (its position in ``model_params``),
        returned by reference; one param group with this branch's
        hyperparameters (``adjust_lr_fn`` ``"original"`` written as torch's
        ``None``)."""
        state = {i: {"momentum_buffer": self._momentum(p)} for i, p in enumerate(self.model_params)}
        group = {"lr": self.lr, "weight_decay": self.weight_decay, "momentum": self.beta,
                 "nesterov": self.is_nesterov, "ns_coefficients": (self.a, self.b, self.c), "eps": self.eps,
                 "ns_steps": self.steps,
                 "adjust_lr_fn": None if self.adjust_lr_fn == "original" else self.adjust_lr_fn,
                 "params": list(range(len(self.model_params)))}
        return {"state": state, "param_groups": [group]}

    def load_state_dict(self, state_dict: dict) -> None:
        """Restore a state produced by :meth:`state_dict` or by ``torch.optim.Muon``.

        Parameters are matched by position; momentum buffers are copied into
        this branch's own (parameters without saved state restart from zero,
        as torch's lazily created buffers do).
        """
        groups = state_dict["param_groups"]
        ids = [i for g in groups for i in g["params"]]
        if len(ids) != len(self.model_params):
            raise ValueError("loaded state dict contains a parameter group that doesn't match the size of "
                             "optimizer's group")
        keys = ("lr", "weight_decay", "momentum", "nesterov", "ns_coefficients", "eps", "ns_steps", "adjust_lr_fn")
        hyper = {tuple(tuple(g[k]) if k == "ns_coefficients" else g[k] for k in keys) for g in groups}
        if len(hyper) > 1:
            raise ValueError("parameter groups with different hyperparameters cannot be loaded into one Muon branch")
        pos = {pid: k for k, pid in enumerate(ids)}
        with torch.no_grad():
            for p in self.model_params:
                self._momentum(p).zero_()
            for pid, st in state_dict["state"].items():
                self._momentum(self.model_params[pos[pid]]).copy_(st["momentum_buffer"])
        if hyper:
            lr, wd, beta, nesterov, coeffs, eps, steps, adjust = hyper.pop()
            adjust = "original" if adjust is None else adjust
            if adjust not in _ADJUST_FNS:
                raise AssertionError(f"Invalid adjust_lr_fn: {adjust}")
            self.lr, self.weight_decay, self.beta, self.is_nesterov = lr, wd, beta, nesterov
            self.a, self.b, self.c = coeffs
            self.eps, self.steps, self.adjust_lr_fn = eps, steps, adjust


# The reference's class name, for drop-in imports.
TritonMuon = HipMuon
