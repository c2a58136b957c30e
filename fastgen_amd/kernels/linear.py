"""``y = x W^T`` for the two precisions of the engine.

float32: the engine's own matrix-core kernels (``gemm.hip``), a true
32-bit product whose rows do not depend on one another.  bfloat16: several
kernels can take a product (the engine's weight-streaming MFMA kernels of
``gemm_skinny.hip``, narrow and wide, with or without a cut of the k range, its
large tiles of ``gemm_large.hip`` for prompts, and
the vendor library's product through ``torch``, which the reference uses for
all of them: cuBLAS through ``F.linear``, ``fastgen/forward.py:433-513``).
Which one is the fastest depends on the matrix and on the number of rows, so
it is measured: the first time a product of some shape ``(N, K)`` meets some
number of rows, the kernels that can take it are timed on the model's matrices of that shape
(the caches emptied before each run) and the winner is kept in one table (``choices``) for this and every later product of
that shape and row bucket; times that are close are a tie, which a fixed order decides.  No size of any model stands here or in the parts.

A part hands ``linear`` its matrix as a :class:`StreamedMatrix` (made by :func:`streamed` when the part
loads): the matrix row by row and, where a model's weights fit the GPU twice over, a second copy in the order
in which the streaming kernels read it, which those kernels take.
"""

from __future__ import annotations

import functools
import itertools
import os
import weakref
from contextlib import contextmanager
from dataclasses import dataclass
from typing import Callable, Dict, List, Optional, Sequence, Tuple

import torch

from . import ops

_mm_out_dtype_ok: Optional[bool] = None


def _library_mm_f32_out(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """bf16 x bf16 -> fp32 through the library if this torch build offers it."""
    global _mm_out_dtype_ok
    if _mm_out_dtype_ok is False:
        return None
    try:
        y = torch.mm(x, w.t(), out_dtype=torch.float32)
        _mm_out_dtype_ok = True
        return y
    except (TypeError, RuntimeError):
        if _mm_out_dtype_ok is None:
            _mm_out_dtype_ok = False
            return None
        raise


# what the kernels take (their limits, not a model's sizes)
SKINNY_ROWS = 16  # one 16-row block of x: the narrow kernel (16 output columns a workgroup) and every folded epilogue
WIDE_ROWS = ops.SKINNY_MAX_ROWS  # the wide kernel (64 columns a workgroup): up to eight blocks of x
# the tiled kernel takes any number of rows; it is offered where it has been seen to win or come close (from the
# wide kernel's range up to a few hundred rows; beyond, the library's large tiles are twice as fast), where the large tiles below do
# not take the matrix (us at 192 rows, o and down of 4,096 x 4,096 and x 14,336: 24 / 54 against 17 / 43)
TILED_MIN_ROWS, TILED_MAX_ROWS = 65, 512
# The large tiles (:func:`~fastgen_amd.kernels.ops.gemm_large`) take any number of rows of a packed matrix and run without being
# measured, so that a first step takes no longer and every process takes the same kernel, where they are the faster ones (`_large_way`).
# Times against the kernel that is measured to be the fastest otherwise, of 44 matrices (512 to 128,256 columns, 512 to 14,336 of k) at 17 to 4,096 rows, with the
# norm behind where the result may be partial sums:
# * gated products: 0.45 to 1.11 beyond 64 rows, 0.78 on average (above 1.02 in 16 of 250, where the library's tiles happen to fill the chip). Up to 64
#   rows they are bound by how many workgroups read the matrix, 64 rows x 128 columns each: from 80 columns a compute unit on 0.91 to 1.0; fewer 0.97
#   to 1.17, 1.09 on average (the wide kernel's workgroups are twice as many, and it takes them), but for short k beyond 32 rows (k = 1,024
#   and less: 0.78 to 1.02);
# * products that may leave partial sums: 0.40 to 1.10 at 33 to 512 rows, 0.87 on average (above 1.02 in 20 of 342).  Up to 32 rows 0.91 to 1.04 from 2^24
#   elements of the matrix on, with fewer 0.87 to 1.17, 1.06 on average (the wide kernel's);
# * wide fp32 outputs (logits) 0.75 to 1.05 from 96 columns a compute unit on; 16,384 x 2,048 is 1.1 to 1.19 up to 64 rows, and at 129 to 384
#   rows, which fill tiles of 128 and 256 badly, 32,000 columns are 0.81 to 1.17, 50,304 and more 0.75 to 1.05;
# * beyond LARGE_ROWS plain products and partial sums too: 0.62 to 1.18, 0.93 on average (above 1.02 in 41 of 256).  Where k is long and one round of tiles leaves a
#   fifth of the compute units or more without one, the library is 1.09 times as fast (0.93 to 1.21 at 19 sizes, the most at
#   3,000 x 2,048 x 8,192, 192 tiles).
# A plain product of fewer rows has no splits to fill the chip with and goes the other ways (6,144 x 4,096 at 65 rows 34 us against
# 23 of the library, at 320 36 against 30).
LARGE_ROWS = TILED_MAX_ROWS
# The q/k/v product of up to this many rows leaves partial sums to the kernel that rotates and writes the cache; both together, us,
# against the library's product and that kernel on its rows: 6,144 x 4,096 at 17 / 64 / 128 rows 15.7 / 18.6 / 23.1 against 20.3 /
# 23.5 / 31.4, 5,120 x 3,072 11.7 / 14.0 / 18.5 against 14.9 / 18.4 / 24.7, 12,288 x 4,096 25.1 / 29.7 / 37.9 against 30.2 / 33.9 /
# 41.7, 2,048 x 1,536 8.5 / 9.8 / 10.9 against 10.4 / 11.2 / 11.0.  Beyond, small matrices lose (at 192 rows 2,048 x 1,536 12.2
# against 11.7), and the sums' bytes grow with the rows where W's do not.
QKV_PARTS_ROWS = 128


# ------------------------------------------------------- a weight, stored for its readers
@dataclass
class StreamedMatrix:
    """A weight matrix ``[N, K]`` as its products read it: ``rows`` is the matrix row by row (what the
    library's and the tiled product take, and the 32-bit path); ``packed``, where there is memory for
    a second copy, the same matrix in the order in which the streaming kernels' waves read it
    (:class:`~fastgen_amd.kernels.ops.PackedWeight`): the products of up to 128 rows then ask the
    memory for whole cache lines and take 8 to 13 % less time."""

    rows: torch.Tensor
    packed: Optional[ops.PackedWeight] = None
    part_of: Optional["StreamedMatrix"] = None  # the matrix whose first rows these are
    cut: Optional[ops.CutWeight] = None  # of a float32 matrix: its parts, for products of many rows

    @property
    def shape(self):
        return self.rows.shape

    @property
    def dtype(self) -> torch.dtype:
        return self.rows.dtype

    @property
    def streaming(self):
        """What the streaming kernels are given: the packed copy if there is one."""
        return self.packed if self.packed is not None else self.rows

    def first_rows(self, n: int) -> "StreamedMatrix":
        """The matrix of the first ``n`` rows (views; the packed copy only if ``n`` is a multiple of 16)."""
        keep = self.packed is not None and (n % 16 == 0 or n == self.rows.shape[0])
        cut = self.cut.first_rows(n) if self.cut is not None and (n % 16 == 0 or n == self.rows.shape[0]) else None
        return StreamedMatrix(self.rows[:n], self.packed.first_rows(n) if keep else None, self, cut)

    def alike(self) -> List["StreamedMatrix"]:
        """This matrix and the others of its kind, other layers' as a rule: what a measurement is made on."""
        if self.part_of is not None:
            return [self] + [m.first_rows(self.rows.shape[0]) for m in self.part_of.alike()[1:]]
        others = (ref() for ref in _stored.get(_kind(self), ()))
        return [self] + [m for m in others if m is not None and m is not self]

    def nbytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in self.tensors())

    def tensors(self) -> List[torch.Tensor]:
        """The matrix and its second copy."""
        return [self.rows] + [copy.data for copy in (self.packed, self.cut) if copy is not None]


# the stored matrices of a kind, as long as their parts hold them
_stored: Dict[tuple, List["weakref.ref[StreamedMatrix]"]] = {}


def _kind(m: StreamedMatrix) -> tuple:
    return tuple(m.rows.shape), m.rows.stride(), m.rows.dtype, m.rows.device, m.rows.data_ptr() % 16, m.packed is not None


# whether `streamed` makes the second copy: set for the time a model loads (`packing`)
_pack_now = False


@contextmanager
def packing(on: bool):
    """While a model's parts load: whether their matrices get the second, packed copy."""
    global _pack_now
    before, _pack_now = _pack_now, bool(on)
    try:
        yield
    finally:
        _pack_now = before


def packing_fits(matrix_bytes: int, device, budget_bytes: Optional[int] = None, may_be_forced: bool = True) -> bool:
    """The rule for the second copy when nobody says otherwise (``FG_PACKED_WEIGHTS=0`` / ``1`` does; ``1`` only if it
    ``may_be_forced``): the weights twice take at most half of the memory that the model and its cache may use
    (``budget_bytes``; default: all of the GPU's), so that at least half stays for the cache."""
    forced = os.environ.get("FG_PACKED_WEIGHTS", "")
    if forced == "0" or (forced == "1" and may_be_forced):
        return forced == "1"
    dev = torch.device(device)
    if dev.type != "cuda":
        return False
    if budget_bytes is None:
        budget_bytes = torch.cuda.get_device_properties(dev).total_memory
    return 2 * matrix_bytes <= budget_bytes // 2


def streamed(w: torch.Tensor, many_rows: bool = True) -> StreamedMatrix:
    """A part's weight matrix, placed on the device, as the products take it.  ``many_rows``: whether a step's tokens go through it (not
    only the rows that logits are wanted of): a float32 matrix's second copy serves those."""
    pack = _pack_now and w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2
    m = StreamedMatrix(w, ops.pack_weight(w) if pack else None, None,
                       ops.cut_weight(w) if _pack_now and many_rows and ops.cut_weight_ok(w) else None)
    if w.dtype == torch.bfloat16:  # (a 32-bit product is not measured)
        _stored[_kind(m)] = [ref for ref in _stored.get(_kind(m), ()) if ref() is not None] + [weakref.ref(m)]
    return m


def _rows_of(w) -> torch.Tensor:
    return w.rows if isinstance(w, StreamedMatrix) else w


def _aligned(x: torch.Tensor, w) -> bool:
    w = _rows_of(w)
    (ldx, unit_x), (ldw, unit_w) = x.stride(), w.stride()
    return (x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.shape[1] % 8 == 0
            and unit_x == 1 and unit_w == 1 and ldx % 8 == 0 and ldw % 8 == 0
            and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def skinny_ok(x: torch.Tensor, w) -> bool:
    """Few rows (decode): the engine's own weight-streaming kernels take the product, with the
    epilogues that are folded into them."""
    return x.shape[0] <= SKINNY_ROWS and _aligned(x, w)


def fold_ok(x: torch.Tensor, w) -> bool:
    """Few rows of bfloat16: the norms around a product can be folded into the products
    (:class:`~fastgen_amd.kernels.ops.ScaledRows`)."""
    return skinny_ok(x, w)


def k_splits_for(n_out: int, k: int, rows: int = 0) -> int:
    """Splits of the k range that give the wide kernel (64 output columns a workgroup) about two
    workgroups per compute unit, at most 8; with many rows a split keeps at least 1,024 of k (the
    partial sums it writes grow with the rows), else 512.  1: the output is wide enough by itself."""
    blocks = -(-n_out // 64)
    return max(1, min(8, 2 * ops.compute_units() // blocks, k // (1024 if rows > 48 else 512)))


# ------------------------------------------------------------------ the table
# (what is asked for, N, K, row bucket) -> name of the kernel that measured fastest
choices: Dict[Tuple[str, int, int, int], str] = {}
# the same keys -> what each candidate took when it was measured (milliseconds on average, the consumer's cost included)
timings: Dict[Tuple[str, int, int, int], Dict[str, float]] = {}
_samples: Dict[Tuple[str, int, int, int], List[Dict[str, float]]] = {}  # of the keys that are still measured
# set to a candidate's name to take that kernel wherever it is among the candidates, to "large" for the large tiles
# wherever they can take a product of more than 16 rows, under any other name not by their rule (tests run the
# engine once under each name, so that every kernel that may be chosen is compared with the plain run)
force: Optional[str] = None
_TIMED_RUNS = 2  # of every candidate, each of the _SAMPLES times
# How long a product takes depends on where its matrix happens to lie (64 rows of 28,672 x 4,096: the library's takes 49 to
# 51 us on one layer's matrix and 59 to 63 on the next ones, in every process; the wide kernel 52 to 57 on all of them), so
# the candidates are measured on as many of the model's matrices, one layer's after the other's; not again where one of them
# leads by more than that.
_SAMPLES, _CLEAR = 3, 0.25
# A lead smaller than this decides nothing: the same program would take one kernel today and another tomorrow, and their
# results differ by a rounding.
_TIE = 0.04
# Before each timed run this many bytes are read, so that a candidate finds the weights where a model's step
# finds them: in memory, not in the caches (a memory-side cache of 256 MB and the L2s; a decode step streams
# gigabytes of other weights between two uses of a matrix).  Timed warm, the wide kernel looks faster than the
# narrow one on matrices that fit the cache and is the slower one in the model.  (Read, not written: modified
# lines would be written back while the candidate runs, which costs the candidates unequally.)
_FLUSH_BYTES = 384 << 20


def row_bucket(rows: int) -> int:
    """Products of up to 16 rows are measured per number of rows, above that per block of 16 rows
    (the kernels work on such blocks) up to 256, per block of 64 up to the last size at which an own
    kernel is offered, and as one beyond."""
    if rows <= SKINNY_ROWS:
        return rows
    if rows <= 256:
        return -(-rows // 16) * 16
    return min(-(-rows // 64) * 64, TILED_MAX_ROWS + 64)


def tiled_splits(n_out: int, k: int, rows: int, tile_rows: int) -> int:
    """Splits of the k range that give the tiled kernel about two workgroups a compute unit, at most 16,
    each with at least 512 of k."""
    tiles = -(-rows // tile_rows) * -(-n_out // 128)
    return max(1, min(16, 2 * ops.compute_units() // tiles, k // 512))


def _capturing() -> bool:
    return torch.cuda.is_current_stream_capturing()


def _winner(best: Dict[str, float], order: List[str]) -> str:
    """Of the candidates whose time is within ``_TIE`` of the shortest the first in ``order``."""
    limit = (1 + _TIE) * min(best.values())
    return next(name for name in order if best[name] <= limit)


def _choose(what: str, n: int, k: int, rows: int, candidates: List[Tuple[str, Callable[[], torch.Tensor]]],
            handicap: Optional[Dict[str, float]] = None, library_ties: bool = False) -> str:
    """The candidate to run: the forced one, the one the table holds, or, measured once more, the fastest so far.
    Timing needs the device to itself (events and a wait for them), so a product that is first met while
    a step is being recorded runs the first candidate, unrecorded in the table; the engine runs every
    step once, unrecorded, before it records it.  The candidates are timed in turn on the same
    operands, each run behind a sweep of memory that empties the caches.  ``handicap``: milliseconds added to a candidate's time
    for what its result costs the consumer (partial sums that are still to be added).  ``library_ties``: the library
    takes a tie, else the earlier candidate does."""
    names = [c[0] for c in candidates]
    if force in names:
        return force
    if len(candidates) == 1:
        return names[0]
    key = (what, n, k, row_bucket(rows))
    got, seen = choices.get(key), _samples.get(key)
    known = got in names
    if known and seen is None:  # settled, or put there from outside
        return got
    if _capturing():
        return got if known else names[0]
    seen = seen if known and seen else []
    order = sorted(names, key=lambda name: name != "library") if library_ties else names
    seen = seen + [_measure(candidates, handicap or {}, first=not seen)]
    timings[key] = {name: sum(t[name] for t in seen) / len(seen) for name in names}
    choices[key] = winner = _winner(timings[key], order)
    clear = (1 + _CLEAR) * timings[key][winner]
    if len(seen) < _SAMPLES and any(timings[key][name] <= clear for name in names if name != winner):
        _samples[key] = seen
    else:
        _samples.pop(key, None)
    return winner


def _settle(what: str, n: int, k: int, rows: int, candidates: List[Tuple[str, Callable]], matrices: Callable[[], Sequence],
            handicap: Optional[Dict[str, float]] = None, library_ties: bool = False) -> str:
    """:func:`_choose` until the table's entry stays, before anything is computed by it: with the best so far, a step that
    is recorded after one warm-up would keep a kernel that the next engine of the process does not take, and their results would
    differ by a rounding.  ``candidates``: functions of a matrix; ``matrices()``: the matrices that they are timed on in turn."""
    key = (what, n, k, row_bucket(rows))
    if choices.get(key) in (c[0] for c in candidates) and key not in _samples and force is None:
        return choices[key]
    for m in itertools.cycle(matrices()):
        name = _choose(what, n, k, rows, [(c, lambda fn=fn: fn(m)) for c, fn in candidates], handicap, library_ties)
        if key not in _samples or _capturing():
            return name


def _measure(candidates: List[Tuple[str, Callable[[], torch.Tensor]]], handicap: Dict[str, float],
             first: bool) -> Dict[str, float]:
    """What each candidate takes on the operands at hand, in milliseconds."""
    best: Dict[str, float] = {}
    if first:  # once each, unmeasured: libraries load, the library picks its kernel
        for _, fn in candidates:
            fn()
    try:
        flush = torch.zeros(_FLUSH_BYTES // 4, dtype=torch.int32, device=torch.cuda.current_device())
        torch.cuda.current_stream().synchronize()  # (its zeros are in memory before anything is timed)
    except RuntimeError:  # no memory to spare: the candidates are timed on what the caches hold
        flush = None
    events = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
               for _ in range(_TIMED_RUNS)] for _ in candidates]
    for r in range(_TIMED_RUNS):
        for ev, (_, fn) in zip(events, candidates):
            if flush is not None:
                flush.amax()
            ev[r][0].record()
            fn()
            ev[r][1].record()
    torch.cuda.current_stream().synchronize()
    del flush
    for ev, (name, _) in zip(events, candidates):
        best[name] = min(a.elapsed_time(b) for a, b in ev) + handicap.get(name, 0.0)
    return best


@functools.lru_cache(maxsize=4096)
def _large_way(M: int, N: int, K: int, ldx: int, gated: bool, partials: bool, wide_out: bool, forced: bool) -> Optional[Tuple[int, int]]:
    """Tile and splits of k of a product that goes to the large tiles (``LARGE_ROWS``; ``forced``: wherever they can take it), ``(0,
    splits)`` for the wide kernel, or None: one of those that are measured.  ``wide_out``: fp32 output."""
    if M <= SKINNY_ROWS or not ops.gemm_large_takes(M, N, K, ldx) or (gated and (N % 16 or wide_out)):
        return None
    units = ops.compute_units()
    if forced or M > LARGE_ROWS:
        takes = True
    elif gated:
        takes = M > 64 or N >= 80 * units or (M > 32 and K <= 1024)
    elif partials:
        takes = M > 32 or N * K >= 1 << 24
    else:
        takes = wide_out and N >= (192 if 128 < M <= 384 else 96) * units
    if not takes:
        return (0, k_splits_for(N, K, M) if partials else 1) if gated or partials else None
    tile, splits = ops.large_plan(M, N, K, gated, partials)
    if M > LARGE_ROWS and not (forced or gated or wide_out) and K >= 4096 * splits:
        tiles = -(-M // (tile // 1000)) * -(-N // (tile % 1000)) * splits
        if tiles <= 0.8 * units:
            return None
    return tile, splits


@functools.lru_cache(maxsize=4096)
def _qkv_way(M: int, N: int, K: int, ldx: int) -> Optional[Tuple[int, int]]:
    """Tile and splits of a q/k/v product that leaves partial sums (``QKV_PARTS_ROWS``), or None."""
    if not SKINNY_ROWS < M <= QKV_PARTS_ROWS or not ops.gemm_large_takes(M, N, K, ldx):
        return None
    tile, splits = ops.parts_plan(M, N, K)
    return (tile, splits) if splits > 1 else None


def qkv_parts(x: torch.Tensor, w) -> Optional[torch.Tensor]:
    """The q/k/v product of a decoding batch as fp32 partial sums ``[S, M, N]`` for
    :func:`~fastgen_amd.kernels.ops.rope_kv_parts`, or None where they are not the way (``QKV_PARTS_ROWS``)."""
    if force not in (None, "large") or not isinstance(w, StreamedMatrix) or w.packed is None:
        return None
    way = _qkv_way(x.shape[0], *w.rows.shape, x.stride(0))
    if way is None or not _aligned(x, w.rows):
        return None
    return ops.gemm_large(x, w.packed, k_splits=way[1], tile=way[0])


def linear(x, w, out_dtype: Optional[torch.dtype] = None,
           partials_ok: bool = False, residual: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None,
           epilogue: Optional[str] = None):
    """``x @ w.T`` for ``w`` a matrix or a :class:`StreamedMatrix` (whose packed copy, if it has one, the
    streaming kernels read).  With ``partials_ok`` the result may come as fp32 ``[S, M, N]``
    partial sums whose sum over ``S`` is the product (the caller hands it to a
    norm, which adds them in order).

    ``epilogue="silu_mul"``: ``w`` is a gate and an up matrix interleaved by
    :func:`~fastgen_amd.kernels.ops.interleave_gate_up` and the result is
    ``silu(gate) * up`` ``[M, N/2]``, in the product's kernel where one that does so is the fastest;
    ``"gelu_tanh_mul"``: the same with the tanh form of GELU.

    ``x`` may be :class:`~fastgen_amd.kernels.ops.ScaledRows`.  ``residual`` = (h, norm weight,
    eps) asks for more than the product: add it to the fp32 residual stream ``h`` and prepare the
    RMSNorm that follows.  Where that can be folded into the product's kernel (few rows, bfloat16)
    the result is ``ScaledRows`` and ``h`` is updated; where not, the plain product comes back and
    adding and norming are the caller's.  A float32 product with ``residual`` is finished, :class:`~fastgen_amd.kernels.ops.NormedRows`."""
    silu = epilogue in ("silu_mul", "gelu_tanh_mul")  # a gated epilogue: act(gate) * up
    if epilogue not in (None, "silu_mul", "gelu_tanh_mul"):
        raise ops.KernelArgumentError(f"linear: unknown epilogue {epilogue!r}")
    gated = "gelu_tanh" if epilogue == "gelu_tanh_mul" else True  # what the kernels' epilogue argument takes
    act_mul = ops.gelu_mul if epilogue == "gelu_tanh_mul" else ops.silu_mul
    matrix = w if isinstance(w, StreamedMatrix) else StreamedMatrix(w)
    sw, w = matrix.streaming, matrix.rows  # what the streaming kernels read, and the library
    scaled = x if isinstance(x, ops.ScaledRows) else None
    if scaled is not None:
        if not fold_ok(scaled.rows, w) or out_dtype not in (None, torch.bfloat16):
            x, scaled = scaled.materialize(), None
        else:
            x = scaled.rows
    if not x.is_cuda:
        raise ops.KernelArgumentError("fastgen_amd runs on the GPU only; got a tensor on " + str(x.device))
    if x.dtype == torch.float32:
        if out_dtype not in (None, torch.float32):
            raise ops.KernelArgumentError("a float32 product has float32 output")
        if silu:
            return ops.gemm_f32_gated(x, w, "gelu_tanh" if gated == "gelu_tanh" else "silu", matrix.cut)
        if residual is not None and ops.gemm_f32_norm_ok(x, w, residual[0], residual[1]):
            return ops.NormedRows(ops.gemm_f32_norm(x, w, *residual, matrix.cut))
        return ops.gemm_f32(x, w, matrix.cut)
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise ops.KernelArgumentError(f"linear: unsupported dtypes {x.dtype}, {w.dtype}")
    out_dtype = out_dtype or torch.bfloat16
    rows, (N, K) = x.shape[0], w.shape
    own = _aligned(x, w)
    src = scaled or x  # what the own kernels are given: they finish a norm that is still open

    if residual is not None and own and rows <= SKINNY_ROWS and out_dtype == torch.bfloat16 and not silu:
        h, norm_w, eps = residual
        if h.dtype == torch.float32 and h.is_contiguous() and h.shape == (rows, N):
            return ops.gemm_skinny_residual(src, sw, h, norm_w, eps)

    if own and rows > SKINNY_ROWS and sw is not w and (force is None or force == "large"):  # (no open norm: those have few rows)
        way = _large_way(rows, N, K, x.stride(0), silu, partials_ok and out_dtype == torch.bfloat16, out_dtype == torch.float32,
                         force is not None)
        if way is not None:
            if way[0]:
                return ops.gemm_large(x, sw, out_dtype, gated if silu else False, way[1], way[0])
            return ops.gemm_skinny(x, sw, out_dtype, gated if silu else False, way[1], wide=True)

    def library(m: StreamedMatrix) -> torch.Tensor:
        xin = scaled.materialize() if scaled is not None else x
        if out_dtype == torch.bfloat16:
            y = torch.nn.functional.linear(xin, m.rows)
        else:
            y = _library_mm_f32_out(xin, m.rows)
            if y is None:
                y = ops.gemm_nt(xin, m.rows, out_dtype=torch.float32)
        return act_mul(y) if silu else y

    candidates: List[Tuple[str, Callable[[StreamedMatrix], torch.Tensor]]] = []
    handicap: Dict[str, float] = {}
    tiled_ok = own and TILED_MIN_ROWS <= rows <= TILED_MAX_ROWS and (
        force in ("tiled", "tiled256") or sw is w or not ops.gemm_large_takes(rows, N, K, x.stride(0)))

    def sums_cost(splits: int) -> float:
        """Milliseconds the consumer takes to read the partial sums beyond the first (at 4 TB/s)."""
        return (splits - 1) * rows * N * 4 / 4e9

    if own and silu and out_dtype == torch.bfloat16 and N % 16 == 0:
        if rows <= SKINNY_ROWS:
            candidates.append(("narrow", lambda m: ops.gemm_skinny(src, m.streaming, silu_mul_epilogue=gated, wide=False)))
        if rows <= WIDE_ROWS:
            candidates.append(("wide", lambda m: ops.gemm_skinny(src, m.streaming, silu_mul_epilogue=gated, wide=True)))
        if tiled_ok:
            candidates.append(("tiled256", lambda m: ops.gemm_tiled(x, m.streaming, silu_mul_epilogue=gated, tile_rows=256)))
    elif own and not silu:
        if rows <= SKINNY_ROWS:
            candidates.append(("narrow", lambda m: ops.gemm_skinny(src, m.streaming, out_dtype, wide=False)))
        elif rows <= WIDE_ROWS and partials_ok:
            splits = k_splits_for(N, K, rows)
            candidates.append(("wide", lambda m: ops.gemm_skinny(x, m.streaming, out_dtype, k_splits=splits, wide=True)))
            handicap["wide"] = sums_cost(splits)
        elif rows <= 64:
            candidates.append(("wide", lambda m: ops.gemm_skinny(x, m.streaming, out_dtype, wide=True)))
        if tiled_ok and partials_ok and out_dtype == torch.bfloat16:
            for name, tile_rows in zip(("tiled", "tiled256"), ops.TILED_TILE_ROWS):
                s_t = tiled_splits(N, K, rows, tile_rows)
                candidates.append((name, lambda m, tile_rows=tile_rows, s_t=s_t: ops.gemm_tiled(
                    x, m.streaming, out_dtype, k_splits=s_t, tile_rows=tile_rows)))
                handicap[name] = sums_cost(s_t)
    if scaled is None or not candidates:
        candidates.append(("library", library))
    what = (epilogue if silu else "store") + ("+partials" if partials_ok and rows > SKINNY_ROWS else "") + (
        "+f32" if out_dtype == torch.float32 else "") + ("+scaled" if scaled is not None else "") + (
        "+packed" if sw is not w else "")
    # Ties: the kernel with the epilogue in it, and with few rows the narrow one, both the least launches; a plain
    # product of more rows goes to the library, whose result is whole (no partial sums to add).
    name = _settle(what, N, K, rows, candidates, matrix.alike, handicap, library_ties=not silu and rows > SKINNY_ROWS)
    return dict(candidates)[name](matrix)
