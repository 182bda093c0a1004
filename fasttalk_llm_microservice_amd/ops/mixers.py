"""Sequence-mixer and mixture-of-experts ops: latent (low-rank KV) attention over a
paged latent cache, windowed attention (softmax or sigmoid weights, distance bias,
several score maps per head, capped scores, a sink in the softmax) over a paged key / value
cache, attention that mixes its scores across the heads, the gated delta-rule recurrence (a
decay per channel or per head), retention and the selective state-space scan over state
slots, short causal convolutions (alone, or fused with per-head norms, rotation and the cache
write, or with the delta rule's preparation), routing (grouped softmax top-k, or top-k on the
logits with softmax or sigmoid weights, optionally limited to the best groups), clamped-GLU,
silu-GLU and relu^2 experts (per-pair kernels for few rows, a grouped product for many), and the fp32-residual norms (RMS pre/post norms, optionally with a token shift, layer
norm with bias) that tie them together.

GPU tensors run the gfx950 kernels of the ``_C_mixers`` extension (``csrc/mixers``),
fp32 or bf16 activations with fp32 statistics / scores / state; CPU tensors run the
PyTorch implementations in :mod:`.mixers_ref`.  As in :mod:`fasttalk_llm_microservice_amd.ops`
there is no silent fallback for GPU tensors.

A step's rows are described by :class:`Segments`: every scheduled sequence contributes
one segment of consecutive rows (a decode row is a segment of one row, a prefill chunk
a longer one), with the position of its first row, its state slot and its block table.
"""
from __future__ import annotations

import contextlib
import dataclasses
import functools
import importlib
import os
import threading
from typing import NamedTuple, Optional, Union

import torch

from . import mixers_ref as ref

_lock = threading.Lock()
_M = None


def native_mixers():
    """The loaded ``_C_mixers`` extension, built in-tree on first use if allowed."""
    global _M
    if _M is not None:
        return _M
    with _lock:
        if _M is not None:
            return _M
        try:
            mod = importlib.import_module("fasttalk_llm_microservice_amd._C_mixers")
        except ImportError as e:
            if os.environ.get("FT_AUTOBUILD", "1") == "0":
                raise RuntimeError("fasttalk native extension _C_mixers is not built; run "
                                   "`python -m fasttalk_llm_microservice_amd.ops.build --only mixers`") from e
            from .build import build_mixers

            build_mixers(verbose=True)
            mod = importlib.import_module("fasttalk_llm_microservice_amd._C_mixers")
        _M = mod
        return _M


@dataclasses.dataclass
class Segments:
    """Row segments of one step (device int32 tensors; ``num`` / ``max_rows`` host ints)."""
    start: torch.Tensor          # [num + 1] first row of each segment, then the row count
    pos0: torch.Tensor           # [num] sequence position of the segment's first row
    slot: torch.Tensor           # [num] recurrent-state slot (-1: padding, state untouched)
    kv_len: torch.Tensor         # [num] context length once this step's rows are written
    block_tables: torch.Tensor   # [num, max_blocks]
    num: int
    max_rows: int                # longest segment (rows)
    max_kv: int = 0              # longest context (tokens); 0 = unknown
    # host copies of start / pos0 / kv_len (eager steps; None inside captured graphs)
    host: Optional[tuple] = None


def _plain16(*tensors) -> bool:
    """Dense tensors at 16-byte addresses, as kernels take them that read and write whole pieces."""
    return all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in tensors)


def _device_segments(seg: Segments) -> bool:
    """Whether a kernel can read the segments itself (the product forms go by the host's copies)."""
    return all(t.is_cuda and t.dtype == torch.int32 and t.is_contiguous()
               for t in (seg.start, seg.pos0, seg.kv_len, seg.block_tables))


# ---------------------------------------------------------------------------------
# products with weights [out, in]
# ---------------------------------------------------------------------------------

# most rows of a product that streams its weights once through the few-rows kernel (a decode
# step's; the vendor's tiles fill up beyond)
FEW_ROWS = 64
# activations of the few-rows kernels and the sorted experts (csrc/mixers/few_rows.h)
FEW_TANH_CAP = 6       # linear_f32 with a cap
FEW_ACTS = {None: 0, "gelu_tanh": 1, "relu": 2, "silu": 3, "clamp_glu": 4, "relu_sq": 5, "silu_glu": 3}


def _piece_rows(x, w) -> bool:
    """bf16 rows and weights of whole 16-byte pieces on a GPU."""
    return bool(x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2
                and x.shape[0] >= 1 and x.shape[1] % 8 == 0 and x.shape[1] >= 8 and x.stride(1) == 1
                and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and w.is_contiguous())


def _few_rows(x, w) -> bool:
    """The same, at most FEW_ROWS rows."""
    return x.shape[0] <= FEW_ROWS and _piece_rows(x, w)


@functools.lru_cache(maxsize=8192)
def _tile_gemm_pays(rows: int, n: int, k: int, act: Optional[str] = None) -> bool:
    """Where a product of more than FEW_ROWS rows runs in the kernels of csrc/mixers/tile_gemm.hip (``n`` rows of w; with
    ``act`` in their epilogue): k of whole 64 and an expected time that is near the vendor's, which lies between 6 and 20 us
    above that of its operations at 1.3 PFLOP/s, and the activation's kernel, which takes 4 us and its bytes at 3.5 TB/s.  Up to
    1024 rows a step is issued by the host, where a call of the vendor's product takes 21 us and this one 5, so the kernel may
    be behind by a few (2 to 4 us of 25 to 35 from 640 rows on; at most 13 of 82 were seen: gated 2 x 6144, k = 4096, 640
    rows); captured steps: :func:`_tile_gemm_behind`.  Beyond, the sooner full tiles keep the vendor's product at its rate, the
    less.  us at 100 / 300 / 777 / 2048 / 4096 rows, the vendor's (with the activation) beside it:
      n = 2048, k = 2048     7 10 14 22 40 (9 11 15 23 35)         k = 8192            22 31 49 90 128 (21 33 47 74 118)
      n = 10272, k = 2048    18 21 47 82 155 (18 26 41 96 180)     n = 64              6 7 7 7 8 (8 8 8 9 10)
      gated, 2 x 8192, k = 2048    20 34 55 109 225 (28 40 66 137 270)
      n = 4096, k = 14336    44 93 121 215 338 (50 76 115 204 316)"""
    if rows <= FEW_ROWS or k % 64 or k < 64:
        return False
    glu = act is not None and act != "relu_sq"
    out = n // 2 if glu else n
    if max(rows * k, n * k) * 2 > 0xffffffff or out < 1:
        return False
    us, tail = native_mixers().tile_gemm_us(rows, out, k, glu)
    flops_us = 2.0 * rows * n * k / (1.3e9 if rows <= 1024 else 1.35e9)
    rounds = -(-rows // 256) * -(-n // 256) / 256
    if tail and act is None and rows > 1024 and n % 8 == 0 and k <= 3072 and rounds < 2:
        # A round of large tiles and a part, in halves: the vendor's product has that part too, and of what stays empty in it at
        # least 0.4 shows in its time; these sizes take 0.93 of the expected time.  Of 393 products of 1100 to 4096 rows and k of 512 to
        # 8192 and 390 drawn ones this takes 85, at 0.92 of the vendor's time in the mean and 1.04 at most.  Left out: columns that
        # leave in pieces below 16 bytes (up to 1.19), longer sums, whose empty part the vendor's products fill along k (9216 columns of
        # 2048 rows, k = 2048 / 3072 / 4096 / 8192: 0.94, 1.00, 1.04, 1.08), and two whole rounds and a part (up to 1.05).
        return 0.93 * us <= 7 + flops_us * (1 + 0.4 * (2 / rounds - 1))
    spare = (20 if rows <= 1024 else 7) + (0 if act is None else 4 + rows * out * (6 if glu else 4) / 3.5e6)
    return us <= spare + flops_us


_replayed = threading.local()


@contextlib.contextmanager
def replayed_step():
    """What this thread issues inside is captured, or warms up what is: no call of its replays costs the host anything."""
    before = getattr(_replayed, "on", False)
    _replayed.on = True
    try:
        yield
    finally:
        _replayed.on = before


def _tile_gemm_behind(n: int, k: int, act: Optional[str]) -> bool:
    """Where :func:`_tile_gemm_pays` lets the tiles be behind the vendor's product for its host time: few columns, and long
    sums of few tiles.  A :func:`replayed_step` has none to save and leaves these to the vendor's.  us in a graph at 65 / 128 /
    256 rows, the vendor's beside it: n = 256, k = 2048 6.5 6.5 6.5 (5.6 8.2 8.3); 64 6.2 6.4 6.5 (5.8 5.9 5.7); 2048, 8192 19.8
    24.7 24.0 (19.9 20.5 26.1); 14336, 4096 32.7 34.8 43.4 (29.4 32.5 50.0); kept: 2048, 2048 7.2 7.5 7.6 (8.8 8.8 9.8); 1024, 1024
    5.2 5.3 5.2 (5.6 5.6 8.3); 8192, 2048 12.0 13.4 17.2 (13.5 15.5 24.6); gated, 2 x 8192, k = 2048 20.9 21.0 26.2 (22.5 24.6 34.1)."""
    return act is None and (n < 1024 or k >= 4096)


def _tile_gemm(x, w, bias, act: Optional[str] = None, limit: float = 0.0):
    """The product where :func:`_tile_gemm_pays`, else None: also where rows overlap, w is one row or a gated form's two matrices
    and one row more, or the bias is broadcast."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[0] <= FEW_ROWS or not _piece_rows(x, w) or x.stride(0) < x.shape[1] \
            or x.stride(0) * x.shape[0] * 2 > 0xffffffff or not _tile_gemm_pays(x.shape[0], w.shape[0], x.shape[1], act) \
            or (bias is not None and not (bias.dtype == torch.bfloat16 and bias.is_contiguous() and bias.shape == w.shape[:1])):
        return None
    glu = act is not None and act != "relu_sq"
    if (glu and w.shape[0] % 2) or (getattr(_replayed, "on", False) and _tile_gemm_behind(*w.shape, act)):
        return None
    y = torch.empty(x.shape[0], w.shape[0] // 2 if glu else w.shape[0], dtype=x.dtype, device=x.device)
    native_mixers().tile_gemm(y, x, w, bias, FEW_ACTS[act], float(limit), -1)
    return y


def _few_rows_pays(rows: int, n: int, k: int, act: Optional[str] = None) -> bool:
    """Where the few-rows kernel is at least level with the vendor's product and, with ``act``, the activation's kernel
    (``n`` rows of w: a gated form's two matrices), or behind by a microsecond or so: it takes 5 us on the host where the
    vendor's call takes 20, which counts in steps that are not replayed.  Its waves take long sums in a chain and share one read of X per
    workgroup, so it loses with k, the sooner the more rows there are; most columns below 16384 go to workgroups of four
    waves, whose chains are twice as long.  us at 1 / 16 / 32 / 64 rows, the vendor's beside it (weights from HBM):
      n = 2048, k = 4096      8 9 11 14 (15 15 12 14)        k = 12288   19 21 28 39 (19 19 24 34)
      n = 5120, k = 2048      10 10 11 18 (12 12 12 13)      k = 13824   48 47 57 88 (30 32 37 48)
      n = 14336, k = 4096     24 28 38 33 (29 29 26 27)      n = 32768, k = 2048   28 28 28 33 (34 34 34 35)
      gated, 2 x 1024, k = 2048   8 8 9 12 (11 12 12 13)     2 x 2048, k = 8192   32 32 36 38 (20 20 22 28)"""
    if act == "relu_sq":
        if n >= 16384:
            longest = 6144
        elif n > 4096:
            longest = 4096 if rows <= 16 else 2048 if rows <= 32 else 1024
        else:
            longest = 8192 if rows <= 16 else 6144 if rows <= 32 else 4096
    elif act is not None:
        if rows <= 16:
            longest = 6144 if n >= 8192 else 4096
        elif n < 512 or (rows <= 32 and n >= 16384):
            longest = 4096
        else:
            longest = 3072 if (8192 if rows <= 32 else 5120) <= n < 16384 else 2048
    elif n >= 32768:
        longest = 8192 if rows <= 32 else 6144 if rows <= 48 else 2048
    elif n > 4096:
        if rows <= 16:
            longest = 6144 if n >= 16384 else 4096 if n >= 10240 else 3072 if n >= 8192 else 2048
        else:
            longest = 2048 if rows <= 32 and not 12288 < n < 16384 else 0
    elif rows <= 16:
        longest = max(4096, min(8192, 4 * n))
    elif rows <= 32:
        longest = 6144 if n >= 2048 else 4096
    else:
        longest = 4096 if n >= 512 else 2048
    return k <= longest


def linear(x, w, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x w^T (+ bias) in x's dtype, fp32 accumulation."""
    if _few_rows(x, w) and _few_rows_pays(x.shape[0], w.shape[0], x.shape[1]):
        y = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
        native_mixers().few_rows_gemm(y, x, w, bias, 0, 0.0)
        return y
    y = _tile_gemm(x, w, bias)
    return torch.nn.functional.linear(x, w, bias) if y is None else y


def linear_out(x, w, parts: bool, bias: Optional[torch.Tensor] = None):
    """:func:`linear`, a sublayer's last product; with ``parts`` its result may be :class:`ExpertParts`, the product with k cut
    into parts that the norm step behind adds up: few columns leave a product of few rows, or of long sums, half the chip."""
    n, few = _out_parts(x.shape[0], *w.shape) if parts and x.is_cuda else (1, False)
    if n > 1 and _piece_rows(x, w) and (bias is None or (bias.dtype == x.dtype and bias.is_contiguous() and bias.shape == w.shape[:1])) \
            and (few or x.shape[1] <= x.stride(0) <= 0x7fffffff // x.shape[0]):
        d = torch.empty(x.shape[0] * n, w.shape[0], dtype=torch.float32, device=x.device)
        (native_mixers().few_rows_gemm_parts if few else native_mixers().tile_gemm_parts)(d, x, w, bias)
        return ExpertParts(d, None, None, None)
    return linear(x, w, bias)


@functools.lru_cache(maxsize=8192)
def _out_parts(rows: int, n: int, k: int):
    """(The parts of k of a product whose norm step adds them, whether the kernel of few rows makes them)."""
    N, few = native_mixers(), rows <= FEW_ROWS
    if not N.expert_rows_fit(n) or k > (16384 if few else 0x7fffffff // n):
        return 1, few
    return (N.few_rows_parts(n, k) if few else N.tile_parts(rows, n, k)), few


def linear_pair(x, w, x2, w2):
    """(:func:`linear` of x and w, of x2 and w2); one launch where the kernel of few rows takes both and they are alike in sizes
    and strides."""
    if x.shape == x2.shape and w.shape == w2.shape and x.stride() == x2.stride() and _few_rows(x, w) and _few_rows(x2, w2) \
            and _few_rows_pays(x.shape[0], w.shape[0], x.shape[1]):
        y, y2 = (torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device) for _ in range(2))
        native_mixers().few_rows_pair(y, y2, x, x2, w, w2)
        return y, y2
    return linear(x, w), linear(x2, w2)


def linear_side_gate(x, w, table, ids, col0: int, sd: int):
    """:func:`side_gate` of x w^T; one launch, the product fp32 up to the gate's result, for few rows."""
    if _few_rows(x, w) and _few_rows_pays(x.shape[0], w.shape[0], x.shape[1]) and table.dtype == torch.bfloat16 \
            and table.stride(1) == 1 and ids.dtype == torch.int32:
        y = torch.empty(x.shape[0], sd, dtype=x.dtype, device=x.device)
        native_mixers().few_rows_side_gate(y, x, w, table, ids, col0)
        return y
    return side_gate(linear(x, w), table, ids, col0, sd)


def linear_f32(x, w, cap: float = 0.0) -> torch.Tensor:
    """x w^T with fp32 accumulation and fp32 output, through :func:`tanh_cap_` if there is a ``cap``."""
    if _few_rows(x, w) and _few_rows_pays(x.shape[0], w.shape[0], x.shape[1]):
        y = torch.empty(x.shape[0], w.shape[0], dtype=torch.float32, device=x.device)
        native_mixers().few_rows_gemm(y, x, w, None, FEW_TANH_CAP if cap else 0, float(cap))
        return y
    y = mm_f32(x, w.t())
    return tanh_cap_(y, cap) if cap else y


def linear_act(x, w, act: str, limit: float = 0.0) -> torch.Tensor:
    """act of x w^T: w = [gate | up] rows for the gated forms ("gelu_tanh", "relu", "silu",
    "clamp_glu" with ``limit``), one matrix for "relu_sq".  Where the few-rows kernel or the tiles pay,
    one kernel, the products stay fp32 up to the activation's result."""
    if _few_rows(x, w) and _few_rows_pays(x.shape[0], w.shape[0], x.shape[1], act):
        n = w.shape[0] if act == "relu_sq" else w.shape[0] // 2
        y = torch.empty(x.shape[0], n, dtype=x.dtype, device=x.device)
        native_mixers().few_rows_gemm(y, x, w, None, FEW_ACTS[act], float(limit))
        return y
    y = _tile_gemm(x, w, None, act, limit)
    if y is not None:
        return y
    u = torch.nn.functional.linear(x, w)
    if act == "relu_sq":
        return relu_sq(u)
    return clamp_swiglu(u, limit) if act == "clamp_glu" else {"gelu_tanh": gelu_glu, "relu": relu_glu, "silu": silu_glu,
                                                              "silu_glu": silu_glu}[act](u)


# ---------------------------------------------------------------------------------
# residual stream (fp32) and norms
# ---------------------------------------------------------------------------------

def embed_rows(ids: torch.Tensor, table: torch.Tensor, scale: float = 1.0,
               positions: Optional[torch.Tensor] = None,
               pos_freqs: Optional[torch.Tensor] = None) -> torch.Tensor:
    """fp32 residual rows table[ids] * scale; with ``pos_freqs`` (fp32 [ceil(width/2)],
    :func:`sinusoid_freqs`) a sinusoidal position vector is added: column 2i gets
    sin(p f_i), column 2i+1 cos(p f_i), angles in fp32."""
    if ids.is_cuda:
        return _embed_norm(ids, table, scale, positions, pos_freqs, None, 0, None, None, None, 0.0)[0]
    return ref.embed_rows(ids, table, scale, positions, pos_freqs)


def _embed_norm(ids, table, scale, positions, freqs, pair, norm, w, b, out_dtype, eps):
    x = torch.empty(ids.shape[0], table.shape[1], dtype=torch.float32, device=ids.device)
    out = torch.empty(x.shape, dtype=out_dtype, device=ids.device) if out_dtype is not None else None
    pairs, hashed = [], []
    if pair is not None:
        ptable, mul_prev, mul_cur, buckets, seg, last_tok = pair
        pairs, hashed = [ptable, seg.start, seg.pos0, seg.slot, last_tok], [int(mul_prev), int(mul_cur), int(buckets), seg.num]
    native_mixers().embed_norm(x, ids, table, float(scale), positions if freqs is not None else None, freqs, pairs, hashed, norm, out,
                               w, b, float(eps))
    return x, out


def embed_norm_rows(ids: torch.Tensor, table: torch.Tensor, scale: float, eps: float, out_dtype, w: Optional[torch.Tensor] = None,
                    b: Optional[torch.Tensor] = None, positions: Optional[torch.Tensor] = None,
                    pos_freqs: Optional[torch.Tensor] = None, pair: Optional[tuple] = None):
    """The rows of :func:`embed_rows`, or with ``pair`` (table, mul_prev, mul_cur, buckets, segments, last tokens) of
    :func:`pair_embed_rows`, and what the first sublayer reads of them, one launch where a row is whole fours: (x, rms_norm(x) * w
    in ``out_dtype``) with ``w``; with ``b`` as well x itself is layer_norm(x) * w + b and comes in ``out_dtype`` beside it."""
    width = table.shape[1]
    if ids.is_cuda and w is not None and native_mixers().embed_norm_fits(width) and \
            all(t is None or t.data_ptr() % 16 == 0 for t in (table, w, b, None if pair is None else pair[0])):
        own = b is not None and out_dtype == torch.float32                    # (the residual itself)
        x, h = _embed_norm(ids, table, scale, positions, pos_freqs, pair, 1 if b is None else 2, w, b, None if own else out_dtype, eps)
        return x, x if own else h
    x = embed_rows(ids, table, scale, positions, pos_freqs) if pair is None else pair_embed_rows(ids, table, scale, *pair)
    if w is None:
        return x, None
    return x, rms_norm_rows(x, w, eps, out_dtype) if b is None else add_layer_norm_rows(x, None, w, b, eps, out_dtype)


sinusoid_freqs = ref.sinusoid_freqs


def layer_norm_rows(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor, eps: float, out_dtype) -> torch.Tensor:
    """(x - mean) / sqrt(var + eps) * w + b of fp32 rows x (var = mean squared deviation),
    rounded to ``out_dtype``; x is left as it is."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        native_mixers().layer_norm(x, None, w, b, out, None, None, None, eps)
        return out
    return ref.layer_norm_rows(x, w, b, eps, out_dtype)


class ExpertParts(NamedTuple):
    """The outputs of a mixture of few rows not yet summed: row t is sum_k wts[t, k] * d[t * top + k] + shared[t] (times the
    sigmoid of gate[t], if there is one).  The norm steps take it for their ``y`` and sum it as they read it, which saves a
    launch between the experts and the norm (4.6 us of a decode step per layer).  Without ``wts`` every one is 1: the parts of
    a product (:func:`linear_out`)."""
    d: torch.Tensor                   # fp32 [rows * top, width]
    wts: Optional[torch.Tensor]       # fp32 [rows, top]
    shared: Optional[torch.Tensor]    # fp32 [rows, width]
    gate: Optional[torch.Tensor]      # fp32 [rows]


class SortedParts(NamedTuple):
    """The same of many rows (:func:`experts_many`): row t is sum_k wts[t, k] * d[place[t, k]] + shared[t] (times sigmoid(h[t] .
    gate_w), if there is one), for :func:`add_rms_norm_rows` and :func:`add_layer_norm_rows`."""
    d: torch.Tensor                   # bf16 [rows * top, width], sorted by expert
    place: torch.Tensor               # int32, its first rows * top entries
    wts: torch.Tensor                 # fp32 [rows, top]
    shared: Optional[torch.Tensor]    # bf16 [rows, width]
    h: torch.Tensor                   # bf16 [rows, width]
    gate_w: Optional[torch.Tensor]    # bf16 [width]


def add_layer_norm_rows(residual: torch.Tensor, y: Optional[torch.Tensor], w: torch.Tensor, b: torch.Tensor,
                        eps: float, out_dtype, next_norm: Optional[tuple] = None) -> torch.Tensor:
    """residual (fp32, in place) += layer_norm(y) * w + b, or, without y, residual <-
    layer_norm(residual) * w + b.  Returns the new residual in ``out_dtype`` (the residual
    itself when that is fp32): what the next sublayer of a post-norm stack reads; with ``next_norm`` (weight, bias) its layer
    norm by these instead.  y may be :class:`ExpertParts` or :class:`SortedParts`."""
    if isinstance(y, (ExpertParts, SortedParts)):
        cast = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
        f = native_mixers().layer_norm_sorted if isinstance(y, SortedParts) else native_mixers().layer_norm_experts
        f(residual, *y, w, b, cast, *(next_norm or (None, None)), eps)
        return cast
    if residual.is_cuda:
        cast = None if out_dtype == torch.float32 and next_norm is None else \
            torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
        native_mixers().layer_norm(residual, y, w, b, None, cast, *(next_norm or (None, None)), eps)
        return residual if cast is None else cast
    h = ref.add_layer_norm_rows(residual, y, w, b, eps, out_dtype)
    return h if next_norm is None else ref.layer_norm_rows(residual, *next_norm, eps, out_dtype)


def tanh_cap_(x: torch.Tensor, cap: float) -> torch.Tensor:
    """fp32 x <- cap * tanh(x / cap) in place; infinite entries stay as they are."""
    if x.is_cuda:
        native_mixers().tanh_cap(x, float(cap))
        return x
    return ref.tanh_cap_(x, cap)


def rms_norm_rows(x: torch.Tensor, w: torch.Tensor, eps: float, out_dtype,
                  add_vec: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = x / sqrt(mean(x^2) + eps) * w of fp32 rows x, rounded to ``out_dtype``;
    with ``add_vec`` the rows are first updated in place, x += add_vec."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        native_mixers().add_rms_norm(x, None, None, add_vec, w, out, None, eps)
        return out
    return ref.rms_norm_rows(x, w, eps, out_dtype, add_vec)


def add_rms_norm_rows(residual: torch.Tensor, y: torch.Tensor, wb: Optional[torch.Tensor], eps: float,
                      add_vec: Optional[torch.Tensor] = None, next_w: Optional[torch.Tensor] = None,
                      out_dtype=None, want_cast: bool = False):
    """residual (fp32, in place) += rms_norm(y) * wb (y as it is without ``wb``) (+ add_vec); returns
    (rms_norm(residual) * next_w or None, residual cast to out_dtype or None).  y may be :class:`ExpertParts` or
    :class:`SortedParts`."""
    if isinstance(y, (ExpertParts, SortedParts)):
        out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device) if next_w is not None else None
        cast = torch.empty(residual.shape, dtype=out_dtype, device=residual.device) if want_cast else None
        f = native_mixers().add_rms_norm_sorted if isinstance(y, SortedParts) else native_mixers().add_rms_norm_experts
        f(residual, *y, wb, add_vec, next_w, out, cast, eps)
        return out, cast
    out_dtype = out_dtype or y.dtype
    if residual.is_cuda:
        out = torch.empty(residual.shape, dtype=out_dtype, device=y.device) if next_w is not None else None
        cast = torch.empty(residual.shape, dtype=out_dtype, device=y.device) if want_cast else None
        native_mixers().add_rms_norm(residual, y, wb, add_vec, next_w, out, cast, eps)
        return out, cast
    return ref.add_rms_norm_rows(residual, y, wb, eps, add_vec, next_w, out_dtype, want_cast)


def _rows_or_parts(y, rows):
    """(A norm step's rows or a product's :class:`ExpertParts`, how many a row has)."""
    if not isinstance(y, ExpertParts):
        return y, 1
    if y.wts is not None or y.shared is not None:
        raise ValueError("a mixture's results where a product's parts are read")
    return y.d, y.d.shape[0] // rows


def add_scaled_rms_norm_rows(residual: torch.Tensor, y1: Optional[torch.Tensor], y2: Optional[torch.Tensor],
                             mult: float, next_w: Optional[torch.Tensor], eps: float, out_dtype):
    """residual (fp32, in place) += mult * (y1 + y2); returns rms_norm(residual) * next_w in
    ``out_dtype`` (None without ``next_w``).  y1 and y2 may be fp32 or bf16 each; y2, or
    both, may be absent (then only the norm is taken), or be a product's parts.  The step between the layers of a
    stack whose mixer and feed-forward read one shared norm and are added together."""
    if residual.is_cuda:
        out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device) if next_w is not None else None
        (y1, p1), (y2, p2) = _rows_or_parts(y1, residual.shape[0]), _rows_or_parts(y2, residual.shape[0])
        native_mixers().add_scaled_rms_norm(residual, y1, y2, float(mult), next_w, out, eps, p1, p2)
        return out
    return ref.add_scaled_rms_norm_rows(residual, y1, y2, mult, next_w, eps, out_dtype)


def add_norm_shift_rows(residual: torch.Tensor, y: Optional[torch.Tensor], wb: Optional[torch.Tensor], w: torch.Tensor,
                        shift: torch.Tensor, eps: float, out_dtype, prev_state: torch.Tensor, seg: "Segments"):
    """One step between layers with a token shift: x = residual + rms_norm(y) * wb (x =
    residual without y), h = rms_norm(x) * w, and what the next sublayer reads is
    h + (h' - h) * shift element by element, h' being the h of the token before in its
    sequence (zeros for a sequence's first token).  ``prev_state`` [slots, width] fp32
    holds each sequence's last h and is updated.  Returns (x fp32, shifted h in
    ``out_dtype``); x may or may not be ``residual`` itself, which must not be read
    afterwards.  h and the shift are fp32, rounded once.  y may be :class:`ExpertParts` where no segment has two rows."""
    if isinstance(y, ExpertParts):
        h = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
        native_mixers().add_norm_shift_experts(residual, *y, wb, w, shift, h, prev_state, seg.start, seg.pos0, seg.slot,
                                               seg.num, eps)
        return residual, h
    if residual.is_cuda:
        h = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
        # rows read their predecessor's old residual: in place only if no row has one in this step
        x = residual if y is None or seg.max_rows <= 1 else torch.empty_like(residual)
        native_mixers().add_norm_shift(x, residual, y, wb, w, shift, h, prev_state, seg.start, seg.pos0, seg.slot,
                                       seg.num, seg.max_rows, eps)
        return x, h
    return ref.add_norm_shift_rows(residual, y, wb, w, shift, eps, out_dtype, prev_state, seg)


def dual_rms_mean(a, b, wa: torch.Tensor, wb: torch.Tensor, eps: float, scale: float = 0.5,
                  rows: Optional[int] = None) -> torch.Tensor:
    """fp32 scale * (rms_norm(a) * wa + rms_norm(b) * wb) of two rows of equal width: the
    outputs of two mixers that run side by side, each normed on its own.  a and b may be a product's parts of ``rows`` rows."""
    if wa.is_cuda:
        (a, pa), (b, pb) = _rows_or_parts(a, rows), _rows_or_parts(b, rows)
        out = torch.empty(a.shape[0] // pa, a.shape[1], dtype=torch.float32, device=a.device)
        native_mixers().dual_rms_mean(out, a, b, wa, wb, eps, float(scale), pa, pb)
        return out
    return ref.dual_rms_mean(a, b, wa, wb, eps, scale)


def scaled_pair_rows(a: torch.Tensor, a_scale: float, o: torch.Tensor, gate: torch.Tensor, o_scale: float, eps: float,
                     heads: int, dv: int, out_dtype) -> torch.Tensor:
    """Rows [a_scale * a | o_scale * head_norm(o) * silu(gate)] in ``out_dtype``: what the
    joint output product of two side-by-side mixers reads.  a fp32 [T, n]; o fp32 [T,
    heads*dv], every head divided by its root mean square; gate [T, heads*dv] (may be a
    column range)."""
    if o.is_cuda:
        out = torch.empty(o.shape[0], a.shape[1] + heads * dv, dtype=out_dtype, device=o.device)
        native_mixers().scaled_pair_rows(out, a, float(a_scale), o, gate, float(o_scale), eps, heads, dv)
        return out
    return ref.scaled_pair_rows(a, a_scale, o, gate, o_scale, eps, heads, dv, out_dtype)


def pair_embed_add(x: torch.Tensor, ids: torch.Tensor, table: torch.Tensor, mul_prev: int, mul_cur: int,
                   buckets: int, seg: "Segments", last_tok: torch.Tensor) -> torch.Tensor:
    """x (fp32 rows, in place) += table[(prev * mul_prev + cur * mul_cur) mod buckets], prev
    being the token before the row's own in its sequence; a sequence's first token takes
    row ``buckets``.  The token before a segment's first row comes from ``last_tok``
    [slots] int32 (the sequence's state slot), which is then set to the segment's last
    token."""
    if x.is_cuda:
        native_mixers().pair_embed_add(x, ids, table, int(mul_prev), int(mul_cur), int(buckets), seg.start,
                                       seg.pos0, seg.slot, seg.num, last_tok)
        return x
    return ref.pair_embed_add(x, ids, table, mul_prev, mul_cur, buckets, seg, last_tok)


def pair_embed_rows(ids: torch.Tensor, embed: torch.Tensor, scale: float, table: torch.Tensor, mul_prev: int,
                    mul_cur: int, buckets: int, seg: "Segments", last_tok: torch.Tensor) -> torch.Tensor:
    """:func:`embed_rows` and :func:`pair_embed_add` in one launch: fp32 rows
    embed[ids] * scale + table[hash(previous token, token)]."""
    if ids.is_cuda:
        return _embed_norm(ids, embed, scale, None, None, (table, mul_prev, mul_cur, buckets, seg, last_tok), 0, None, None, None, 0.0)[0]
    return ref.pair_embed_add(ref.embed_rows(ids, embed, scale), ids, table, mul_prev, mul_cur, buckets, seg, last_tok)


def sigmoid_gate(o: torch.Tensor, g: torch.Tensor, out_dtype) -> torch.Tensor:
    """o * sigmoid(g) element by element (o fp32 [T, n]; g [T, n], may be a column range of
    wider rows), rounded to ``out_dtype``."""
    if o.is_cuda:
        out = torch.empty(o.shape, dtype=out_dtype, device=o.device)
        native_mixers().sigmoid_gate(out, o, g)
        return out
    return ref.sigmoid_gate(o, g, out_dtype)


# ---------------------------------------------------------------------------------
# rotary positions (partial, rotate-half pairs, fp32 angles)
# ---------------------------------------------------------------------------------

rope_table = ref.rope_table
ramp_frequencies = ref.ramp_frequencies
distance_bias_table = ref.distance_bias_table


# ---------------------------------------------------------------------------------
# short convolution + gated delta rule (recurrent state slots)
# ---------------------------------------------------------------------------------

def short_conv_silu(x: torch.Tensor, conv_w: torch.Tensor, conv_state: torch.Tensor, seg: Segments,
                    bias: Optional[torch.Tensor] = None):
    """Per-channel causal convolution over time (+ ``bias`` [C] fp32), then SiLU.
    ``conv_w`` [C, taps] fp32 (last column = the current row); ``conv_state`` [slots,
    taps-1, C] fp32 holds each sequence's last inputs and is updated; a segment at
    position 0 starts from zeros.  ``x`` may be a column range of wider rows."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        native_mixers().short_conv_silu(out, x, conv_w, bias, conv_state, seg.start, seg.pos0, seg.slot,
                                        seg.num, seg.max_rows)
        return out
    return ref.short_conv_silu(x, conv_w, conv_state, seg, bias)


def gated_delta_rule(qkv, a, b, a_log, dt_bias, state, seg: Segments, heads: int, kv_heads: int,
                     dk: int, dv: int) -> torch.Tensor:
    """Gated delta rule with one decay per head and key channel.

    Rows of ``qkv`` are [q (kv_heads*dk) | k (kv_heads*dk) | v (heads*dv)] after the
    short convolution; q and k are unit-normalised per head here (q also * dk^-1/2),
    beta = sigmoid(b), decay = exp(-exp(a_log) * softplus(a + dt_bias)).  Per head and
    row:  S <- decay (.) S (rows of S);  u = beta (v - S^T k);  S <- S + k u^T;
    o = S^T q.  ``state`` [slots, heads, dk, dv] fp32 is read (zeros at position 0)
    and left at the segment's last row.  Returns o fp32 [T, heads*dv]."""
    if qkv.is_cuda:
        o = torch.empty(qkv.shape[0], heads * dv, dtype=torch.float32, device=qkv.device)
        chunk = CHANNEL_CHUNK_ROWS if _delta_chunks_pay(seg, heads, dk, dv) else NO_CHUNKS
        native_mixers().gated_delta_rule(o, qkv, a, b, a_log, dt_bias, state, seg.start, seg.pos0, seg.slot, seg.num,
                                         seg.max_rows, heads, kv_heads, dk, dv, _walk_below(seg, chunk), chunk)
        return o
    return ref.gated_delta_rule(qkv, a, b, a_log, dt_bias, state, seg, heads, kv_heads, dk, dv)


def conv_delta_prep(qkv, a, b, conv_w, conv_state, a_log, dt_bias, seg: Segments, heads: int, kv_heads: int, dk: int,
                    dv: int):
    """What the delta rule with one decay per head reads, in one launch over rows [q
    (kv_heads*dk) | k (kv_heads*dk) | v (heads*dv)] of a fused projection: per-channel causal
    convolution over time (as in :func:`conv_attn_prep`) and silu, q and k made unit vectors
    per head (x / sqrt(sum x^2 + 1e-6); q also * dk^-1/2), the decay's logarithm
    -exp(a_log) * softplus(a + dt_bias) and beta = sigmoid(b) (a, b [T, heads], may be column
    ranges).  All fp32: (q [T, kv_heads, dk], k, v [T, heads, dv], log decay [T, heads],
    beta [T, heads])."""
    if qkv.is_cuda:
        t, dev = qkv.shape[0], qkv.device
        f32 = dict(dtype=torch.float32, device=dev)
        q, k = torch.empty(t, kv_heads, dk, **f32), torch.empty(t, kv_heads, dk, **f32)
        v = torch.empty(t, heads, dv, **f32)
        lg, beta = torch.empty(t, heads, **f32), torch.empty(t, heads, **f32)
        native_mixers().conv_delta_prep(q, k, v, lg, beta, qkv, a, b, conv_w, conv_state, a_log, dt_bias, seg.start,
                                        seg.pos0, seg.slot, seg.num, seg.max_rows)
        return q, k, v, lg, beta
    return ref.conv_delta_prep(qkv, a, b, conv_w, conv_state, a_log, dt_bias, seg, heads, kv_heads, dk, dv)


# rows from which a segment's recurrence runs chunk by chunk as matrix products; shorter segments
# and decode rows are walked row by row
CHUNK_ROWS = 32
# the same with a decay per channel, and for the state-space scan, whose walks are cheaper and whose
# chunk form has four launches.  One segment of 64 / 100 / 200 / 777 rows, 16 (state space: 32) heads of
# 128 x 128, us: delta rule 58 61 70 99 (walk 43 62 114 423), linear attention 38 39 43 66 (25 39 70
# 245), state space 40 41 46 98 (19 28 49 169; four segments of 200: 108, walk 97)
CHANNEL_CHUNK_ROWS = 96
SSD_CHUNK_ROWS = 256
# of the state-space scan where its chunks take one launch for the weights and one for the walk over them (csrc/mixers/state_scan.hip):
# us, 32 heads of 128 x 128, a row at a time beside it: one segment of 40 rows 14 16, of 64 12 18, eight of 40 40 49, 64 of 33 244 264
SCAN_ROWS = 64
NO_CHUNKS = 1 << 30


def _chunks_pay(seg: Segments, least: int, heads: int, dk: int, dv: int, cols: int, walk, launch: float, link: float,
                short_entry: float, products) -> bool:
    """Whether a step's segments of ``least`` rows or more run in chunks (and only the others in walks): by the time, us, of
    both forms, fitted to 2238 steps of 1 to 65 segments, 1 to 128 heads of 8 x 8 to 128 x 256 (the form chosen takes 1.004 to
    1.008 times the better one's time in the mean, 1.25 times or more in one step of a
    hundred; the chunks' a tenth up, their fit is the coarser).
    A walk takes a row after the other, ``cols`` state columns a workgroup and a few hundred workgroups at a time (``walk``:
    launch, a row and more per dk, workgroups at a time and fewer per dk, a state's entry, a row's preparation per head).
    Chunks take ``launch``, ``products`` (of chunks times heads, dk, tiles of 64 columns), ``link`` for each of the longest
    segment's in the carry and, after the walk of the others, ``short_entry`` for an entry of those states."""
    if seg.host is None or seg.max_rows < least:
        return True
    lens = [b - a for a, b in zip(seg.host[0][:-1], seg.host[0][1:])]
    short = [n for n in lens if n < least]

    def walked(lens):
        begin, row, row_dk, room, room_dk, entry, prep = walk
        busy = sum(lens) * heads * (-(-dv // cols)) / max(room - room_dk * dk, 50.0)
        return begin + (row + row_dk * dk) * (max(lens) ** 4 + busy ** 4) ** 0.25 + \
            heads * (entry * len(lens) * dk * dv + prep * sum(lens))

    pad = 16 if dk <= 16 else 32 if dk <= 32 else 64 if dk <= 64 else 128
    chunked = launch + link * ((max(lens) + 63) // 64) + \
        products(heads * sum((n + 63) // 64 for n in lens if n >= least), pad, -(-dv // 64))
    if short:
        chunked += walked(short) + short_entry * heads * len(short) * dk * dv
    return 1.1 * chunked <= walked(lens)


def _turns(units: int, turn: int, share: float) -> float:
    """``units`` workgroups, ``share`` of their time in whole turns of the chip."""
    return (1 - share) * units + share * turn * -(-units // turn)


def _delta_chunks_pay(seg: Segments, heads: int, dk: int, dv: int) -> bool:
    """us, chunks (walks): 32 heads of 64 x 64, 16 and 64 segments of 100 rows 124 489 (113 403), 32 of 256 472 (497); of
    16 x 32 79 264 (51 130), 266 (168); 16 heads of 128 x 128 135 554 (261 1057)."""
    return _chunks_pay(seg, CHANNEL_CHUNK_ROWS, heads, dk, dv, 32, (7.0, 0.18, 0.0025, 940, 5.5, 1.8e-6, 6.4e-4), 11, 1.0,
                       2.2e-6, lambda n, pad, tall: _turns(n, 256 if pad >= 64 else 512, 0.3) *
                       (0.041 + 4.9e-6 * pad * pad + tall * (3.3e-4 * pad + 0.013)))


def _linear_chunks_pay(seg: Segments, heads: int, dk: int, dv: int) -> bool:
    """The same of linear attention: 128 heads of 64 x 16, 32 segments of 130 rows 625 (248); 128 of 8 x 8, 8 of 130 67 (44);
    64 of 32 x 32 55 (44); 16 of 128 x 128, one of 200 43 (70); 4 of 64 x 128, two of 130 23 (36)."""
    return _chunks_pay(seg, CHANNEL_CHUNK_ROWS, heads, dk, dv, 16, (5.6, 0.12, 0.0014, 600, 1.4, 5.2e-6, 1.3e-5), 10, 0.71,
                       2.8e-6, lambda n, pad, tall: _turns(n, 256 if pad >= 64 else 512, 0.3) *
                       (0.0068 + 3.1e-6 * pad * pad + tall * (2.8e-4 * pad + 0.0089)))


def _ssd_chunks_pay(seg: Segments, heads: int, n: int, dv: int) -> bool:
    """The same of the state-space scan: 16 heads of 128 x 128, 32 segments of 256 rows 420 (388), four of 2000 370 (459), one
    of 300 beside 64 decode rows 120 (86); of 128 x 256, 4 heads, eight of 300 95 (78); 32 of 64 x 64 82 (74), 32 of 256
    193 (201); of 16 x 32 99 (87); 128 heads of 16 x 32, one of 3000 beside 64 decode rows 187 (436)."""
    return _chunks_pay(seg, SSD_CHUNK_ROWS, heads, n, dv, 16, (5.0, 0.13, 5.7e-4, 1100, 4.3, 1.2e-6, 0), 14, 0.28,
                       3.1e-6, lambda n, pad, tall: _turns(n * tall, 512 if pad >= 64 else 768, 0.42) *
                       (0.015 + 2.4e-4 * pad + 2e-6 * pad * pad))


def head_delta_rule(q, k, v, log_decay, beta, state, seg: Segments) -> torch.Tensor:
    """Gated delta rule with one decay per head, on the outputs of :func:`conv_delta_prep`.
    Per head and row:  S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q with g =
    exp(log_decay).  ``state`` [slots, heads, dk, dv] fp32 is read (zeros at position 0) and
    left at the segment's last row.  Returns o fp32 [T, heads*dv]."""
    if v.is_cuda:
        t, heads, dv = v.shape
        o = torch.empty(t, heads * dv, dtype=torch.float32, device=v.device)
        native_mixers().head_delta_rule(o, q, k, v, log_decay, beta, state, seg.start, seg.pos0, seg.slot, seg.num,
                                        seg.max_rows, _walk_below(seg, CHUNK_ROWS), CHUNK_ROWS)
        return o
    return ref.head_delta_rule(q, k, v, log_decay, beta, state, seg)


def retention(qkv, table, rot_dims: int, log_decay, state, seg: Segments, heads: int, dk: int, dv: int,
              interleaved: bool = False) -> torch.Tensor:
    """Linear attention with one fixed decay per head.  Rows of ``qkv`` are [q (heads*dk) | k
    (heads*dk) | v (heads*dv) | ...]; q and k are rotated by position (``table`` =
    :func:`rope_table` over the first ``rot_dims`` entries of a head, pairs (i, i + rot_dims/2),
    or (2i, 2i + 1) if ``interleaved``; None: no rotation), k is scaled by dk^-1/2.  Per head
    and row:  S <- d S + k v^T;  o = S^T q with d = exp(log_decay[head]) (``log_decay`` fp64
    [heads]: powers of d are formed from it).  ``state`` [slots, heads, dk, dv] fp32 is read
    (zeros at position 0) and left at the segment's last row.  Returns o fp32 [T, heads*dv]."""
    if qkv.is_cuda:
        o = torch.empty(qkv.shape[0], heads * dv, dtype=torch.float32, device=qkv.device)
        native_mixers().retention(o, qkv, table, rot_dims, bool(interleaved), log_decay, state, seg.start, seg.pos0,
                                  seg.slot, seg.num, seg.max_rows, heads, dk, dv, _walk_below(seg, CHUNK_ROWS), CHUNK_ROWS)
        return o
    return ref.retention(qkv, table, rot_dims, interleaved, log_decay, state, seg, heads, dk, dv)


def _walk_below(seg: Segments, chunk_rows: int) -> bool:
    """Whether a step may hold segments short enough to be walked row by row."""
    if seg.max_rows < chunk_rows or seg.host is None:
        return True
    start = seg.host[0]
    return min(b - a for a, b in zip(start[:-1], start[1:])) < chunk_rows


def gated_linear_attention(qkv, a, a_bias, tau: float, state, seg: Segments, heads: int, dk: int,
                           dv: int) -> torch.Tensor:
    """Linear attention with a decay per head and key channel.

    Rows of ``qkv`` are [q (heads*dk) | k (heads*dk) | v (heads*dv) | ...]; q is scaled by
    dk^-1/2; decay = sigmoid(a + a_bias)^(1/tau), evaluated as exp(log sigmoid(.) / tau) in
    fp32.  Per head and row:  S <- diag(decay) S + k v^T;  o = S^T q.  ``state`` [slots,
    heads, dk, dv] fp32 is read (zeros at position 0) and left at the segment's last row.
    Returns o fp32 [T, heads*dv]."""
    if qkv.is_cuda:
        o = torch.empty(qkv.shape[0], heads * dv, dtype=torch.float32, device=qkv.device)
        chunk = CHANNEL_CHUNK_ROWS if _linear_chunks_pay(seg, heads, dk, dv) else NO_CHUNKS
        native_mixers().gated_linear_attention(o, qkv, a, a_bias, float(tau), state, seg.start, seg.pos0,
                                               seg.slot, seg.num, seg.max_rows, heads, dk, dv,
                                               _walk_below(seg, chunk), chunk)
        return o
    return ref.gated_linear_attention(qkv, a, a_bias, tau, state, seg, heads, dk, dv)


ROW_CHANNEL, ROW_HEAD, ROW_LINEAR = 0, 1, 2


def row_step(kind: int, x, a, b, gate, conv_w, conv_state, a_log, dt_bias, tau: float, norm, eps: float, silu: bool, state,
             seg: Segments, heads: int, kv_heads: int, dk: int, dv: int) -> Optional[torch.Tensor]:
    """One row per sequence (a decode step) of a recurrent mixer, from its projection to the rows of its output product, in
    one launch: :func:`short_conv_silu` and :func:`gated_delta_rule` (ROW_CHANNEL), :func:`conv_delta_prep` and
    :func:`head_delta_rule` (ROW_HEAD) or :func:`gated_linear_attention` (ROW_LINEAR; ``dt_bias`` its a_bias), and
    :func:`head_rms_gate` in x's dtype.  None where the kernel does not take the step: segments of several rows, heads that
    share q and k (whose history several workgroups would write), sizes."""
    if not x.is_cuda or seg.max_rows != 1 or kv_heads != heads or \
            not native_mixers().row_step_fits(kind, 0 if conv_w is None else conv_w.shape[1], dk, dv) or \
            state.data_ptr() % 16:
        return None
    out = torch.empty(x.shape[0], heads * dv, dtype=x.dtype, device=x.device)
    native_mixers().row_step(kind, out, x, a, b, gate, conv_w, conv_state, a_log, dt_bias, float(tau), norm, eps, silu, state,
                             seg.start, seg.pos0, seg.slot, seg.num, heads, dk, dv)
    return out


def group_step(xbc, z, dt, conv_w, conv_b, conv_state, a_log, dt_bias, d_skip, norm, eps: float, norm_groups: int, state,
               seg: Segments, heads: int, groups: int, n: int, dv: int) -> Optional[torch.Tensor]:
    """One row per sequence (a decode step) of a state-space mixer in one launch: :func:`short_conv_silu`, :func:`ssd_scan` and
    :func:`gate_group_norm` in xbc's dtype.  None where the kernel does not take the step: segments of several rows, norm groups
    that are not those of B and C, sizes."""
    if not xbc.is_cuda or seg.max_rows != 1 or norm_groups != groups or \
            state.data_ptr() % 16 or not native_mixers().group_step_fits(conv_w.shape[1], heads, groups, n, dv):
        return None
    out = torch.empty(xbc.shape[0], heads * dv, dtype=xbc.dtype, device=xbc.device)
    native_mixers().group_step(out, xbc, z, dt, conv_w, conv_b, conv_state, a_log, dt_bias, d_skip, norm, eps, state, seg.start,
                               seg.pos0, seg.slot, seg.num, heads, groups, n, dv)
    return out


def head_rms_gate(o, w, gate_pre, eps: float, heads: int, dv: int, out_dtype, silu: bool = False):
    """Per head: o / rms(o) * w * sigmoid(gate_pre) (or * silu(gate_pre)), rounded to
    ``out_dtype``; ``gate_pre`` [T, heads*dv] may be a column range of wider rows."""
    if o.is_cuda:
        out = torch.empty(o.shape, dtype=out_dtype, device=o.device)
        native_mixers().head_rms_gate(out, o, w, gate_pre, eps, heads, dv, bool(silu))
        return out
    return ref.head_rms_gate(o, w, gate_pre, eps, heads, dv, out_dtype, silu)


# ---------------------------------------------------------------------------------
# latent attention (paged cache of [normed latent | rotated shared key])
# ---------------------------------------------------------------------------------

def latent_kv_write(dkv, norm_w, eps: float, table, rot_dims: int, positions, slot_mapping, cache,
                    rank: int, interleaved: bool = False):
    """Cache row = [rms_norm(dkv[:rank]) * norm_w | rope(dkv[rank:])] at each row's slot
    (rotary pairs (i, i + rot_dims/2), or (2i, 2i + 1) if ``interleaved``)."""
    if dkv.is_cuda:
        native_mixers().latent_kv_write(dkv, norm_w, eps, table, rot_dims, positions, slot_mapping,
                                        cache, rank, bool(interleaved), None, None, None)
    else:
        ref.latent_kv_write(dkv, norm_w, eps, table, rot_dims, positions, slot_mapping, cache, rank, interleaved)


def latent_down_prep(dq, q_norm_w, dkv, norm_w, eps: float, table, rot_dims: int, positions, slot_mapping, cache,
                     rank: int, interleaved: bool = False):
    """:func:`latent_kv_write` of ``dkv`` and the queries' latent in one launch: returns
    rms_norm(dq) * q_norm_w in dq's dtype.  ``dq`` and ``dkv`` are adjacent column ranges
    [q latent | kv latent | rotated part] of one product."""
    if dkv.is_cuda:
        cq = torch.empty(dq.shape, dtype=dq.dtype, device=dq.device)
        native_mixers().latent_kv_write(dkv, norm_w, eps, table, rot_dims, positions, slot_mapping, cache, rank,
                                        bool(interleaved), cq, dq, q_norm_w)
        return cq
    return ref.latent_down_prep(dq, q_norm_w, dkv, norm_w, eps, table, rot_dims, positions, slot_mapping, cache, rank,
                                interleaved)


def latent_q_rope(q, table, rot_dims: int, positions, heads: int, dn: int, dr: int, interleaved: bool = False):
    """q rows [heads x (dn unrotated | dr rotated)] -> fp32 ([T, heads, dn], [T, heads, dr]
    rotated: entry i paired with i + rot_dims/2, or 2i with 2i + 1 if ``interleaved``)."""
    if q.is_cuda:
        t = q.shape[0]
        qn = torch.empty(t, heads, dn, dtype=torch.float32, device=q.device)
        qr = torch.empty(t, heads, dr, dtype=torch.float32, device=q.device)
        native_mixers().latent_q_rope(qn, qr, q, table, rot_dims, positions, heads, dn, dr, bool(interleaved))
        return qn, qr
    return ref.latent_q_rope(q, table, rot_dims, positions, heads, dn, dr, interleaved)


# rows up to which a fp32 matrix per head goes through head_product.hip: it takes eight rows at a time, the library's batched
# product all of them, in two launches with what is around it.  us of both products at 3 8 16 24 32 rows (rotation, gate and
# rounding in the second): 16 heads, 128 -> 512 -> 128: 8 11 17 24 31 (library 23 23 22 22 22); 128 heads 15 22 36 52 65
# (59 60 59 65 62); 40 heads, 64 -> 256 -> 64: 7 10 16 22 27 (19 20 20 22 22)
HEAD_PRODUCT_ROWS = 16
# rows from which the values' product goes through head_tiles.hip where the matrix allows it; the queries' always does.  us of
# queries + values, 16 heads, 128 -> 512 -> 128, 1 4 8 16 64 rows: 2.9 + 4.7, 3.0 + 4.8, 3.2 + 4.9, 3.4 + 5.1, 4.8 + 6.1 (head_product.hip
# 3.1 + 3.2, 3.8 + 4.4, 4.7 + 6.1, 7.4 + 10.2; library 10.6 + 20.1 at 64); 300 and 4096 rows 7.5 + 11 and 44 + 34 (library 17 + 14 and
# 104 + 89)
HEAD_TILES_ROWS = 5


def _head_product(rows: int, w) -> bool:
    """Whether the kernels of few rows (csrc/mixers/head_product.hip) take a fp32 matrix per head."""
    return bool(w.is_cuda and rows <= HEAD_PRODUCT_ROWS and w.dtype == torch.float32 and w.is_contiguous()
                and w.data_ptr() % 16 == 0 and native_mixers().head_product_fits(w.shape[1], w.shape[2]))


def head_tiles(w) -> Optional[torch.Tensor]:
    """Matrices ``w`` fp32 [heads, K, N] in the order in which csrc/mixers/head_tiles.hip reads them, bf16 [heads, N / 32, K / 32,
    2, 512], if that holds them: all values are finite bf16 ones (a bf16 checkpoint's); else None."""
    if not w.is_cuda or w.dtype != torch.float32 or not native_mixers().head_tiles_fits(w.shape[1], w.shape[2]):
        return None
    b = w.to(torch.bfloat16)
    if not bool(((b.float() == w) & w.isfinite()).all()):
        return None
    h, k, n = w.shape
    # K = (step, hi, e), N = (pair, tile, lo): a lane (hi, lo) holds 8 entries of column lo of a tile
    b = b.view(h, k // 32, 4, 8, n // 32, 2, 16).permute(0, 4, 1, 5, 2, 6, 3)
    return b.reshape(h, n // 32, k // 32, 2, 512).contiguous()


def latent_q_absorb(q, wuk, table, rot_dims: int, positions, heads: int, dn: int, dr: int, interleaved: bool = False,
                    tiles: Optional[torch.Tensor] = None):
    """:func:`latent_q_rope` and the unrotated parts' way into latent space: (fp32 [heads, T, rank] = q W_uk per head, ``wuk``
    fp32 [heads, dn, rank]; the rotated parts fp32 [T, heads, dr]).  One launch for few rows, and for all of them with ``tiles``
    = :func:`head_tiles` of ``wuk``."""
    t = q.shape[0]

    def reads(n):                                # whether q can be read n entries at a time
        return q.stride(1) == 1 and q.stride(0) % n == 0 and (dn + dr) % n == 0 and q.data_ptr() % (n * q.element_size()) == 0

    tiled = tiles is not None and reads(16 // q.element_size())
    if tiled or (_head_product(t, wuk) and reads(4)):
        qa = torch.empty(heads, t, wuk.shape[2], dtype=torch.float32, device=q.device)
        qr = torch.empty(t, heads, dr, dtype=torch.float32, device=q.device)
        native_mixers().latent_q_absorb(qa, qr, q, tiles if tiled else wuk, table, rot_dims, positions, dr, bool(interleaved), tiled)
        return qa, qr
    qn, qr = latent_q_rope(q, table, rot_dims, positions, heads, dn, dr, interleaved)
    return torch.bmm(qn.transpose(0, 1), wuk), qr


def head_values(ol, wuv, gate, out_dtype, tiles: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Latent-space sums ``ol`` fp32 [heads, T, rank] through ``wuv`` fp32 [heads, rank, dv], times sigmoid(gate[t, h]) if there
    is a ``gate`` [T, heads], as rows [T, heads * dv] in ``out_dtype``.  One launch for few rows, and for all of them with
    ``tiles`` = :func:`head_tiles` of ``wuv``."""
    heads, t = ol.shape[:2]
    tiled = tiles is not None and t >= HEAD_TILES_ROWS
    if ol.is_contiguous() and (tiled or _head_product(t, wuv)):
        out = torch.empty(t, heads * wuv.shape[2], dtype=out_dtype, device=ol.device)
        native_mixers().head_values(out, ol, tiles if tiled else wuv, gate, tiled)
        return out
    o = torch.bmm(ol, wuv)                                               # [heads, T, dv]
    if gate is not None:
        return head_gate(o, gate, out_dtype)
    return o.transpose(0, 1).reshape(t, heads * wuv.shape[2]).to(out_dtype)


def latent_attention(qa, qr, cache, seg: Segments, scale: float, rank: int,
                     skip_from: int = 0, out: Optional[torch.Tensor] = None,
                     sink: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal softmax attention over the paged latent cache.  ``qa`` fp32 [heads, T,
    rank]: the unrotated query parts carried into latent space (q W_uk); ``qr`` fp32
    [T, heads, dr]: the rotated parts.  Score = (qa . c + qr . k_rot) * scale; all heads
    share the cached row, whose first ``rank`` entries are also the value.  Returns
    fp32 [heads, T, rank].  ``skip_from`` > 0: segments of that many rows or more are
    left to the caller (:func:`latent_attention_products`).  ``sink`` fp32 [heads]: the
    softmax's denominator gains exp(sink[h]), as a key with that score and no value."""
    if qa.is_cuda:
        if out is None:
            out = torch.empty_like(qa)
        native_mixers().latent_attention(out, qa, qr, cache, seg.start, seg.pos0, seg.kv_len,
                                         seg.block_tables, seg.num, seg.max_rows, scale, rank,
                                         skip_from, seg.max_kv, sink)
        return out
    r = ref.latent_attention(qa, qr, cache, seg, scale, rank, sink)
    if out is not None:
        out.copy_(r)
        return out
    return r


def causal_softmax(s, rows_per_head: int, first_pos: int, scale: float, out_dtype,
                   sink: Optional[torch.Tensor] = None):
    """P = softmax(scale * S) per row over the keys j <= first_pos + (row mod
    rows_per_head), zeros beyond; S fp32 [heads * rows_per_head, keys].  ``sink`` fp32
    [heads]: exp(sink[head]) joins the denominator."""
    if s.is_cuda:
        p = torch.empty(s.shape, dtype=out_dtype, device=s.device)
        native_mixers().causal_softmax(p, s, rows_per_head, first_pos, scale, sink)
        return p
    return ref.causal_softmax(s, rows_per_head, first_pos, scale, out_dtype, sink)


def head_gate(o, gate, out_dtype) -> torch.Tensor:
    """o fp32 [heads, T, dv] times sigmoid(gate[t, h]), one number per row and head, as rows
    [T, heads*dv] in ``out_dtype``; ``gate`` [T, heads] may be a column range."""
    if o.is_cuda:
        heads, t, dv = o.shape
        out = torch.empty(t, heads * dv, dtype=out_dtype, device=o.device)
        native_mixers().head_gate(out, o, gate)
        return out
    return ref.head_gate(o, gate, out_dtype)


_MM_F32_OUT = {}


def mm_f32(a, b):
    """a @ b with fp32 accumulation and fp32 output (operands fp32, or bf16 where the
    vendor library returns fp32 from bf16 operands; otherwise widened first)."""
    if a.dtype == torch.float32:
        return torch.mm(a, b)
    ok = _MM_F32_OUT.get(a.device.type)
    if ok is None and a.is_cuda:
        try:
            torch.mm(a[:1], b[:, :1], out_dtype=torch.float32)
            ok = True
        except (TypeError, RuntimeError):
            ok = False
        _MM_F32_OUT[a.device.type] = ok
    return torch.mm(a, b, out_dtype=torch.float32) if ok else torch.mm(a.float(), b.float())


# bytes of fp32 scores the product path holds at once
PRODUCT_SCORE_BYTES = 1 << 30


def latent_prefill_ok(qa, cache, rank: int, dtype) -> bool:
    """Whether long segments run in one kernel (csrc/mixers/latent_prefill.hip) instead of two products."""
    return bool(qa.is_cuda and dtype == torch.bfloat16 and cache.dtype == torch.bfloat16
                and native_mixers().latent_prefill_fits(rank, cache.shape[2] - rank, cache.shape[1]))


def _latent_prefill_pays(seg: Segments, heads: int, min_rows: int) -> bool:
    """A workgroup of the one kernel owns 128 (row, head) pairs and walks their keys, 32 in 1.9 us, so few
    pairs with many earlier keys leave the chip idle: 64 rows of 16 heads at position 4000 take 245 us, the two
    products 105; 512 rows at 3500 238 and 250; 300 rows from 0 41 and 93.  The products cost about 80 us of
    launches a segment and 4.8 us per million pairs times keys."""
    start, _, kv_len = seg.host
    blocks = keys = products = 0
    for a, b, kv in zip(start[:-1], start[1:], kv_len):
        if b - a >= min_rows:
            blocks += ((b - a) * heads + 127) // 128
            keys = max(keys, kv)
            products += 80 + 4.8e-6 * (b - a) * heads * kv
    return 20 + 0.06 * keys * ((blocks + 255) // 256) <= products


def latent_rows_pay(qa, cache, seg: Segments, rank: int, dtype, min_rows: int) -> bool:
    """Whether a prompt's step stays with the rows' kernel (:func:`latent_attention`, csrc/mixers/latent_decode.hip) although it has
    segments of ``min_rows`` rows or more.  That kernel takes about 11 us, 0.065 a row and 0.2 a thousand pairs of row and key, the
    tiles' kernel 28 and 0.05 a key of the longest segment (from some 600 on the products are the faster ones).  us, 16 heads, rows and
    tiles: 32 rows 17 29, 128 18 35, 300 40 43, 400 52 48, 600 81 59, four of 40 19 31, of 100 36 34, of 200 68 42, 64 behind
    600 keys 31 60, behind 2000 49 62.  A step with shorter segments as well saves their launch beside it."""
    if qa.shape[0] > 16 or not latent_prefill_ok(qa, cache, rank, dtype):
        return False
    start, pos0, kv_len = seg.host
    rows = [b - a for a, b in zip(start[:-1], start[1:])]
    pairs = sum(n * (p + 1 + kv) / 2 for n, p, kv in zip(rows, pos0, kv_len))
    keys = max((kv for n, kv in zip(rows, kv_len) if n >= min_rows), default=0)
    return 11 + 0.065 * sum(rows) + 2e-4 * pairs <= 28 + 0.05 * min(keys, 600)


def latent_attention_products(out, qa, qr, cache, seg: Segments, scale: float, rank: int,
                              min_rows: int, dtype, sink: Optional[torch.Tensor] = None):
    """Segments of ``min_rows`` rows or more, in one kernel (csrc/mixers/latent_prefill.hip: bf16, ranks of 512 + 64, dense
    operands, where :func:`_latent_prefill_pays`) or as two matrix products: all heads share
    the cached rows, so with M = heads x rows the scores are Q [M, rank+dr] C^T and the
    sums P [M, keys] C[:, :rank], with a causal softmax (fp32 statistics) in between.
    Needs the segments' host copies; writes its rows of ``out`` [heads, T, rank]."""
    start, pos0, kv_len = seg.host
    heads = qa.shape[0]
    bs = cache.shape[1]
    width = cache.shape[2]
    if latent_prefill_ok(qa, cache, rank, dtype) and _latent_prefill_pays(seg, heads, min_rows) \
            and qa.dtype == qr.dtype == out.dtype == torch.float32 \
            and _plain16(out, qa, qr, cache) and _device_segments(seg):
        ns = [n for n in (b - a for a, b in zip(start[:-1], start[1:])) if n >= min_rows]
        native_mixers().latent_prefill(out, qa, qr, cache, seg.start, seg.pos0, seg.kv_len, seg.block_tables, seg.num,
                                       len(ns), sum(ns), float(scale), rank, min_rows, sink)
        return out
    for s in range(seg.num):
        a, b = start[s], start[s + 1]
        n = b - a
        if n < min_rows:
            continue
        nblk = (kv_len[s] + bs - 1) // bs
        kv = cache.index_select(0, seg.block_tables[s, :nblk].long()).view(nblk * bs, width)
        step = max(1, min(n, PRODUCT_SCORE_BYTES // (4 * heads * max(1, kv_len[s]))))
        for c0 in range(0, n, step):
            c1 = min(n, c0 + step)
            keys = min(kv_len[s], pos0[s] + c1)          # the chunk's last row sees this many
            q = torch.cat([qa[:, a + c0:a + c1], qr[a + c0:a + c1].transpose(0, 1)], -1) \
                .reshape(heads * (c1 - c0), width).to(dtype)
            sc = mm_f32(q, kv[:keys].t())
            p = causal_softmax(sc, c1 - c0, pos0[s] + c0, scale, dtype, sink)
            out[:, a + c0:a + c1] = mm_f32(p, kv[:keys, :rank]).view(heads, c1 - c0, rank)
    return out


# ---------------------------------------------------------------------------------
# selective state-space scan (recurrent state slots)
# ---------------------------------------------------------------------------------

def ssd_scan(xbc, dt, a_log, dt_bias, d_skip, state, seg: Segments, heads: int, groups: int, n: int,
             dv: int) -> torch.Tensor:
    """State-space recurrence with one scalar decay per head and row.

    Rows of ``xbc`` are [x (heads*dv) | B (groups*n) | C (groups*n)] after the short
    convolution; ``dt`` [T, heads] is the raw step projection (may be a column range).
    step = softplus(dt + dt_bias), decay = exp(-exp(a_log) * step); per head (group
    floor(h / (heads / groups))) and row:  S <- decay S + step B x^T (S is n x dv);
    y = S^T C + d_skip x.  ``state`` [slots, heads, n, dv] fp32 is read (zeros at
    position 0) and left at the segment's last row.  Returns y fp32 [T, heads*dv]."""
    if xbc.is_cuda:
        y = torch.empty(xbc.shape[0], heads * dv, dtype=torch.float32, device=xbc.device)
        if native_mixers().state_scan_takes(y, xbc, heads, groups, n, dv, seg.max_rows):
            chunk = SCAN_ROWS
        else:
            chunk = SSD_CHUNK_ROWS if _ssd_chunks_pay(seg, heads, n, dv) else NO_CHUNKS
        native_mixers().ssd_scan(y, xbc, dt, a_log, dt_bias, d_skip, state, seg.start, seg.pos0, seg.slot,
                                 seg.num, seg.max_rows, heads, groups, n, dv, _walk_below(seg, chunk), chunk)
        return y
    return ref.ssd_scan(xbc, dt, a_log, dt_bias, d_skip, state, seg, heads, groups, n, dv)


def gate_group_norm(y, z, w, eps: float, groups: int, out_dtype):
    """v = y * silu(z); each of ``groups`` equal parts of a row divided by its own root
    mean square; times w.  y fp32 [T, n], z [T, n] (may be a column range)."""
    if y.is_cuda:
        out = torch.empty(y.shape, dtype=out_dtype, device=y.device)
        native_mixers().gate_group_norm(out, y, z, w, eps, groups)
        return out
    return ref.gate_group_norm(y, z, w, eps, groups, out_dtype)


# ---------------------------------------------------------------------------------
# windowed attention (paged key cache + paged value cache)
# ---------------------------------------------------------------------------------

def attn_prep(qkv, nq: int, nk: int, q_norm_w, k_norm_w, eps: float, table, rot_dims: int,
              head_dim: int, positions, slot_mapping, k_cache, v_cache) -> torch.Tensor:
    """Rows [q (nq) | k (nk) | v] of a fused projection -> fp32 queries [T, nq]; keys and
    values go to the rows' cache slots.  Optional steps, in this order: RMS norm of the
    whole q part and of the whole k part with weights ``q_norm_w`` / ``k_norm_w``; rotary
    positions on the first ``rot_dims`` entries of every ``head_dim`` chunk of q and k
    (entry i paired with i + rot_dims/2, ``table`` = :func:`rope_table`).  Without caches
    (``nk`` 0, rows of q alone) only the queries are prepared."""
    if qkv.is_cuda:
        q = torch.empty(qkv.shape[0], nq, dtype=torch.float32, device=qkv.device)
        native_mixers().attn_prep(q, qkv, nq, nk, q_norm_w, k_norm_w, eps, table, rot_dims, head_dim,
                                  positions, slot_mapping, k_cache, v_cache)
        return q
    return ref.attn_prep(qkv, nq, nk, q_norm_w, k_norm_w, eps, table, rot_dims, head_dim, positions,
                         slot_mapping, k_cache, v_cache)


def conv_attn_prep(qkv, nq: int, nk: int, conv_w, conv_state, seg: Segments, q_norm_w, k_norm_w, eps: float,
                   head_dim: int, slot_mapping, k_cache, v_cache, table=None, rot_dims: int = 0,
                   interleaved: bool = False) -> torch.Tensor:
    """Rows [q (nq) | k (nk) | v] of a fused projection pass a per-channel causal
    convolution over time (``conv_w`` [C, taps] fp32, last column = the current row, no
    bias, no activation; ``conv_state`` [slots, taps-1, C] fp32 holds each sequence's last
    projected rows and is updated; a segment at position 0 starts from zeros), then every
    ``head_dim`` chunk of q and of k is divided by its root mean square and multiplied by
    ``q_norm_w`` / ``k_norm_w`` ([head_dim], shared by the heads; None: no norm), then rotated
    by position on its first ``rot_dims`` entries (``table`` = :func:`rope_table`; pairs
    (i, i + rot_dims/2), or (2i, 2i + 1) if ``interleaved``; None: no rotation).
    Convolution, norm and rotation are fp32.  Returns fp32 queries [T, nq]; keys and values go to
    the rows' cache slots."""
    if qkv.is_cuda:
        q = torch.empty(qkv.shape[0], nq, dtype=torch.float32, device=qkv.device)
        native_mixers().conv_attn_prep(q, qkv, nq, nk, conv_w, conv_state, seg.start, seg.pos0, seg.slot, seg.num,
                                       seg.max_rows, q_norm_w, k_norm_w, eps, head_dim, slot_mapping, k_cache, v_cache,
                                       table, rot_dims, bool(interleaved))
        return q
    return ref.conv_attn_prep(qkv, nq, nk, conv_w, conv_state, seg, q_norm_w, k_norm_w, eps, head_dim,
                              slot_mapping, k_cache, v_cache, table, rot_dims, interleaved)


@dataclasses.dataclass
class WindowSpec:
    """A windowed attention's constants.  Query head a = h * maps + m (head h, score map
    m) reads key head floor(h / (heads / kv_heads)) * maps + m and value head
    floor(h / (heads / kv_heads)).  Position i sees j iff 0 <= i - j < window (window 0:
    every earlier key); with ``blocks`` the window is a block instead, j <= i and
    floor(i / window) = floor(j / window), blocks counted from position 0; with
    ``keep_first`` f > 0 the positions j < f stay visible whatever the window.
    s = q.k * scale; with ``softcap`` c > 0, s <- c tanh(s / c);
    score = s - r1[a] ln(1 + r2[a] (i - j)) + dist_bias[min(i - j, nd - 1), a]; weight =
    softmax over the visible keys, or sigmoid(score + pb[a]) without normalisation.
    ``sink`` (softmax only; one score, or fp32 [heads * maps], one per query head): the
    softmax's denominator gains exp(sink), as if one more key with that score and no value
    were always visible."""
    heads: int
    kv_heads: int
    dk: int
    dv: int
    window: int
    scale: float
    maps: int = 1
    sigmoid: bool = False
    r1: Optional[torch.Tensor] = None     # fp32 [heads * maps] (with r2)
    r2: Optional[torch.Tensor] = None
    pb: Optional[torch.Tensor] = None     # fp32 [heads * maps] (sigmoid weights only)
    softcap: float = 0.0
    sink: Union[float, torch.Tensor, None] = None
    blocks: bool = False
    keep_first: int = 0
    dist_bias: Optional[torch.Tensor] = None   # fp32 [nd, heads * maps], :func:`distance_bias_table`


def _sink_args(sink):
    """(one score for all heads, scores per head), each None when not given."""
    return (None, sink) if isinstance(sink, torch.Tensor) else (sink, None)


def _plain_tiles(sp: WindowSpec, k_cache) -> bool:
    """Softmax attention over a window (or every earlier key) without distance terms, bf16 rows of
    whole 16-byte pieces, query heads that fit the tile kernel's LDS: all heads of a row share
    its key tiles there, scores on the matrix units."""
    return bool(k_cache.dtype == torch.bfloat16 and not sp.sigmoid and sp.maps == 1 and not sp.blocks and sp.r1 is None
                and sp.dist_bias is None and sp.dk % 8 == 0 and sp.dv % 8 == 0 and sp.dv <= 512
                and sp.heads <= 64 and sp.heads * sp.dk <= 4096)


def window_out_dtype(q, k_cache, v_cache, spec: WindowSpec, dtype, long: bool):
    """The type :func:`window_attention` (and, ``long``, :func:`window_attention_products`) can leave rows in that are
    wanted in ``dtype``: itself where the kernels of these sizes round on their way out, else fp32."""
    sp = spec
    if dtype != torch.bfloat16 or not q.is_cuda or k_cache.dtype != dtype:
        return torch.float32
    n = native_mixers()
    rows = _plain_tiles(sp, k_cache) or n.window_decode_fits(q, k_cache, v_cache, sp.heads, sp.maps, sp.kv_heads, sp.dk, sp.dv)
    return dtype if rows and (not long or n.band_attention_fits(sp.dk, sp.dv, k_cache.shape[1])) else torch.float32


def window_attention(q, k_cache, v_cache, seg: Segments, spec: WindowSpec, skip_from: int = 0,
                     out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """q fp32 [T, heads*maps*dk] against the paged caches; [T, heads*maps, dv], fp32 or as ``out``
    (:func:`window_out_dtype`).
    ``skip_from`` > 0: segments of that many rows or more are left to the caller
    (:func:`window_attention_products`)."""
    sp = spec
    if q.is_cuda:
        if out is None:
            out = torch.empty(q.shape[0], sp.heads * sp.maps, sp.dv, dtype=torch.float32, device=q.device)
        if _plain_tiles(sp, k_cache):
            # the tile kernel of the head-mixing attention, without a mix
            native_mixers().talk_attention(out.view(q.shape[0], -1), q, None, k_cache, v_cache, seg.start, seg.pos0,
                                           seg.kv_len, seg.block_tables, seg.num, seg.max_rows, sp.heads, sp.kv_heads,
                                           sp.dk, sp.dv, sp.window, sp.keep_first, float(sp.softcap), None, skip_from,
                                           seg.max_kv, float(sp.scale), *_sink_args(sp.sink))
            return out
        native_mixers().window_attention(out, q, k_cache, v_cache, seg.start, seg.pos0, seg.kv_len,
                                         seg.block_tables, seg.num, seg.max_rows, sp.heads, sp.maps,
                                         sp.kv_heads, sp.dk, sp.dv, sp.window, sp.scale, sp.sigmoid,
                                         sp.r1, sp.r2, sp.pb, skip_from, float(sp.softcap), *_sink_args(sp.sink),
                                         bool(sp.blocks), int(sp.keep_first), sp.dist_bias)
        return out
    r = ref.window_attention(q, k_cache, v_cache, seg, sp.heads, sp.maps, sp.kv_heads, sp.dk, sp.dv,
                             sp.window, sp.scale, sp.sigmoid, sp.r1, sp.r2, sp.pb, sp.softcap, sp.sink,
                             sp.blocks, sp.keep_first, sp.dist_bias)
    if out is not None:
        out.copy_(r)
        return out
    return r


def band_weights(s, first_pos: int, key0: int, spec: WindowSpec, rep_rows: int, ext: int = 0):
    """Raw dot products fp32 [kv_heads*maps, rep*rows, keys] (the query heads that share
    a key head stacked along the rows, ``rep_rows`` = rows of one of them) -> attention
    weights fp32, in place: row r of a head is position first_pos + r; the first ``ext``
    columns are the positions 0 .. ext-1 (kept first tokens in front of the band), column
    c >= ext is position key0 + c - ext."""
    sp = spec
    if s.is_cuda:
        native_mixers().band_weights(s, rep_rows, first_pos, key0, sp.heads, sp.maps, sp.kv_heads,
                                     sp.window, sp.scale, sp.sigmoid, sp.r1, sp.r2, sp.pb, float(sp.softcap),
                                     *_sink_args(sp.sink), bool(sp.blocks), int(sp.keep_first), int(ext), sp.dist_bias)
        return s
    g, rr, keys = s.shape
    rep = sp.heads // sp.kv_heads
    # [G, maps, rep, rows, keys] -> query-head order (g, r, m)
    v = s.view(sp.kv_heads, sp.maps, rep, rep_rows, keys).permute(0, 2, 1, 3, 4) \
        .reshape(sp.heads * sp.maps, rep_rows, keys)
    w = ref.band_weights(v, first_pos, key0, sp.window, sp.scale, sp.sigmoid, sp.r1, sp.r2, sp.pb, sp.softcap,
                         sp.sink, sp.blocks, sp.keep_first, ext, sp.dist_bias)
    s.copy_(w.view(sp.kv_heads, rep, sp.maps, rep_rows, keys).permute(0, 2, 1, 3, 4).reshape(g, rr, keys))
    return s


def band_attention_ok(out, q, k_cache, v_cache, seg: Segments, spec: WindowSpec) -> bool:
    """Whether long segments run in one kernel (csrc/mixers/band_attn.hip) instead of banded products: bf16 caches of
    heads that fit its tiles, all operands dense and aligned."""
    return bool(q.is_cuda and k_cache.dtype == v_cache.dtype == torch.bfloat16 and q.dtype == torch.float32 and q.dim() == 2
                and out.dtype in (torch.float32, torch.bfloat16) and _plain16(out, q, k_cache, v_cache)
                and _device_segments(seg)
                and native_mixers().band_attention_fits(spec.dk, spec.dv, k_cache.shape[1]))


def _band_pays(seg: Segments, sp: WindowSpec, min_rows: int) -> bool:
    """A workgroup of the one kernel owns 64 (row, query head) pairs and walks their keys, so a few rows behind a long
    context leave the chip idle, where the products' widened copies and library kernels fill it: 64 rows of 16 heads of
    128 on 4 key heads at position 8000 take 174 us and the products 144, at 30000 609 and 566; 32 at 2000 54 and 122, 300
    at 4000 101 and 245, 2000 from 0 72 and 510.  A key costs the longest walk 20 ns (26 with a table or sigmoids, 31 with a cap;
    38 with distance terms in a softmax, 48 to 79 with terms that only the general form of the kernel has), a CU one walk at
    a time; the products, whose 25 launches take 100 us to issue, the reads of the cache and the pairs' sums, by an estimate
    that is up to a fifth above them near the line."""
    start, _, kv_len = seg.host
    wide, rep = (sp.dk + sp.dv) / 256, sp.heads // sp.kv_heads
    cap, table, terms = sp.softcap > 0, sp.dist_bias is not None, sp.r1 is not None
    if (cap or table) if sp.sigmoid else (terms or (cap and table)):
        kind = 26 + 13 * cap + 19 * table + 9 * bool(sp.sigmoid)
    else:
        kind = (20 if terms else 14) if sp.sigmoid else 14 if table else 19 if cap else 8
    a = 4 + 4 * sp.kv_heads * (sp.maps * sp.dk + sp.dv) / 1024
    b = sp.heads * sp.maps * (0.0053 + 0.0049 * wide)
    longest = total = products = 0.0
    for n, kv in zip((y - x for x, y in zip(start[:-1], start[1:])), kv_len):
        if n < min_rows:
            continue
        keys = kv if sp.window <= 0 else min(kv, sp.window + (0 if sp.blocks else n))
        longest = max(longest, keys)
        total += keys * sp.kv_heads * sp.maps * (-(-n * rep // 64))
        products += max(100.0, 20 + 1e-3 * keys * (a + b * n) * (0.8 if sp.sigmoid else 1.0))
    return 10 + 1e-3 * (kind + 12 * wide) * max(longest, total / 256) <= 0.92 * products


def _band_groups(seg: Segments, sp: WindowSpec, min_rows: int) -> int:
    """Groups of waves in a workgroup of the one kernel.  Two walk a block's tiles of 64 keys in turn, 1.3 us a tile where one
    takes 1.7 to 2; but one leaves room for a second workgroup on the CU, which hides its own start and end (8 and 11 us) and
    gets 1.35 us a tile out of the CU where two groups get 1.5.  So two where the longest walk is what counts: us with one / two,
    16 heads of 128 on 4 key heads: 300 rows 15.7 16.5, 600 23.5 22.1, 777 30 28, 1000 37 33, 2048 74 70, 4096 206 216, 8192 699
    772; 64 at 2000 64 52, at 30000 822 608; 1500 at 3000 160 169; 16 of 100 16 25, five of 258 to 542 30 35; 2048 in a window
    of 512 35 45, of two maps 96 107."""
    start, _, kv_len = seg.host
    rep, heads = sp.heads // sp.kv_heads, sp.kv_heads * sp.maps
    longest = tiles = groups = 0.0
    for n, kv in zip((y - x for x, y in zip(start[:-1], start[1:])), kv_len):
        if n < min_rows:
            continue
        top, mean, blocks = kv, kv - n / 2, -(-n * rep // 64) * heads
        if sp.window > 0:
            top, mean = min(top, sp.window), min(mean, sp.window / 2 if sp.blocks and kv > sp.window else sp.window)
        longest = max(longest, top / 64)
        tiles += blocks * max(1.0, mean / 64)
        groups += blocks
    return 2 if longest > 5 and tiles / 256 + 4 * max(0.0, groups / 256 - 1) < 1.2 * longest else 1


def window_attention_products(out, q, k_cache, v_cache, seg: Segments, spec: WindowSpec, min_rows: int):
    """Segments of ``min_rows`` rows or more as banded matrix products: a chunk of rows
    [c0, c1) only sees the keys c0 - window + 1 .. c1 - 1 (or from the start of c0's block;
    plus the kept first positions, gathered in front of the band), so per chunk and key head the
    scores are one product with M = (query heads of the group) x rows, the weights come
    from :func:`band_weights` (fp32) and the sums are a second product with the value
    head.  Operands are fp32 (cached rows are widened), so scores, weights and sums are
    true fp32.  bf16 caches whose heads fit its tiles run in one kernel for all segments instead
    (:func:`band_attention_ok`), to the same exactness, unless a few rows see a long context
    (:func:`_band_pays`).  Needs the segments' host copies; writes its rows of ``out``."""
    sp = spec
    start, pos0, kv_len = seg.host
    bs = k_cache.shape[1]
    if band_attention_ok(out, q, k_cache, v_cache, seg, sp) and _band_pays(seg, sp, min_rows):
        # one kernel for all segments, scores never in memory
        ns = [n for n in (b - a for a, b in zip(start[:-1], start[1:])) if n >= min_rows]
        native_mixers().band_attention(out, q, k_cache, v_cache, seg.start, seg.pos0, seg.kv_len, seg.block_tables,
                                       seg.num, len(ns), sum(ns), sp.heads, sp.maps, sp.kv_heads, sp.dk, sp.dv,
                                       sp.window, float(sp.scale), bool(sp.sigmoid), sp.r1, sp.r2, sp.pb, min_rows,
                                       float(sp.softcap), *_sink_args(sp.sink), bool(sp.blocks), int(sp.keep_first),
                                       sp.dist_bias, _band_groups(seg, sp, min_rows))
        return out
    rep = sp.heads // sp.kv_heads
    gk = sp.kv_heads * sp.maps
    for s in range(seg.num):
        a, b = start[s], start[s + 1]
        n = b - a
        if n < min_rows:
            continue
        # without a window a chunk sees every earlier key anyway: long chunks, few launches
        step = PRODUCT_FULL_CHUNK_ROWS if sp.window <= 0 else max(PRODUCT_CHUNK_ROWS, min(sp.window, 1024))
        # the fp32 scores of a chunk ([heads*maps, rows, keys]) stay under PRODUCT_SCORE_BYTES
        span = sp.window if sp.window > 0 else kv_len[s]
        while step > 32 and 4 * sp.heads * sp.maps * step * (step + span) > PRODUCT_SCORE_BYTES:
            step //= 2
        for c0 in range(0, n, step):
            c1 = min(n, c0 + step)
            rows = c1 - c0
            i0 = pos0[s] + c0
            lo = ref.mask_first_key(i0, sp.window, sp.blocks)
            ext = min(sp.keep_first, lo) if sp.window > 0 else 0
            hi = min(kv_len[s], pos0[s] + c1)
            b0, b1 = lo // bs, (hi + bs - 1) // bs
            blocks = seg.block_tables[s, b0:b1].long()
            off = lo - b0 * bs
            k = k_cache.index_select(0, blocks).view((b1 - b0) * bs, gk, sp.dk)[off:off + hi - lo].float()
            v = v_cache.index_select(0, blocks).view((b1 - b0) * bs, sp.kv_heads, sp.dv)[off:off + hi - lo].float()
            if ext:
                # the kept first positions 0 .. ext-1 lie before the band: their rows go in front
                eb = seg.block_tables[s, :(ext + bs - 1) // bs].long()
                k = torch.cat([k_cache.index_select(0, eb).view(-1, gk, sp.dk)[:ext].float(), k], 0)
                v = torch.cat([v_cache.index_select(0, eb).view(-1, sp.kv_heads, sp.dv)[:ext].float(), v], 0)
            # q rows [rows, (g, r, m), dk] -> [(g, m), (r, rows), dk]
            qc = q[a + c0:a + c1].view(rows, sp.kv_heads, rep, sp.maps, sp.dk).permute(1, 3, 2, 0, 4) \
                .reshape(gk, rep * rows, sp.dk)
            sc = torch.bmm(qc, k.permute(1, 2, 0))                       # [gk, rep*rows, keys]
            band_weights(sc, i0, lo, sp, rows, ext)
            # both maps of a group read the same value head: [G, maps*rep*rows, keys] x [G, keys, dv]
            o = torch.bmm(sc.view(sp.kv_heads, sp.maps * rep * rows, ext + hi - lo), v.transpose(0, 1))
            out[a + c0:a + c1] = o.view(sp.kv_heads, sp.maps, rep, rows, sp.dv).permute(3, 0, 2, 1, 4) \
                .reshape(rows, sp.heads * sp.maps, sp.dv)
    return out


# rows of a segment that one pair of banded products covers (at least; a window wider
# than this takes a chunk of its own width, up to 1024 rows)
PRODUCT_CHUNK_ROWS = 256
# rows per chunk when every earlier key is visible (halved until the chunk's scores fit
# PRODUCT_SCORE_BYTES)
PRODUCT_FULL_CHUNK_ROWS = 2048


def diff_combine(a, gate, lam: float, post_scale: float, eps: float, heads: int, dv: int, out_dtype):
    """Two score maps per head -> one output: o = a[:, 2h] - lam * a[:, 2h+1], divided by
    its root mean square over dv, times post_scale * sigmoid(gate[:, h]).  a fp32
    [T, heads*2, dv]; gate [T, heads] (may be a column range); [T, heads*dv]."""
    if a.is_cuda:
        out = torch.empty(a.shape[0], heads * dv, dtype=out_dtype, device=a.device)
        native_mixers().diff_combine(out, a, gate, float(lam), float(post_scale), eps, heads, dv)
        return out
    return ref.diff_combine(a, gate, lam, post_scale, eps, heads, dv, out_dtype)


# ---------------------------------------------------------------------------------
# attention whose scores are mixed across the heads (paged key cache + paged value cache)
# ---------------------------------------------------------------------------------

@dataclasses.dataclass
class TalkSpec:
    """Constants of an attention that mixes scores across its heads before the softmax.
    Query head h reads key and value head floor(h / (heads / kv_heads)).  Position i sees
    j iff 0 <= i - j < window (window 0: every earlier key) or j < keep_first (<= i).
    With dot products s_g = q_g.k (queries come scaled): s_g <- softcap tanh(s_g /
    softcap) (softcap 0: as they are), z_h = sum_g talk[h, g] s_g, weights = softmax of
    z_h over the visible keys."""
    heads: int
    kv_heads: int
    dk: int
    dv: int
    window: int
    keep_first: int
    softcap: float
    talk: torch.Tensor          # fp32 [heads, heads]


def rot_norm_prep(qk, nq: int, nk: int, head_dim: int, table, rot_dims: int, eps: float, q_scale, positions,
                  slot_mapping, k_cache, v_cache, interleaved: bool = False) -> torch.Tensor:
    """Rows [q (nq) | k (nk) | ...] of a fused projection, head by head (``head_dim``
    entries): rotary positions on the first ``rot_dims`` entries (``table`` =
    :func:`rope_table`; None: no rotation), then the head divided by its root mean square.
    Queries are also multiplied by ``q_scale`` fp32 [q heads] and returned in fp32 [T,
    nq]; keys go to the rows' key-cache slots, and the k rows as projected (neither rotated
    nor normed) to the value-cache slots."""
    if qk.is_cuda:
        q = torch.empty(qk.shape[0], nq, dtype=torch.float32, device=qk.device)
        native_mixers().rot_norm_prep(q, qk, nq, nk, head_dim, table, rot_dims, bool(interleaved), eps, q_scale,
                                      positions, slot_mapping, k_cache, v_cache)
        return q
    return ref.rot_norm_prep(qk, nq, nk, head_dim, table, rot_dims, interleaved, eps, q_scale, positions,
                             slot_mapping, k_cache, v_cache)


def talk_attention(out, q, gate, k_cache, v_cache, seg: Segments, spec: TalkSpec, skip_from: int = 0):
    """q fp32 [T, heads*dk] against the paged caches; writes ``out`` [T, heads*dv] (the
    weighted sums, times sigmoid(gate) element by element when ``gate`` [T, heads*dv] is
    given).  ``skip_from`` > 0: segments of that many rows or more are left to the caller
    (:func:`talk_attention_products`)."""
    sp = spec
    if q.is_cuda:
        native_mixers().talk_attention(out, q, gate, k_cache, v_cache, seg.start, seg.pos0, seg.kv_len,
                                       seg.block_tables, seg.num, seg.max_rows, sp.heads, sp.kv_heads, sp.dk, sp.dv,
                                       sp.window, sp.keep_first, float(sp.softcap), sp.talk, skip_from, seg.max_kv,
                                       1.0, None, None)
        return out
    r = ref.talk_attention(q, k_cache, v_cache, seg, sp.heads, sp.kv_heads, sp.dk, sp.dv, sp.window, sp.keep_first,
                           sp.softcap, sp.talk)
    out.copy_(r if gate is None else ref.sigmoid_gate(r, gate, out.dtype))
    return out


# Segments of a prompt whose (row, key) pairs are no more, or whose band is no wider, stay with the rows' kernel, which reads the
# caches in place, all segments in one launch; the products gather the keys, write all scores and take a dozen launches a
# segment.  us, 16 heads of 128 on 4 key heads, kernel / products: 64 rows 20 64, 300 44 70, 600 90 118, 1024 175 175, four of 200
# 67 293, 400 behind 1500 keys 135 187; a window of 1024 and 64 kept, 1000 behind 1500 keys 268 328, 4096 rows 891 1114; no
# window, 300 behind 3000 (0.95 M pairs) 346 291, 700 behind 1500 (1.3 M) 364 298.  Only forms of the kernel whose waves' heads share a
# value head (talk_attn.hip, AHEAD) of up to 16 heads: 16 heads on 16, 1100 rows 854 320; 32 on 8, 400 behind 1500 335 297.
TALK_ROWS_PAIRS = 768 << 10
TALK_ROWS_BAND = 1152


def talk_product_rows(seg: Segments, spec: TalkSpec, k_cache, least: int) -> int:
    """The rows (``least`` or more) from which a step's segments are left to :func:`talk_attention_products`; the others are
    :func:`talk_attention`'s.  Needs the segments' host copies."""
    sp = spec
    per = 1
    while 4 * per < sp.heads:                      # heads of a wave
        per *= 2
    if not k_cache.is_cuda or k_cache.dtype != torch.bfloat16 or sp.heads > 16 or (sp.heads // sp.kv_heads) % per or \
            sp.dk % 8 or sp.dv % 8 or max(sp.dk, sp.dv) > 128:
        return least
    none = 1 << 30
    band = sp.window + sp.keep_first if sp.window > 0 else none
    if band <= TALK_ROWS_BAND:
        return none
    start, pos0, kv_len = seg.host
    rows = [b - a for a, b in zip(start[:-1], start[1:])]
    return min([n for n, p, kv in zip(rows, pos0, kv_len) if n >= least and n * min(band, (p + 1 + kv) // 2) > TALK_ROWS_PAIRS],
               default=none)


def talk_weights(s, first_pos: int, key0: int, ext: int, spec: TalkSpec):
    """Dot products fp32 [heads, rows, keys] -> unnormalised weights exp(z - max) in place
    (zeros where a key is not visible) and the reciprocals of their row sums, fp32 [heads,
    rows]; row r is position first_pos + r, the first ``ext`` columns are the positions
    0 .. ext-1 and column c >= ext is position key0 + c - ext."""
    sp = spec
    if s.is_cuda:
        inv = torch.empty(s.shape[:2], dtype=torch.float32, device=s.device)
        native_mixers().talk_weights(s, inv, first_pos, key0, ext, sp.window, sp.keep_first, float(sp.softcap),
                                     sp.talk)
        return inv
    s.copy_(ref.talk_weights(s, s.shape[1], first_pos, key0, ext, sp.window, sp.keep_first, sp.softcap, sp.talk))
    return torch.ones(s.shape[:2], dtype=torch.float32, device=s.device)


def scaled_heads_gate(out, o, inv, gate):
    """out rows [T, heads*dv] = o [heads, T, dv] * inv [heads, T] (* sigmoid(gate [T, heads*dv]))."""
    if o.is_cuda:
        native_mixers().scaled_heads_gate(out, o, inv, gate)
        return out
    heads, t, dv = o.shape
    r = (o * inv[:, :, None]).transpose(0, 1).reshape(t, heads * dv)
    out.copy_(r if gate is None else ref.sigmoid_gate(r, gate, out.dtype))
    return out


def talk_attention_products(out, q, gate, k_cache, v_cache, seg: Segments, spec: TalkSpec, min_rows: int):
    """Segments of ``min_rows`` rows or more as banded matrix products in fp32 (see
    :func:`window_attention_products`), with :func:`talk_weights` between the two and the
    normalisation and gate in the step that puts the heads back into rows.  Needs the
    segments' host copies; writes its rows of ``out``."""
    sp = spec
    start, pos0, kv_len = seg.host
    bs = k_cache.shape[1]
    rep = sp.heads // sp.kv_heads
    for s in range(seg.num):
        a, b = start[s], start[s + 1]
        n = b - a
        if n < min_rows:
            continue
        step = PRODUCT_FULL_CHUNK_ROWS if sp.window <= 0 else max(PRODUCT_CHUNK_ROWS, min(sp.window, 1024))
        span = sp.window + sp.keep_first if sp.window > 0 else kv_len[s]
        while step > 32 and 4 * sp.heads * step * (step + span) > PRODUCT_SCORE_BYTES:
            step //= 2
        for c0 in range(0, n, step):
            c1 = min(n, c0 + step)
            rows = c1 - c0
            i0 = pos0[s] + c0
            lo = ref.mask_first_key(i0, sp.window, False)
            ext = min(sp.keep_first, lo) if sp.window > 0 else 0
            hi = min(kv_len[s], pos0[s] + c1)
            k = _band_rows(k_cache, seg.block_tables[s], lo, hi, ext, bs).view(-1, sp.kv_heads, sp.dk)
            v = _band_rows(v_cache, seg.block_tables[s], lo, hi, ext, bs).view(-1, sp.kv_heads, sp.dv)
            # q rows [rows, (g, r), dk] -> [g, (r, rows), dk]
            qc = q[a + c0:a + c1].view(rows, sp.kv_heads, rep, sp.dk).permute(1, 2, 0, 3) \
                .reshape(sp.kv_heads, rep * rows, sp.dk)
            sc = torch.bmm(qc, k.permute(1, 2, 0)).view(sp.heads, rows, -1)
            inv = talk_weights(sc, i0, lo, ext, sp)
            o = torch.bmm(sc.view(sp.kv_heads, rep * rows, -1), v.transpose(0, 1)).view(sp.heads, rows, sp.dv)
            scaled_heads_gate(out[a + c0:a + c1], o, inv, None if gate is None else gate[a + c0:a + c1])
    return out


def _band_rows(cache, table, lo: int, hi: int, ext: int, bs: int):
    """Cached rows (fp32) of positions 0 .. ext-1 followed by lo .. hi-1."""
    b0, b1 = lo // bs, (hi + bs - 1) // bs
    r = cache.index_select(0, table[b0:b1].long()).view((b1 - b0) * bs, -1)[lo - b0 * bs:hi - b0 * bs].float()
    if ext:
        e = cache.index_select(0, table[:(ext + bs - 1) // bs].long()).view(-1, r.shape[1])[:ext].float()
        r = torch.cat([e, r], 0)
    return r


# ---------------------------------------------------------------------------------
# mixture of experts
# ---------------------------------------------------------------------------------

def moe_topk(z, correction, top: int, groups: int, keep: int):
    """Router: s = softmax(z) (fp32); choice = s + correction; experts outside the
    ``keep`` best of ``groups`` equal groups (by their best choice score) are excluded;
    the ``top`` best choices are returned with their s as weights (not renormalised)."""
    if z.is_cuda:
        t = z.shape[0]
        idx = torch.empty(t, top, dtype=torch.int32, device=z.device)
        wts = torch.empty(t, top, dtype=torch.float32, device=z.device)
        native_mixers().moe_topk(idx, wts, z, correction, top, groups, keep)
        return idx, wts
    return ref.moe_topk(z, correction, top, groups, keep)


def moe_top_logits(z, top: int):
    """Router: the ``top`` largest logits of each fp32 row (ties to the lower index) and,
    as weights, the softmax over just those."""
    if z.is_cuda:
        t = z.shape[0]
        idx = torch.empty(t, top, dtype=torch.int32, device=z.device)
        wts = torch.empty(t, top, dtype=torch.float32, device=z.device)
        native_mixers().moe_top_logits(idx, wts, z, top, False, 1.0, 1, 1)
        return idx, wts
    return ref.moe_top_logits(z, top)


def moe_top_sigmoid(z, top: int, scale: float, groups: int = 1, keep: int = 1):
    """Router: the ``top`` largest logits of each fp32 row (ties to the lower index); the
    weights are the chosen ones' sigmoids divided by the sum of those, times ``scale``.
    With ``keep`` < ``groups`` only experts of the ``keep`` best of ``groups`` equal groups of
    neighbours can be chosen; a group's score is the sum of its two largest sigmoids."""
    if z.is_cuda:
        t = z.shape[0]
        idx = torch.empty(t, top, dtype=torch.int32, device=z.device)
        wts = torch.empty(t, top, dtype=torch.float32, device=z.device)
        native_mixers().moe_top_logits(idx, wts, z, top, True, float(scale), groups, keep)
        return idx, wts
    return ref.moe_top_sigmoid(z, top, scale, groups, keep)


def moe_route_top_logits(h, router, bias, top: int, sigmoid: bool = False, scale: float = 1.0, groups: int = 1,
                         keep: int = 1):
    """:func:`moe_top_logits` (or, ``sigmoid``, :func:`moe_top_sigmoid` with ``scale`` and
    groups) of z = router h + bias (fp32 router [E, width] and bias, h fp32 or bf16, fp32
    accumulation) in one launch: the router of few rows (decode steps)."""
    if h.is_cuda:
        t = h.shape[0]
        idx = torch.empty(t, top, dtype=torch.int32, device=h.device)
        wts = torch.empty(t, top, dtype=torch.float32, device=h.device)
        native_mixers().moe_route_top_logits(idx, wts, h, router, bias, top, bool(sigmoid), float(scale), groups, keep)
        return idx, wts
    z = torch.nn.functional.linear(h.float(), router, bias)
    return ref.moe_top_sigmoid(z, top, scale, groups, keep) if sigmoid else ref.moe_top_logits(z, top)


def moe_route_softmax(h, router, correction, top: int, groups: int, keep: int):
    """:func:`moe_topk` of z = router h (fp32 router [E, width], h fp32 or bf16, fp32 accumulation) in one launch: the
    router of few rows (decode steps)."""
    if h.is_cuda:
        idx = torch.empty(h.shape[0], top, dtype=torch.int32, device=h.device)
        wts = torch.empty(h.shape[0], top, dtype=torch.float32, device=h.device)
        native_mixers().moe_route_softmax(idx, wts, h, router, correction, top, groups, keep)
        return idx, wts
    return ref.moe_topk(torch.nn.functional.linear(h.float(), router), correction, top, groups, keep)


def moe_route_softmax_pays(experts: int) -> bool:
    """Where :func:`moe_route_softmax`, a workgroup per row that takes the experts sixteen at a time, beats a library
    product and :func:`moe_topk`: 32 experts 9 us (17 for 64 rows of 2048), 64 10 (18), 128 25 (20)."""
    return experts <= 64


ROUTE_MODES = {"top_logits": 0, "top_sigmoid": 1, "grouped_softmax": 2}


# Rows up to which a workgroup a row routes (csrc/mixers/moe_route.hip route_rows_kernel; beyond, a workgroup for sixteen with
# the router on the matrix units), alone and with the norm step in front: two such workgroups fit a CU, and one.  us, 32 experts
# of 2048 (64 of 2048, 8 of 4096), rows / sixteen a workgroup: 256 rows 9.2 15.4 (11 17, 6.0 9.8), 512 12.8 15.5 (17 17, 9.2
# 11.1), 777 19.8 15.7 (28 17, 15 12); with the norm 256 rows 11.3 19.1 (13 21, 8.4 14.6), 300 20.5 19.5 (23 21, 14.6 15.3).
ROUTE_ROWS = 512
NORM_ROUTE_ROWS = 256


def moe_route_by_row(h, router) -> bool:
    """Whether a workgroup a row is the faster router (:func:`moe_route_top_logits`, :func:`moe_route_softmax`)."""
    return bool(h.is_cuda and h.shape[0] <= ROUTE_ROWS and h.dtype == torch.bfloat16 and h.stride(1) == 1 and h.stride(0) % 4 == 0
                and h.data_ptr() % 8 == 0 and router.data_ptr() % 16 == 0
                and native_mixers().norm_route_fits(h.shape[1], router.shape[0]))


def norm_route_fits(x, y, wb, w, b, router) -> bool:
    """Whether :func:`norm_route` takes these rows: up to NORM_ROUTE_ROWS bf16 or fp32 sublayer outputs y on a GPU, at most 64
    experts (a lane each), widths of whole 256 up to 8192 (a row in LDS), all at 16-byte addresses; or a product's two or four parts."""
    if isinstance(y, ExpertParts):
        return bool(y.wts is None and y.shared is None and x.shape[0] <= NORM_ROUTE_ROWS and x.is_contiguous()
                    and y.d.shape[0] in (2 * x.shape[0], 4 * x.shape[0])
                    and all(t is None or t.data_ptr() % 16 == 0 for t in (x, y.d, wb, w, b, router))
                    and native_mixers().norm_route_fits(x.shape[1], router.shape[0]))
    return bool(y.is_cuda and y.shape[0] <= NORM_ROUTE_ROWS and x.is_contiguous() and y.dim() == 2 and y.shape == x.shape
                and y.stride(1) == 1 and y.stride(0) % 4 == 0 and y.data_ptr() % (4 * y.element_size()) == 0
                and all(t is None or t.data_ptr() % 16 == 0 for t in (x, wb, w, b, router))
                and native_mixers().norm_route_fits(x.shape[1], router.shape[0]))


def norm_route(x, y, wb, w, b, eps: float, router, bias, top: int, routing: str, scale: float = 1.0, groups: int = 1,
               keep: int = 1):
    """For few rows: the norm step in front of a mixture, :func:`add_rms_norm_rows` (``wb``, ``next_w`` = w) or, with ``b``,
    :func:`add_layer_norm_rows` (w, b), and the router (the fp32 one itself; ``bias``, ``routing`` and the rest as in
    :func:`moe_route`) of the rows h that it makes, in one launch.  x fp32, in place; returns (h bf16, (idx, wts))."""
    h = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    idx = torch.empty(x.shape[0], top, dtype=torch.int32, device=x.device)
    wts = torch.empty(x.shape[0], top, dtype=torch.float32, device=x.device)
    native_mixers().norm_route(idx, wts, h, x, y.d if isinstance(y, ExpertParts) else y, b is not None, wb, w, b, eps, router, bias, top, ROUTE_MODES[routing],
                               float(scale), groups, keep)
    return h, (idx, wts)


def route_parts(router) -> Optional[torch.Tensor]:
    """fp32 router [E, width] as three bf16 parts whose sum is it (hi, mid and lo: 24 bits), in the operand order of
    :func:`moe_route`: [width / 32, tiles of 16 experts, 3, 64, 8].  None where it takes no such router
    (:func:`moe_route_fits`).  A copy: a router that is written to needs new parts."""
    e, width = router.shape
    if width % 2048 or e > 64:
        return None
    tiles = (e + 15) // 16
    w = torch.nn.functional.pad(router, (0, 0, 0, 16 * tiles - e))
    hi = w.to(torch.bfloat16)
    mid = (w - hi.float()).to(torch.bfloat16)
    parts = torch.stack([hi, mid, (w - hi.float() - mid.float()).to(torch.bfloat16)])
    # [part, tile, expert n, step, group g, 8] -> a lane (g, n) of a step's tile reads its 8
    return parts.view(3, tiles, 16, width // 32, 4, 8).permute(3, 1, 0, 4, 2, 5).reshape(width // 32, tiles, 3, 64, 8) \
        .contiguous()


def moe_route_fits(h, parts, experts: int) -> bool:
    """Whether :func:`moe_route` takes these rows: bf16 on a GPU, at most 64 experts (a lane each), widths of whole 2048
    (128 for each of a workgroup's sixteen waves; other widths have not been timed)."""
    return bool(h.is_cuda and parts is not None and native_mixers().moe_route_fits(h, parts, experts))


def moe_route(h, parts, bias, experts: int, top: int, routing: str, scale: float = 1.0, groups: int = 1, keep: int = 1):
    """The routers :func:`moe_topk` (``bias``: its correction), :func:`moe_top_logits` and :func:`moe_top_sigmoid`
    (``bias``: added to the logits, or None) of z = router h in one launch, fp32 throughout; ``parts``: the fp32
    router's :func:`route_parts`."""
    idx = torch.empty(h.shape[0], top, dtype=torch.int32, device=h.device)
    wts = torch.empty(h.shape[0], top, dtype=torch.float32, device=h.device)
    native_mixers().moe_route(idx, wts, h, parts, bias, experts, top, ROUTE_MODES[routing], float(scale), groups, keep)
    return idx, wts


# first matrix and activation of an expert: the code that the per-pair kernels take (moe_pairs.hip; FEW_ACTS of the others)
EXPERT_ACTS = {"clamp_glu": 0, "relu_sq": 1, "silu_glu": 2}


def moe_pairs(out, h, idx, wts, wgu, wdown, limit: float = 0.0, act: str = "clamp_glu"):
    """Few rows (decode): out (fp32, in place) += sum_k wts[:, k] * expert_{idx[:, k]}(h),
    every (row, expert) pair streaming its expert's first matrix ([gate | up] with the
    clamped GLU, ``act`` "clamp_glu", or with silu(gate) * up, "silu_glu"; or up alone with
    relu(.)^2, "relu_sq") and
    its down matrix; no host round trip, so the step can be captured in a hipGraph."""
    if out.is_cuda:
        native_mixers().moe_pairs(out, h, idx, wts, wgu, wdown, float(limit), EXPERT_ACTS[act])
    else:
        ref.moe_pairs(out, h, idx, wts, wgu, wdown, limit, act)


def experts_few_ok(h, wgu, wdown, shared) -> bool:
    """Whether :func:`experts_few` takes these rows and weights (``shared``: the shared expert's two
    matrices, or None)."""
    ws = [wgu, wdown] + (list(shared) if shared is not None else [])
    return bool(_few_rows(h, wgu) and all(w.dtype == torch.bfloat16 and w.shape[-1] % 8 == 0 and w.data_ptr() % 16 == 0
                                          and w.is_contiguous() for w in ws))


def experts_few_pays(pairs: int, experts: int, size: int, shared: bool) -> bool:
    """Where :func:`experts_few` beats a read of the matrices per (row, choice) pair (:func:`moe_pairs`): once enough pairs
    share an expert to make up for a launch over all experts.  us of the layer, matrices from HBM (per pair in brackets):
    32 experts, top 4, relu^2 of 1536 x 2048: 32 40 57 63 71 at 1 2 4 6 8 rows (25 31 46 61 71), 93 at 32 (214); 8 of
    4096 x 4096, top 2: 50 84 93 127 at 1 2 3 4 (40 77 97 137); 64 of 1408 x 4096, top 8: 110 151 169 185 (84 127 164 197);
    128 of 768 x 2048, top 8: 56 87 124 at 1 4 8 (45 74 124); matrices (``size`` entries) of a few hundred KB are all
    launches: 4 of 512 x 512, 14 at 1 to 24 rows (11 to 15).  A shared expert rides in the same launches: level at one
    row, 0.9 of the time from 4."""
    return shared or pairs >= max(min(0.75 * experts, 16 + 0.375 * experts), 24 if size < 1 << 20 else 0)


def experts_few(h, idx, wts, wgu, wdown, act: str, limit: float = 0.0, shared=None, shared_limit: float = 0.0,
                shared_gate: bool = False, parts: bool = False):
    """fp32 sum_k wts[:, k] * expert_{idx[:, k]}(h) (+ the shared expert, times the sigmoid of its
    last row's product if ``shared_gate``), for few rows: every chosen expert's matrices are read
    once for all rows that chose it.  No host round trip.  With ``parts``, where the norm steps take
    rows of this width so, the :class:`ExpertParts` instead of their sum."""
    parts = parts and native_mixers().expert_rows_fit(h.shape[1])
    out = None if parts else torch.empty(h.shape, dtype=torch.float32, device=h.device)
    d, ds, gate = native_mixers().experts_few(out, h, idx, wts, wgu, wdown, float(limit), FEW_ACTS[act],
                                              shared[0] if shared is not None else None,
                                              shared[1] if shared is not None else None, float(shared_limit),
                                              bool(shared_gate))
    return ExpertParts(d, wts, ds, gate) if parts else out


def experts_many_ok(h, wgu, wdown) -> bool:
    """Whether :func:`experts_many` takes these rows and expert weights."""
    return bool(h.is_cuda and all(x.dtype == torch.bfloat16 and x.is_contiguous() and x.shape[-1] % 8 == 0
                                  and x.data_ptr() % 16 == 0 for x in (h, wgu, wdown)))


def experts_many(h, idx, wts, wgu, wdown, act: str, limit: float = 0.0, shared=None, gate_w=None, parts: bool = False):
    """fp32 sum_k wts[:, k] * expert_{idx[:, k]}(h) (+ ``shared``, bf16 rows, times sigmoid(h . gate_w) if
    there is a ``gate_w``), for many rows: (row, choice) pairs sorted by expert, every expert's pairs one
    group of two grouped products.  No host round trip.  With ``parts``, where a norm step takes
    rows of this width so, :class:`SortedParts` instead of the sum."""
    pairs, width = h.shape[0] * idx.shape[1], h.shape[1]
    d = torch.empty(pairs, width, dtype=h.dtype, device=h.device)
    place = torch.empty(2 * pairs + wgu.shape[0], dtype=torch.int32, device=h.device)     # (and what the sort needs beside it)
    parts = parts and native_mixers().expert_rows_fit(width)
    out = None if parts else torch.empty(h.shape, dtype=torch.float32, device=h.device)
    native_mixers().experts_many(out, d, place, h, idx, wts, wgu, wdown, float(limit), FEW_ACTS[act], shared, gate_w)
    return SortedParts(d, place, wts, shared, h, gate_w) if parts else out


def clamp_swiglu(gu, limit: float):
    """[gate | up (| extra)] rows -> min(gate, limit) * sigmoid(1.702 gate') * (clamp(up) + 1)."""
    if gu.is_cuda:
        ff = gu.shape[1] // 2
        out = torch.empty(gu.shape[0], ff, dtype=gu.dtype, device=gu.device)
        native_mixers().clamp_swiglu(out, gu, float(limit))
        return out
    return ref.clamp_swiglu(gu, limit)


def _act_glu(gu, code: int):
    out = torch.empty(gu.shape[0], gu.shape[1] // 2, dtype=gu.dtype, device=gu.device)
    native_mixers().act_glu(out, gu, code)
    return out


def gelu_glu(gu):
    """[gate | up] rows -> gelu_tanh(gate) * up."""
    return _act_glu(gu, 0) if gu.is_cuda else ref.gelu_glu(gu)


def relu_glu(gu):
    """[gate | up] rows -> relu(gate) * up."""
    return _act_glu(gu, 1) if gu.is_cuda else ref.relu_glu(gu)


def silu_glu(gu):
    """[gate | up] rows -> silu(gate) * up."""
    return _act_glu(gu, 2) if gu.is_cuda else ref.silu_glu(gu)


def relu_sq(x):
    if x.is_cuda:
        native_mixers().relu_sq(x)
        return x
    return ref.relu_sq(x)


def relu_sq_rows(u, ff: int):
    """relu(u[:, :ff])^2 of wider rows (a column range of a fused product), dense."""
    if u.is_cuda:
        out = torch.empty(u.shape[0], ff, dtype=u.dtype, device=u.device)
        native_mixers().relu_sq_rows(out, u)
        return out
    return ref.relu_sq_rows(u, ff)


def gather_add_rows(out, y, idx, w):
    """out[r] (fp32, in place) += sum_k w[r, k] * y[idx[r, k]]; idx int32 [rows, top]."""
    if out.is_cuda:
        native_mixers().gather_add_rows(out, y, idx, w)
    else:
        ref.gather_add_rows(out, y, idx, w)


def grouped_mm_is_one_product(a, w) -> bool:
    """Whether :func:`grouped_mm` runs as one kernel without reading group sizes on the host."""
    return bool(a.is_cuda and a.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and a.shape[1] % 8 == 0)


def grouped_mm(a, w, offsets, counts=None):
    """Rows of ``a`` [M, K] sorted by group; group g's rows (up to ``offsets[g]``, the
    running sum of the group sizes, int32 on the device) times w[g]^T, w [G, N, K] ->
    [M, N] in a's dtype.  bf16 on a GPU with K a multiple of 8 is one grouped MFMA kernel
    (no host round trip); otherwise one vendor product per group (``counts``: the group
    sizes on the host, read from ``offsets`` when not given)."""
    if grouped_mm_is_one_product(a, w):
        out = torch.empty(a.shape[0], w.shape[1], dtype=a.dtype, device=a.device)
        native_mixers().grouped_gemm(out, a.contiguous(), w, offsets, 0, 0.0, -1)
        return out
    if counts is None:
        ends = offsets.tolist()
        counts = [e - s for s, e in zip([0] + ends[:-1], ends)]
    out = torch.empty(a.shape[0], w.shape[1], dtype=a.dtype, device=a.device)
    s = 0
    for g, n in enumerate(counts):
        if n:
            torch.mm(a[s:s + n], w[g].t(), out=out[s:s + n])
        s += n
    return out


def side_gate(gpre, table, ids, col0: int, sd: int):
    """gelu_tanh(gpre) * table[ids, col0:col0+sd]."""
    if gpre.is_cuda:
        out = torch.empty_like(gpre)
        native_mixers().side_gate(out, gpre, table, ids, col0)
        return out
    return ref.side_gate(gpre, table, ids, col0, sd)


def scale_add_rows(out, y, rows, weights, sigmoid: bool = False):
    """out[rows[i]] += w_i * y[i] (fp32 out; rows None = identity; w = sigmoid(weights)
    if ``sigmoid``).  ``rows`` must not repeat within one call."""
    if out.is_cuda:
        native_mixers().scale_add_rows(out, y, rows, weights, sigmoid)
    else:
        ref.scale_add_rows(out, y, rows, weights, sigmoid)
