"""Python faces of ``csrc/routed_ffn.hip``: the router's choice of experts and the experts' products."""
from __future__ import annotations

from typing import Optional

import torch

from . import kernels, library
from .kernels import _P, _I, _L, _F, _dev, _f32vec, _i32, _rows, dt, ptr, stream

LIBRARY = "routed_ffn"
MAX_OUTPUTS = 1024

kernels.register_signatures(LIBRARY, {
    "agave_route_topk": [_P, _L, _P, _P, _I, _I, _I, _I, _I, _F, _P, _P, _P],
    "agave_routed_experts_plain": [_I, _P, _L, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _F, _F, _P],
    "agave_route_rows": [_I, _P, _L, _P, _P, _I, _I, _I, _I, _I, _I, _F, _P, _P, _I, _I, _P, _I, _I, _I, _I, _P],
    "agave_routed_few_takes": [_I],
    "agave_route_sort": [_P, _I, _I, _I, _I, _I, _P, _P, _P, _P],
    "agave_routed_chosen_takes": [_I, _I, _I, _I],
    "agave_routed_experts_chosen": [_P, _L, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _F, _F, _P],
    "agave_routed_experts_mfma": [_P, _L, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _I, _F, _F, _P],
    "agave_routed_norm": [_I, _P, _P, _P, _P, _P, _I, _I, _P, _L, _P, _P, _F, _P, _L, _P, _F, _I, _I, _P],
    "agave_routed_combine": [_I, _P, _P, _P, _P, _P, _L, _P, _L, _P, _P, _L, _I, _I, _I, _I, _P],
})


def _lib():
    return kernels.lib(LIBRARY)


def route_topk(logits: torch.Tensor, correction: Optional[torch.Tensor], scratch: torch.Tensor, groups: int, keep: int,
               top: int, scale: float, choice: torch.Tensor, weight: torch.Tensor) -> None:
    """For every row of 32-bit router logits [N, R]: s = softmax; among the outputs of the ``keep`` groups (of
    ``groups`` equal groups of neighbours) whose largest ``s + correction`` is largest, the ``top`` outputs with the
    largest ``s + correction`` go to ``choice`` [N, top] (int32) and ``s * scale`` to ``weight`` [N, top]."""
    _dev(logits, correction, scratch, choice, weight)
    n, r = logits.shape
    if logits.dtype != torch.float32 or logits.stride(1) != 1:
        raise TypeError("route_topk: router logits must be float32 rows")
    _f32vec(correction, "correction", r)
    if scratch.dtype != torch.float32 or not scratch.is_contiguous() or scratch.numel() < n * r:
        raise ValueError("route_topk: scratch must hold a float32 value per logit")
    _i32(choice, "choice", n * top)
    if weight.dtype != torch.float32 or not weight.is_contiguous() or weight.numel() < n * top:
        raise ValueError("route_topk: weight must be contiguous float32 [N, top]")
    library.call(_lib(), "agave_route_topk", ptr(logits), logits.stride(0), ptr(correction), ptr(scratch), n, r, groups, keep,
                 top, float(scale), ptr(choice), ptr(weight), stream())


def experts_plain(x: torch.Tensor, choice: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, w_down: torch.Tensor,
                  act_rows: torch.Tensor, y: torch.Tensor, top: int, activation: int, p0: float = 0.0, p1: float = 1.0) -> None:
    """y[p] = W_down[e] (act(W_gate[e] x_t) * (W_up[e] x_t)) for every pair p = t * top + slot whose choice e is an
    expert with weights (e < E); rows of other pairs are left alone.  ``y`` is float32 [N * top, hidden]."""
    _dev(x, choice, w_gate, w_up, w_down, act_rows, y)
    n, hidden = x.shape
    ldx = _rows(x, "x")
    e, ff, k = w_gate.shape
    if k != hidden or w_up.shape != w_gate.shape or w_down.shape != (e, hidden, ff):
        raise ValueError("experts: weights must be [E, ff, hidden], [E, ff, hidden] and [E, hidden, ff]")
    for w in (w_gate, w_up, w_down):
        if w.dtype != x.dtype or not w.is_contiguous():
            raise TypeError("experts: weights must be contiguous and of the rows' dtype")
    _i32(choice, "choice", n * top)
    if act_rows.dtype != x.dtype or not act_rows.is_contiguous() or act_rows.shape != (n * top, ff):
        raise ValueError(f"experts: inner rows must be [{n * top}, {ff}] of the rows' dtype")
    if y.dtype != torch.float32 or not y.is_contiguous() or y.shape != (n * top, hidden):
        raise ValueError(f"experts: y must be float32 [{n * top}, {hidden}]")
    library.call(_lib(), "agave_routed_experts_plain", dt(x), ptr(x), ldx, ptr(choice), ptr(w_gate), ptr(w_up), ptr(w_down),
                 ptr(act_rows), ptr(y), n, top, e, ff, hidden, activation, float(p0), float(p1), stream())


def _check_pairs(y: Optional[torch.Tensor], place: Optional[torch.Tensor], choice: torch.Tensor, x: torch.Tensor,
                 shared: Optional[torch.Tensor], top: int, shared_gate: Optional[torch.Tensor]) -> int:
    """What is added up to rows like ``x``: the pairs' rows and the shared expert's, whose stride comes back."""
    n, hidden = x.shape
    _f32vec(shared_gate, "shared_gate", n)
    if shared is not None and (shared.shape != x.shape or shared.dtype != x.dtype):
        raise ValueError("combine: the shared expert's rows must have the input's shape and dtype")
    if y is not None and (y.dtype != torch.float32 or not y.is_contiguous() or y.shape[1] != hidden or y.shape[0] < n * top):
        raise ValueError("combine: y must be float32 [>= N * top, hidden]")
    _i32(choice, "choice", n * top)
    _i32(place, "place", n * top)
    return _rows(shared, "shared") if shared is not None else 0


def combine(y: Optional[torch.Tensor], place: Optional[torch.Tensor], choice: torch.Tensor, weight: torch.Tensor,
            x: torch.Tensor, shared: Optional[torch.Tensor], out: torch.Tensor, top: int, n_experts: int,
            shared_gate: Optional[torch.Tensor] = None) -> None:
    """out[t] = sum over the token's pairs of weight * (the pair's expert row of ``y``, or ``x[t]`` itself where the
    choice is an identity expert, e >= n_experts) + shared[t], the latter times ``sigmoid(shared_gate[t])`` where a
    float32 logit per token is given."""
    _dev(y, place, choice, weight, x, shared, out, shared_gate)
    n, hidden = x.shape
    ldx, ldo = _rows(x, "x"), _rows(out, "out")
    if out.shape != x.shape or out.dtype != x.dtype:
        raise ValueError("combine: out must have the input's shape and dtype")
    lds = _check_pairs(y, place, choice, x, shared, top, shared_gate)
    library.call(_lib(), "agave_routed_combine", dt(x), ptr(y), ptr(place), ptr(choice), ptr(weight), ptr(x), ldx, ptr(shared),
                 lds, ptr(shared_gate) if shared is not None else None, ptr(out), ldo, n, top, n_experts, hidden, stream())


def norm_adds_up(n: int, top: int, hidden: int) -> bool:
    """Whether the norm of ``n`` tokens adds up ``top`` pairs each: a workgroup takes a token's rows, so with few tokens many and wide
    ones take longer than in the kernel that spreads them over the chip and the norm's own.  us, those two and the one kernel: 16,384
    columns of 64 pairs, 6 tokens 17.7 and 42, of 16 10.0 and 12.9, of 7 8.9 and 9.2, of 6 8.7 and 8.2; 8,192 of 16 8.2 and 9.0, of 10
    7.6 and 6.2; 7,168 of 12 7.3 and 7.4 (one token); 4,096 of 64 14.5 and 13.6.  48 tokens: 16,384 of 24 20.9 and 21.7, 12,288 of 24
    19.1 and 18.2; 300 tokens 5,120 of 64 84 and 88, of 32 36.0 and 36.7.  Over 17 widths, 14 numbers of pairs, one to 800
    tokens and both types one within these lines was slower by more than 1 % (800 tokens, 4,608 of 16: 48.4 and 50.5)."""
    return hidden <= 4096 or top * hidden <= 84_000 or (n >= 48 and top <= 24 and top * hidden <= 300_000)


class RoutedRows:
    """A routed feed-forward's result that is still its pairs' rows: the arguments of :func:`combine`.  The norm that takes it
    adds the pairs up itself (:meth:`norm_into`) where it can; whoever cannot asks for the rows (:meth:`rows`)."""

    def __init__(self, y, place, choice, weight, x, shared, out, top, n_experts, shared_gate):
        self.arguments = (y, place, choice, weight, x, shared, out, top, n_experts, shared_gate)
        self._rows: Optional[torch.Tensor] = None

    def rows(self) -> torch.Tensor:
        if self._rows is None:
            combine(*self.arguments)
            self._rows = self.arguments[6]
        return self._rows

    def norm_into(self, h: torch.Tensor, post_gain: Optional[torch.Tensor], post_eps: float, out: torch.Tensor,
                  pre_gain: Optional[torch.Tensor], pre_eps: float) -> bool:
        """``h += post(rows)`` and ``out = rmsnorm(h) * pre_gain`` (or the rows of ``h`` without a gain) in one kernel, if it takes
        these sizes, is the faster way (:func:`norm_adds_up`) and nothing was added up yet."""
        y, place, choice, weight, x, shared, _, top, n_experts, shared_gate = self.arguments
        n, e = h.shape
        if y is None or self._rows is not None or not norm_adds_up(n, top, e) or e % 4 or e > 16384 or out.dtype != x.dtype or h.shape != x.shape:
            return False
        for t in (h, y, shared, post_gain, out, pre_gain):
            if t is not None and (t.data_ptr() % 16 or (t.dim() == 2 and (t.stride(1) != 1 or t.stride(0) % 4))):
                return False
        if not h.is_contiguous() or h.dtype != torch.float32 or out.shape != x.shape:
            return False
        _dev(h, y, place, choice, weight, shared, shared_gate, post_gain, out, pre_gain)
        _f32vec(post_gain, "post_gain", e)
        _f32vec(pre_gain, "pre_gain", e)
        lds = _check_pairs(y, place, choice, x, shared, top, shared_gate)
        library.call(_lib(), "agave_routed_norm", dt(out), ptr(h), ptr(y), ptr(place), ptr(choice), ptr(weight), top, n_experts, ptr(shared), lds,
                     ptr(shared_gate) if shared is not None else None, ptr(post_gain),
                     float(post_eps), ptr(out), out.stride(0), ptr(pre_gain), float(pre_eps), n, e, stream())
        return True


STREAMED = (1024, 2048, 4096)        # columns for which the kernel of few pairs is built (agave_routed_few_takes)


def tile_plan(n_pairs: int, n_experts: int, tile_order: bool = False, ff: int = 0, hidden: int = 0):
    """(rows a tile, tiles at most, sorted rows at most) of the sorted list of ``n_pairs`` pairs; every expert's run of rows
    is padded to whole tiles, so there are at most ``ceil(pairs / rows) + experts`` tiles.

    Weights row by row: tiles of 64 rows where an expert gets some 32 pairs or more on average, of 16 otherwise.
    Weights in tile order (``tile_order``, experts of ``ff`` inner rows and ``hidden`` columns): 128 from 128 pairs an expert
    on where their workgroups (128 inner rows, 256 columns each) fill the chip; else 64 from 32 pairs an expert on, and from
    16 on where their workgroups (64 inner rows, 128 columns each) about fill the chip; below that 16.  Where neither product
    has the columns that the kernel of few pairs streams, 64 from two pairs an expert on.  us, both products in tiles of 16 and
    of 64: 16 experts of 2,048 by 2,048 4 pairs an expert 85 and 89, 8 87 and 88, 12 90 and 89, 16 114 and 91; 64 of 512 by
    2,048 4 88 and 101, 12 100 and 104, 16 112 and 106; 32 of 1,024 by 1,024 8 49 and 53, 16 63 and 54; 16 of 1,536 by 1,536
    2 63 and 57, 16 91 and 60.  With workgroups for a part of the chip: 8 of 512 by 512 16 12 and 20, 4 of 2,048 by 1,024 16 23
    and 34.  In tiles of 64 and of 128: 16 experts of 2,048 by 2,048 64 pairs an expert 124 and 128, 128 162 and 150, 750 532
    and 408; 64 of 512 by 2,048 128 169 and 172, 375 349 and 285; 4 of 2,048 by 1,024 512 72 and 82, 1,500 126 and 124; 8 of
    512 by 512 128 25 and 44, 750 45 and 53; 16 of 32 by 32 375 15 and 24 (without LDS 16)."""
    tm = 64 if n_pairs >= 32 * n_experts else 16
    if tile_order:
        live, full = min(n_pairs, n_experts), n_pairs // 128
        if n_pairs >= 128 * n_experts and full * (ff // 128) >= 256 and full * (hidden // 256) >= 128:
            tm = 128
        elif (n_pairs >= (16 if ff in STREAMED or hidden in STREAMED else 2) * n_experts
              and live * (ff // 64) >= 256 and live * (hidden // 128) >= 128):
            tm = 64
    tiles = (n_pairs + tm - 1) // tm + n_experts
    return tm, tiles, tiles * tm


def mfma_ok(x: torch.Tensor, ff: int) -> bool:
    """Whether the matrix-core kernels take these rows (bfloat16, sizes that are multiples of 8, aligned)."""
    return (x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0 and ff % 8 == 0 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0)


def route_sort(choice: torch.Tensor, n_experts: int, tm: int, tiles: int, place: torch.Tensor, sorted_pair: torch.Tensor,
               tile_expert: torch.Tensor) -> None:
    """Sort the pairs by expert on the device: ``place[p]`` the sorted row of pair p (-1 for an identity expert),
    ``sorted_pair[r]`` the pair in sorted row r (-1: padding), ``tile_expert[t]`` the expert of tile t (-1: none)."""
    _dev(choice, place, sorted_pair, tile_expert)
    p = choice.numel()
    _i32(choice, "choice")
    _i32(place, "place", p)
    _i32(sorted_pair, "sorted_pair", tiles * tm)
    _i32(tile_expert, "tile_expert", tiles)
    library.call(_lib(), "agave_route_sort", ptr(choice), p, n_experts, tm, tiles * tm, tiles, ptr(place), ptr(sorted_pair),
                 ptr(tile_expert), stream())


def experts_mfma(x: torch.Tensor, sorted_pair: torch.Tensor, tile_expert: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor,
                 w_down: torch.Tensor, act_rows: torch.Tensor, y: torch.Tensor, tm: int, tiles: int, top: int, activation: int,
                 tile_order: bool = False, p0: float = 0.0, p1: float = 1.0) -> None:
    """The experts' products over the sorted rows on the matrix cores: ``act_rows`` [tiles * tm, ff] bfloat16 and
    ``y`` [tiles * tm, hidden] float32 receive sorted rows (padding rows hold nothing of use).  ``tile_order``: the
    weights were rearranged by :func:`pack_expert_weights` (same shapes)."""
    _dev(x, sorted_pair, tile_expert, w_gate, w_up, w_down, act_rows, y)
    n, hidden = x.shape
    e, ff, k = w_gate.shape
    if k != hidden or w_up.shape != w_gate.shape or w_down.shape != (e, hidden, ff):
        raise ValueError("experts: weights must be [E, ff, hidden], [E, ff, hidden] and [E, hidden, ff]")
    for w in (w_gate, w_up, w_down):
        if w.dtype != torch.bfloat16 or not w.is_contiguous():
            raise TypeError("experts: the matrix-core kernels take contiguous bfloat16 weights")
    if not mfma_ok(x, ff):
        raise ValueError("experts: rows that the matrix-core kernels do not take")
    cap = tiles * tm
    if act_rows.dtype != torch.bfloat16 or not act_rows.is_contiguous() or act_rows.shape != (cap, ff):
        raise ValueError(f"experts: inner rows must be bfloat16 [{cap}, {ff}]")
    if y.dtype != torch.float32 or not y.is_contiguous() or y.shape != (cap, hidden):
        raise ValueError(f"experts: y must be float32 [{cap}, {hidden}]")
    _i32(sorted_pair, "sorted_pair", cap)
    _i32(tile_expert, "tile_expert", tiles)
    library.call(_lib(), "agave_routed_experts_mfma", ptr(x), x.stride(0), ptr(sorted_pair), ptr(tile_expert), ptr(w_gate),
                 ptr(w_up), ptr(w_down), ptr(act_rows), ptr(y), tm, tiles, n, top, e, ff, hidden, activation,
                 1 if tile_order else 0, float(p0), float(p1), stream())


def chosen_takes(n_pairs: int, n_experts: int, ff: int, hidden: int) -> bool:
    """Whether :func:`experts_chosen` takes this many pairs of experts of these sizes (held in tile order)."""
    return bool(_lib().agave_routed_chosen_takes(n_pairs, n_experts, ff, hidden))


def experts_chosen(x: torch.Tensor, choice: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, w_down: torch.Tensor,
                   act_rows: torch.Tensor, y: torch.Tensor, top: int, activation: int, p0: float = 0.0, p1: float = 1.0) -> None:
    """The experts' products of few pairs, straight from the pairs' choices: ``act_rows`` [N * top, ff] bfloat16 and ``y``
    [N * top, hidden] float32 receive a row a pair (nothing where the choice is no expert).  The weights were rearranged by
    :func:`pack_expert_weights`."""
    _dev(x, choice, w_gate, w_up, w_down, act_rows, y)
    n, hidden = x.shape
    e, ff, k = w_gate.shape
    if k != hidden or w_up.shape != w_gate.shape or w_down.shape != (e, hidden, ff):
        raise ValueError("experts: weights must be [E, ff, hidden], [E, ff, hidden] and [E, hidden, ff]")
    for w in (w_gate, w_up, w_down):
        if w.dtype != torch.bfloat16 or not w.is_contiguous():
            raise TypeError("experts: the matrix-core kernels take contiguous bfloat16 weights")
    if not mfma_ok(x, ff) or x.stride(1) != 1 or not chosen_takes(n * top, e, ff, hidden):
        raise ValueError("experts: rows or sizes that the kernel of few pairs does not take")
    if act_rows.dtype != torch.bfloat16 or not act_rows.is_contiguous() or act_rows.shape != (n * top, ff):
        raise ValueError(f"experts: inner rows must be bfloat16 [{n * top}, {ff}]")
    if y.dtype != torch.float32 or not y.is_contiguous() or y.shape != (n * top, hidden):
        raise ValueError(f"experts: y must be float32 [{n * top}, {hidden}]")
    _i32(choice, "choice", n * top)
    library.call(_lib(), "agave_routed_experts_chosen", ptr(x), x.stride(0), ptr(choice), ptr(w_gate), ptr(w_up), ptr(w_down),
                 ptr(act_rows), ptr(y), n, top, e, ff, hidden, activation, float(p0), float(p1), stream())


def route_rows(x: torch.Tensor, router: torch.Tensor, correction: Optional[torch.Tensor], groups: int, keep: int, top: int,
               scale: float, choice: torch.Tensor, weight: torch.Tensor, softmax_top: bool = False,
               extra_out: Optional[torch.Tensor] = None, sigmoid: bool = False, group_top: int = 1,
               normalise: bool = False, shared_expert: Optional[int] = None, shared_gate: bool = False) -> None:
    """The router's 32-bit product ``x router^T`` and :func:`route_topk`'s choice in one kernel (the logits never
    leave the compute unit).  ``router`` is float32 [R, width]; ``x`` [N, width] in either element type.
    ``softmax_top``: the ``top`` largest logits + ``correction`` are chosen (the lower index among equals) and their
    weights are the softmax over the chosen alone, times ``scale`` (no groups, ``top`` <= 64).  ``extra_out``
    (float32 [N, extra]): the router matrix has ``extra`` further rows behind its outputs, whose products with
    the rows are left there as they are.  ``sigmoid``: the scores are the logits' sigmoids instead of their softmax.
    ``group_top`` 2: a group counts by the sum of its two largest scores + correction.  ``normalise``: the chosen
    weights are divided by their sum + 1e-20 before ``scale`` (``top`` <= 64).  ``shared_expert``: ``choice`` and ``weight`` are
    [N, top + 1], and every token's last pair is this expert with the weight 1 or, with ``shared_gate``, the sigmoid of
    the product with one further row of the router matrix."""
    _dev(x, router, correction, choice, weight, extra_out)
    n, k = x.shape
    ldx = _rows(x, "x")
    if router.dtype != torch.float32 or router.dim() != 2 or router.shape[1] != k or not router.is_contiguous():
        raise ValueError(f"route_rows: the router must be contiguous float32 [outputs, {k}]")
    extra = 0
    if extra_out is not None:
        if extra_out.dtype != torch.float32 or extra_out.dim() != 2 or extra_out.shape[0] != n or not extra_out.is_contiguous():
            raise ValueError(f"route_rows: extra_out must be contiguous float32 [{n}, extra]")
        extra = extra_out.shape[1]
    if shared_gate:
        if shared_expert is None or extra:
            raise ValueError("route_rows: a gate is a shared expert's, and then the only further row")
        extra = 1
    pairs = top + (shared_expert is not None)
    r = router.shape[0] - extra
    if r < 1:
        raise ValueError("route_rows: the router has no outputs")
    if softmax_top and (groups != 1 or keep != 1 or top > 64):
        raise ValueError("route_rows: the softmax over the chosen logits takes no groups and at most 64 chosen")
    if softmax_top and (sigmoid or normalise):
        raise ValueError("route_rows: one way of scoring at a time")
    if group_top not in (1, 2) or (normalise and top > 64):
        raise ValueError("route_rows: a group counts by its largest or its two largest scores; weights are divided by their "
                         "sum for at most 64 chosen")
    _f32vec(correction, "correction", r)
    _i32(choice, "choice", n * pairs)
    if weight.dtype != torch.float32 or not weight.is_contiguous() or weight.numel() < n * pairs:
        raise ValueError("route_rows: weight must be contiguous float32, a value per pair")
    library.call(_lib(), "agave_route_rows", dt(x), ptr(x), ldx, ptr(router), ptr(correction), n, k, r, groups, keep, top,
                 float(scale), ptr(choice), ptr(weight), 1 if softmax_top else (2 if sigmoid else 0), extra, ptr(extra_out),
                 int(group_top), 1 if normalise else 0, pairs, -1 if shared_expert is None else int(shared_expert), stream())


def pack_expert_weights(w: torch.Tensor) -> torch.Tensor:
    """[E, N, K] (N a multiple of 16, K of 32) rearranged into the matrix cores' operand tiles: tiles of 16 rows by 32
    columns, each stored as its 64 lanes' 16 bytes one after another (lane c + 16 g holds row c, columns 8 g .. 8 g + 7),
    a row block's tiles along K following each other.  Same shape and bytes; only :func:`experts_mfma` reads it."""
    e, n, k = w.shape
    if n % 16 or k % 32:
        raise ValueError("pack_expert_weights: rows must be a multiple of 16 and columns of 32")
    t = w.view(e, n // 16, 16, k // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()      # [E, nb, kb, g, c, 8]
    return t.view(e, n, k)
