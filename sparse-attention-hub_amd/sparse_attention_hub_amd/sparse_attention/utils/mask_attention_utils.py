"""Masked-softmax attention over the selected KV rows.

Host side of `sah_sparse_attention` (include/sah.h). Same call signature and
results as the reference's `get_masked_attention_output`
(sparse_attention/utils/mask_attention_utils.py:406-491), which computes
fp32 logits over *all* keys, multiplies exp(logit - rowmax) by the inverse mask
weight 1/(w + 1e-6) and divides numerator by denominator; here only the rows the
mask selects are read (an empty or full mask selects every key, as in the
reference, utils/mask.py:733-735).
"""
from __future__ import annotations

import itertools
import threading
from typing import Any, Dict, Optional, Tuple, Union


import numpy as np
import torch
from torch import nn

from ... import _native as N
from .kv_utils import _get_num_key_value_groups
from .mask import Mask
from .native_rows import NativeRows

_WORK_STREAMS = 8  # scratch buffers a thread keeps ...
_WORK_FLOATS = 1 << 24  # ... of at most this size: 64 MiB


class _Scratch(threading.local):
    def __init__(self) -> None:
        self.buffers: Dict[Tuple[Optional[int], int], torch.Tensor] = {}


_WORK = _Scratch()


def _workspace(device: torch.device, floats: int, stream: int, capturing: Optional[bool] = None) -> torch.Tensor:
    """Grow-only fp32 scratch of the calling thread for the current stream of `device` (whose handle is `stream`): calls on
    other streams are not ordered with this one's, and another thread's may come between the two kernels of a call. The
    latest few streams' buffers are kept until the thread ends; one that goes was allocated on its stream, so torch's
    allocator hands its memory to later work of that stream. Large ones (many query vectors of a long pass, merged in
    milliseconds) are the call's. A captured call's scratch is its graph's own: replays use it whatever this thread keeps."""
    if floats > _WORK_FLOATS or (torch.cuda.is_current_stream_capturing() if capturing is None else capturing):
        return torch.empty(floats, dtype=torch.float32, device=device)
    key = (device.index, stream)
    buffers = _WORK.buffers
    buf = buffers.get(key)
    if buf is None or buf.numel() < floats:
        buffers.pop(key, None)
        if len(buffers) >= _WORK_STREAMS:
            del buffers[next(iter(buffers))]
        buf = buffers[key] = torch.empty(max(floats, 1 << 16), dtype=torch.float32, device=device)
    return buf


def dense_rows_possible(n_queries: int, dtype: torch.dtype, head_dim: int) -> bool:
    """May attention over unit-weight rows of this geometry take the matrix-core form (`sah_members_attention`), which needs
    the rows' bitmaps and scratch of its own?"""
    return n_queries > 1 and dtype != torch.float32 and head_dim in (64, 128)


def _inner_contiguous(t: torch.Tensor) -> torch.Tensor:
    return t if t.stride(-1) == 1 else t.contiguous()


def unit_inverse_weight(dtype: torch.dtype) -> float:
    """1 / (1 + 1e-6) evaluated in the mask dtype, as `Mask.apply_inv_mask` does for weight 1.0."""
    if dtype == torch.float32:
        return float(np.float32(1.0) / (np.float32(1.0) + np.float32(1e-6)))
    return 1.0  # bf16 / fp16: 1 + 1e-6 rounds back to 1


def mask_covers(am: torch.Tensor, queries: torch.Tensor, n_keys: int) -> bool:
    """Has the 4-dimensional mask a row for every query, as wide as the keys?"""
    m, q = am.shape, queries.shape
    return m[3] >= n_keys and m[2] == q[2] and m[0] in (1, q[0]) and m[1] in (1, q[1])


def additive_mask_args(attention_mask: Optional[torch.Tensor], queries: torch.Tensor, n_keys: int):
    """(tensor kept alive, ptr, stride_b, stride_h, stride_q) of the additive mask or all-None/0."""
    if attention_mask is None:
        return None, None, 0, 0, 0
    am = attention_mask
    if am.dim() != 4:
        raise ValueError(f"attention_mask must have 4 dimensions, got shape {tuple(am.shape)}")
    if not mask_covers(am, queries, n_keys):
        raise ValueError(f"attention_mask shape {tuple(am.shape)} does not cover queries {tuple(queries.shape)} x {n_keys} keys")
    if am.dtype != queries.dtype:
        am = am.to(queries.dtype)
    am = _inner_contiguous(am)
    N.require_device(am, "attention_mask")
    sb = am.stride(0) if am.shape[0] > 1 else 0
    sh = am.stride(1) if am.shape[1] > 1 else 0
    return am, am.data_ptr(), sb, sh, am.stride(2)


class _AnswerWords(threading.local):
    """Per thread and device: two words of device memory and one of pinned host memory, through which a mask's question is
    answered, and the thread's question that waits for its answer (one at a time; a call that asks takes the answer before it
    returns or raises)."""

    def __init__(self) -> None:
        self.words = {}
        self.blocks = {}  # the argument block of a question, and of its mask
        self.open = {}


_ANSWERS = _AnswerWords()


def _answer_words(device: torch.device):
    words = _ANSWERS.words.get(device.index)
    if words is None:
        with torch.cuda.device(device):
            if torch.cuda.is_current_stream_capturing():
                # (as sah_amask_read itself refuses.) Words made now would lie in the graph's memory, cleared by replays alone.
                raise N.NativeLibraryError("what a mask holds cannot be read back while the stream is captured")
            scratch = torch.zeros(2, dtype=torch.int32, device=device)
            torch.cuda.current_stream().synchronize()  # once: a question refused now is followed by one of another stream
        words = _ANSWERS.words[device.index] = (scratch, torch.zeros(1, dtype=torch.int64, pin_memory=True))
    return words


class MaskQuestion:
    """What does this mask hold? Asked of the device when made; `settle` waits for the answer."""

    def __init__(self, am: torch.Tensor) -> None:
        dev = am.device
        scratch, word = _answer_words(dev)
        earlier = _ANSWERS.open.get(dev.index)
        if earlier is not None:
            earlier.settle()
        # (mask and words stay allocated until the answer)
        self.mask, self.version, self.flags, self._words = am, am._version, None, (scratch, word)
        b, h, n_q, n = am.shape
        sb, sh, sq, _ = am.stride()
        self.one_query = n_q == 1
        block = _ANSWERS.blocks.get(dev.index)
        if block is None:
            args = N.AmaskQuestion()
            args.read.scratch, args.read.host_word = scratch.data_ptr(), word.data_ptr()
            block = _ANSWERS.blocks[dev.index] = args, args.read.mask
        args, m = block
        m.amask, m.ms_b, m.ms_h, m.ms_l, m.dtype = am.data_ptr(), sb, sh, sq, N.dtype_code(am.dtype)
        m.B, m.Hm, m.Lq, m.Lk, m.stream = b, h, n_q, n, N.stream_ptr(dev)
        N.call("sah_amask_ask", args)
        self._args = args
        _ANSWERS.open[dev.index] = self

    def settle(self) -> int:
        if self.flags is None:
            _ANSWERS.open.pop(self.mask.device.index, None)
            N.call("sah_amask_answer", self._args)
            self.flags = self._args.read.flags
        return self.flags

    def __del__(self) -> None:
        # a thread that ends on a call that failed in between: the words go only after the kernel has written them
        if getattr(self, "_args", None) is not None and self.flags is None:
            try:
                N.call("sah_amask_answer", self._args)
            except Exception:
                pass


class AdditiveMaskFacts:
    """What the additive mask of the current forward pass holds, established once per mask tensor.

    HuggingFace builds one mask per forward pass and hands the same tensor to every layer; for a single decode
    query of an unpadded batch its eager mask is all zeros, and adding zeros to scores and logits changes nothing
    (reference: hashattention_top_k.py:367-368, oracle_top_k.py:71-72, utils/mask_attention_utils.py:221-225).
    The device is asked once per tensor (one small launch, answered into host memory, over the mask's whole width: a
    mask that is zero everywhere is zero on the columns of any key count) and the answer remembered for as long as
    the same, unmodified tensor keeps arriving; the tensor is kept referenced meanwhile, so its memory cannot be
    handed to another tensor that would then be mistaken for it.

    What a session's last mask held is the guess for its next one. It is kept in the session's own `sparse_meta_data` (sessions
    with and without padding that take turns are each guessed right), under names of this object's."""

    _numbers = itertools.count()

    def __init__(self) -> None:
        self._seen: Tuple[Optional[torch.Tensor], int, int] = (None, -1, 0)  # tensor, its version, flags
        number = next(self._numbers)
        self._one, self._several = f"{number} one query", f"{number} several queries"

    def known(self, am: torch.Tensor) -> Optional[int]:
        tensor, version, flags = self._seen
        if am is tensor and am._version == version:
            return flags
        if am.dim() != 4 or am.stride(-1) != 1 or not am.is_cuda or am.numel() == 0:
            return N.AMASK_NONZERO | N.AMASK_GENERAL  # nothing established: every consumer reads the mask itself
        return None

    def guess(self, one_query: bool, session: Any) -> Optional[int]:
        """The flags of the session's last mask for one query, or for several."""
        last = session.get("additive_mask_flags") if isinstance(session, dict) else None
        return None if last is None else last.get(self._one if one_query else self._several)

    def take(self, question: MaskQuestion, session: Any = None) -> int:
        flags = question.settle()
        self._seen = (question.mask, question.version, flags)
        if isinstance(session, dict):  # (a dictionary under a name, as the caches are)
            session.setdefault("additive_mask_flags", {})[self._one if question.one_query else self._several] = flags
        return flags

    def flags(self, attention_mask: torch.Tensor) -> int:
        known = self.known(attention_mask)
        return self.take(MaskQuestion(attention_mask)) if known is None else known


def _run_attention(
    queries: torch.Tensor,
    keys: torch.Tensor,
    values: torch.Tensor,
    attention_mask: Optional[torch.Tensor],
    sinks: Optional[torch.Tensor],
    scaling: float,
    rows: Optional[NativeRows],
    return_attention_weights: bool,
    out: Optional[torch.Tensor] = None,
    return_stats: bool = False,
    dropout: Tuple[float, int, int] = (0.0, 0, 0),
    dropout_numerator_only: bool = False,
    score_keys: Optional[Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]] = None,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """rows=None => dense attention over all keys. `return_stats`: the second value is the kernel's
    fp32 (n_rows, 2) tensor of (largest logit among the row's entries, softmax denominator relative to it)
    instead of the dense probabilities. `score_keys`: the (n_rows, >= Lk) 16-bit keys and remainders
    `sah_qk_scores` wrote for these queries and keys without an additive mask, when a masker of this call has scored
    every key already - the kernel then takes its logits from there and does not read K."""
    N.require_device(queries, "queries")
    N.require_device(keys, "keys")
    N.require_device(values, "values")
    B, Hq, Lq, D = queries.shape
    Hkv, Lk = keys.shape[1], keys.shape[2]
    _get_num_key_value_groups(queries, keys)
    _get_num_key_value_groups(queries, values)
    if keys.dtype != queries.dtype or values.dtype != queries.dtype:
        raise ValueError(f"queries/keys/values dtypes differ: {queries.dtype}, {keys.dtype}, {values.dtype}")
    q = _inner_contiguous(queries)
    k = _inner_contiguous(keys)
    v = _inner_contiguous(values)
    dev = q.device
    dt = N.dtype_code(q.dtype)
    n_rows = B * Hq * Lq
    dense = rows is None
    if dense:
        max_cnt = Lk
        rows_struct = N.Rows(None, None, None, None, n_rows, Lk, Lk, (Lk + 31) // 32)
        unit = 1.0
    else:
        rows.zero_if_fresh()
        max_cnt = max(1, rows.max_cnt)
        rows_struct = rows.as_struct()
        unit = unit_inverse_weight(q.dtype)
    am_keep, am_ptr, ms_b, ms_h, ms_l = additive_mask_args(attention_mask, q, Lk)
    sink_t = None
    if sinks is not None:
        assert sinks.ndim == 1, f"sinks must be 1D tensor of shape [H], got {sinks.shape}"
        sink_t = sinks.to(device=dev, dtype=torch.float32).contiguous()
    if out is None:
        out = torch.empty((B, Lq, Hq, D), dtype=q.dtype, device=dev)
    floats = N.work_floats(n_rows, max_cnt, D)
    members = (dense_rows_possible(Lq, q.dtype, D) and not return_attention_weights and not return_stats
               and dropout[0] == 0.0 and (dense or rows.w is None))
    if members:  # many query vectors per KV head: the matrix-core form keeps partial results of its own
        floats = max(floats, N.members_work_floats(B, Hq, Hkv, Lq, Lk, D))
    stream = N.stream_ptr(dev)
    work = _workspace(dev, floats, stream)
    logits = stats = None
    if return_attention_weights:
        logits = torch.empty((n_rows, Lk if dense else rows.cap), dtype=torch.float32, device=dev)
    if return_attention_weights or return_stats:
        stats = torch.empty((n_rows, 2), dtype=torch.float32, device=dev)
    args = N.AttentionArgs(
        rows_struct,
        q.data_ptr(), q.stride(0), q.stride(1), q.stride(2),
        k.data_ptr(), k.stride(0), k.stride(1), k.stride(2),
        v.data_ptr(), v.stride(0), v.stride(1), v.stride(2),
        am_ptr, ms_b, ms_h, ms_l,
        None if sink_t is None else sink_t.data_ptr(),
        dt, B, Hq, Hkv, Lq, Lk, D,
        float(scaling), unit,
        1 if dense else 0,
        0, 0, 0,
        max_cnt,
        out.data_ptr(),
        work.data_ptr(), work.numel(),
        None if logits is None else logits.data_ptr(),
        None if stats is None else stats.data_ptr(),
        stream,
        dropout[0], dropout[1], dropout[2], int(dropout_numerator_only),
    )
    sk, sr = score_keys if score_keys is not None else (None, None)
    if (sk is not None and sr is not None and not dense and sk.dtype == torch.int16 and sk.device == dev
            and sk.ndim == 2 and sk.shape[0] == n_rows and sk.stride(1) == 1 and sk.stride(0) >= Lk
            and sr.dtype == sk.dtype and sr.shape == sk.shape and sr.stride() == sk.stride()):
        args.score_keys, args.score_resid, args.score_pitch = sk.data_ptr(), sr.data_ptr(), sk.stride(0)
    # the rows' bitmap is coherent with their lists here (or the call is dense)
    N.call("sah_members_attention" if members else "sah_sparse_attention", args)
    if return_stats:
        return out, stats
    weights = None
    if return_attention_weights:
        weights = torch.zeros((B, Hq, Lq, Lk), dtype=q.dtype, device=dev)
        wargs = N.AttentionWeightsArgs(
            rows_struct, logits.data_ptr(), stats.data_ptr(), unit, 1 if dense else 0, dt,
            weights.data_ptr(), N.stream_ptr(dev), dropout[0], dropout[1], dropout[2],
        )
        N.call("sah_attention_weights", wargs)
    return out, weights


def _training_dropout(module: Optional[nn.Module], dropout: float) -> Tuple[float, int, int]:
    """(p, seed, offset) for the attention kernel: dropout of the exp weights applies in training mode only
    (reference: mask_attention_utils.py:234-238, `module.training`). The kernel draws with Philox4x32-10 keyed by
    torch's seed and a per-call offset where the reference draws from torch's generator: another stream of the same
    distribution. The offset is itself a draw from torch's default generator, so `torch.manual_seed(s)` followed by the
    same calls gives the same dropout masks again, as it does in the reference."""
    if not (dropout > 0.0 and module is not None and getattr(module, "training", False)):
        return 0.0, 0, 0
    if not dropout < 1.0:
        raise ValueError(f"dropout probability has to be below 1 for the attention kernel, but got {dropout}")
    offset = int(torch.randint(0, 2 ** 62, (1,), dtype=torch.int64).item())
    return float(dropout), int(torch.initial_seed()) & 0xFFFFFFFFFFFFFFFF, offset


def get_true_attention_output(
    module: nn.Module,
    queries: torch.Tensor,
    keys: torch.Tensor,
    values: torch.Tensor,
    attention_mask: Optional[torch.Tensor],
    scaling: float,
    dropout: float,
    **kwargs: Dict[str, Any],
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Dense attention output (B, Lq, Hq, D) (reference: mask_attention_utils.py:11-70). In training mode the
    reference's dense path is scaled_dot_product_attention with dropout_p (:40-52): dropout of the normalised
    probabilities, i.e. a dropped entry leaves the softmax denominator as it is."""
    out, _ = _run_attention(queries, keys, values, attention_mask, None, scaling, None, False,
                            dropout=_training_dropout(module, dropout), dropout_numerator_only=True)
    return out, None


def apply_inv_mask_sum(input_tensor: torch.Tensor, mask: Mask) -> torch.Tensor:
    """sum over the last dim of mask.apply_inv_mask(x); full/empty masks sum x (reference :73-101)."""
    if tuple(input_tensor.shape) != tuple(mask.shape):
        raise ValueError(f"input_tensor.shape must be {mask.shape}, got {input_tensor.shape}")
    if mask.is_full or mask.is_empty:
        return input_tensor.sum(dim=-1, keepdim=True)
    return mask.apply_inv_mask(input_tensor).sum(dim=-1, keepdim=True)


def get_masked_attention_output(
    module: nn.Module,
    queries: torch.Tensor,
    keys: torch.Tensor,
    values: torch.Tensor,
    attention_mask: Optional[torch.Tensor],
    sinks: Optional[torch.Tensor],
    scaling: float,
    dropout: float,
    sparse_attention_mask: Mask,
    return_attention_weights: bool = False,
    **kwargs: Dict[str, Any],
) -> Union[torch.Tensor, Tuple[torch.Tensor, torch.Tensor]]:
    """Masked attention output (B, Lq, Hq, D) in the query dtype, optionally with the
    dense probabilities (B, Hq, Lq, Lk)."""
    mask = sparse_attention_mask
    if mask.is_full or mask.is_empty:
        rows = None
    else:
        rows = mask.to_rows(0)
    out, weights = _run_attention(
        queries, keys, values, attention_mask, sinks, scaling, rows, return_attention_weights,
        dropout=_training_dropout(module, dropout), score_keys=kwargs.get("_score_keys"),
    )
    if return_attention_weights:
        return out, weights
    return out


# ------------------------------------------------------------------ numerator / denominator helpers
def _masked_softmax_parts(queries, keys, values, attention_mask, scaling, mask: Mask, dropout=(0.0, 0, 0)):
    """(out (B, Hq, Lq, D) fp32, den (B, Hq, Lq, 1) fp32, m_all (B, Hq, Lq, 1) fp32) of the masked softmax in the
    reference's scale, i.e. relative to the largest logit over ALL keys of the row
    (mask_attention_utils.py:187-240). Two launches of the attention kernel: one over the mask's rows, one dense
    pass whose statistics give the all-key maximum."""
    B, Hq, Lq, D = queries.shape
    rows = None if (mask.is_full or mask.is_empty) else mask.to_rows(0)
    out, stats = _run_attention(queries, keys, values, attention_mask, None, scaling, rows, False, return_stats=True,
                                dropout=dropout)
    if rows is None:
        all_stats = stats
    else:
        _, all_stats = _run_attention(queries, keys, values, attention_mask, None, scaling, None, False, return_stats=True)
    m_sel = stats[:, 0].view(B, Hq, Lq, 1)
    m_all = all_stats[:, 0].view(B, Hq, Lq, 1)
    den = stats[:, 1].view(B, Hq, Lq, 1) * torch.exp(m_sel - m_all)
    return out.transpose(1, 2).to(torch.float32), den, m_all


def get_attention_denominator(module: Optional[nn.Module], queries: torch.Tensor, keys: torch.Tensor,
                              attention_mask: Optional[torch.Tensor], scaling: float, dropout: float,
                              sparse_attention_mask: Mask, **kwargs: Dict[str, Any]) -> torch.Tensor:
    """sum_j exp(z_j - max_all z) / (w_j + 1e-6) over the mask's entries, (B, Hq, Lq, 1) fp32
    (reference: mask_attention_utils.py:271-311). The kernel needs a value tensor: the keys stand in."""
    _, den, _ = _masked_softmax_parts(queries, keys, keys, attention_mask, scaling, sparse_attention_mask,
                                      _training_dropout(module, dropout))
    return den


def get_attention_numerator(module: Optional[nn.Module], queries: torch.Tensor, keys: torch.Tensor, values: torch.Tensor,
                            attention_mask: Optional[torch.Tensor], scaling: float, dropout: float,
                            sparse_attention_mask: Mask, **kwargs: Dict[str, Any]) -> torch.Tensor:
    """sum_j exp(z_j - max_all z) / (w_j + 1e-6) * V_j, (B, Hq, Lq, D) fp32 (reference :314-355). Rebuilt as the
    kernel's normalised output times the denominator, so for bf16 / fp16 inputs it carries the output's rounding
    (one part in 2^8 / 2^11) where the reference's fp32 product does not."""
    out, den, _ = _masked_softmax_parts(queries, keys, values, attention_mask, scaling, sparse_attention_mask,
                                        _training_dropout(module, dropout))
    return out * den


def apply_sink_bias(num: torch.Tensor, den: torch.Tensor, exp_attention_weights: Optional[torch.Tensor],
                    queries: torch.Tensor, keys: torch.Tensor, attention_mask: Optional[torch.Tensor],
                    sinks: Optional[torch.Tensor], scaling: float):
    """Adds one attention-sink logit per query head to a softmax given as (numerator, denominator[, exp weights])
    in the all-key-maximum scale: everything is rescaled by exp(old_max - max(old_max, sink)) and the
    denominator gains exp(sink - new_max) (reference :357-402). The all-key maximum comes from a dense pass of
    the attention kernel; the rest is arithmetic on (B, Hq, Lq, 1) tensors."""
    if sinks is None:
        return num, den, exp_attention_weights
    assert sinks.ndim == 1, f"sinks must be 1D tensor of shape [H], got {sinks.shape}"
    B, H, Q = queries.shape[0], queries.shape[1], queries.shape[2]
    _, stats = _run_attention(queries, keys, keys, attention_mask, None, scaling, None, False, return_stats=True)
    old_max = stats[:, 0].view(B, H, Q, 1)
    sinks_row = sinks.to(device=old_max.device, dtype=torch.float32).view(1, H, 1, 1).expand(B, H, Q, 1)
    new_max = torch.maximum(old_max, sinks_row)
    scale = torch.exp(old_max - new_max).to(den.dtype)
    num = num * scale
    den = den * scale
    if exp_attention_weights is not None:
        exp_attention_weights = exp_attention_weights * scale
    den = den + torch.exp(sinks_row - new_max).to(den.dtype)
    return num, den, exp_attention_weights


def create_sampling_mask_with_per_head_budget(budgets: torch.Tensor, sampling_probability: torch.Tensor,
                                              seq_len_keys: int, start_idx: int, end_idx: int,
                                              dtype: torch.dtype = torch.float32, seed: Optional[int] = None,
                                              offset: int = 0) -> Mask:
    """Mask (B, H, Lq, seq_len_keys) in which row r holds the DISTINCT columns among `budgets[r]` uniform draws
    (with replacement) from [start_idx, end_idx), each with weight `sampling_probability[r]` rounded to `dtype`
    (reference: mask_attention_utils.py:105-184, one `sah_adaptive_sample` launch here, no host
    synchronisation). The reference lists a column once per draw in its index form; every consumer
    (dense conversion, merge) collapses such repeats to the one weight, which is what the rows hold here.
    Draws are Philox4x32-10 with key `seed` (default torch.initial_seed()) and stream `offset`."""
    if budgets.dim() != 4 or budgets.shape[-1] != 1 or sampling_probability.shape != budgets.shape:
        raise ValueError(f"budgets and sampling_probability must both be (b, h, q, 1), got {tuple(budgets.shape)} "
                         f"and {tuple(sampling_probability.shape)}")
    N.require_device(budgets, "budgets")
    B, H, Lq, _ = budgets.shape
    n = int(end_idx) - int(start_idx)
    if n <= 0 or start_idx < 0 or end_idx > seq_len_keys:
        raise ValueError(f"sampling range [{start_idx}, {end_idx}) is outside the {seq_len_keys} keys")
    dev = budgets.device
    n_rows = B * H * Lq
    rows = NativeRows(n_rows, int(seq_len_keys), n, dev, weighted=True)
    rows.zero_if_fresh()
    bud = budgets.reshape(n_rows).to(torch.int32).contiguous()
    N.dtype_code(dtype)
    prob = sampling_probability.reshape(n_rows).to(dtype).to(torch.float32).contiguous()
    key = (torch.initial_seed() if seed is None else int(seed)) & 0xFFFFFFFFFFFFFFFF
    N.call("sah_adaptive_sample", N.AdaptiveSampleArgs(
        rows.as_struct(), bud.data_ptr(), prob.data_ptr(), N.dtype_code(dtype),
        int(start_idx), n, key, int(offset), 1, N.stream_ptr(dev),
    ))
    rows.note_added(n, exact=False)
    return Mask.create_mask_from_rows((B, H, Lq, int(seq_len_keys)), rows, dtype)
