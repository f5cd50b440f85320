"""ResearchAttention: masker chain, then masked-softmax attention.

Reference: research_attention/base.py:24-196. Per call it starts from an empty
Mask of shape (B, Hq, Lq, Lk), lets every masker add to it in order, and hands the
result to `get_masked_attention_output`. The maskers here keep the mask in the
kernels' row layout, so one decode layer-step is a handful of HIP launches and no
dense (B, Hq, Lq, Lk) tensor unless the caller asks for the attention weights.
"""
from __future__ import annotations

import threading
from dataclasses import dataclass
from typing import Any, Dict, List, Optional, Tuple

import torch
from torch import nn

from ... import _native
from ...metric_logging import MicroMetricLogger
from ..base import SparseAttention, SparseAttentionConfig
from ..utils.mask import Mask
from ..utils.mask_attention_utils import (
    AdditiveMaskFacts, MaskQuestion, get_masked_attention_output, get_true_attention_output,
)
from ..utils.native_rows import NativeRows
from .decode_plan import DecodePlan, plan_kind
from .maskers.base import MaskerConfig, ResearchMasker
from .maskers.fixed.implementations.basic_fixed import LocalMasker, SinkMasker, fused_sink_local
from .maskers.sampling.base import SamplingMasker


# the two metrics of the reference (research_attention/base.py:20-21)
MicroMetricLogger.register_metric("research_attention_density", float)
MicroMetricLogger.register_metric("research_attention_output_error", float)


# Plans of steps whose mask is guessed to be zero that an instance keeps, over geometries, streams and threads: the latest ones made
# (making one at every step takes longer than the wait that a guess saves). Each holds its rows and 2 to 6 bytes of score keys a row
# and key.
_GUESSED_PLANS = 16


@dataclass
class ResearchAttentionConfig(SparseAttentionConfig):
    masker_configs: List[MaskerConfig]


class ResearchAttention(SparseAttention):
    maskers: List[ResearchMasker]

    # The reference always materialises the dense (B, Hq, Lq, Lk) probabilities as the
    # second return value (research_attention/base.py:146). HuggingFace attention modules
    # drop them unless output_attentions is set, so a caller may switch them off and get
    # None instead.
    return_attention_weights: bool = True

    def __init__(self, sparse_attention_config: SparseAttentionConfig, maskers: List[ResearchMasker]) -> None:
        super().__init__(sparse_attention_config)
        if sum(1 for m in maskers if isinstance(m, SamplingMasker)) > 1:
            raise ValueError(
                "Only one sampling masker supported for efficiency; consider implementing all sampling logic in one masker"
            )
        self.maskers = maskers
        self._plan_kind = plan_kind(maskers)
        self._plans: Dict[Any, DecodePlan] = {}
        self._mask_facts = AdditiveMaskFacts()

    def _planned_capacity(self, dims) -> Optional[int]:
        """Entries per row the whole chain can add, if every masker can tell without the device."""
        total = 0
        for masker in self.maskers:
            n = masker.max_new_entries(dims)
            if n is None:
                return None
            total += n
        return total

    def custom_attention(
        self,
        module: nn.Module,
        queries: torch.Tensor,
        keys: torch.Tensor,
        values: torch.Tensor,
        attention_mask: Optional[torch.Tensor],
        scaling: float,
        dropout: float,
        **kwargs: Dict[str, Any],
    ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
        """(attention output (B, Lq, Hq, D), attention weights (B, Hq, Lq, Lk) or None)."""
        if "sparse_meta_data" not in kwargs:
            raise ValueError("sparse_meta_data must be provided in kwargs while calling custom_attention()")
        sparse_meta_data: Dict[Any, Any] = kwargs.pop("sparse_meta_data")

        metrics = MicroMetricLogger()
        want_density = metrics.is_metric_enabled("research_attention_density")
        want_error = metrics.is_metric_enabled("research_attention_output_error")
        # the decode fast path: the whole chain as one native call over cached argument blocks
        plannable = (not (want_density or want_error)  # the metrics read the finished mask: masker-by-masker path
                     and not self.return_attention_weights and self._plan_kind is not None
                     and not isinstance(kwargs.get("s_aux"), torch.Tensor) and queries.dim() == 4
                     and not (dropout > 0.0 and module is not None and getattr(module, "training", False)))

        only_hides, out, question = False, None, None
        if attention_mask is not None:
            attention_mask, only_hides, out, question = self._under_mask(
                queries, keys, values, attention_mask, scaling, sparse_meta_data, kwargs.get("layer_idx"), plannable)
        if out is None and plannable and (attention_mask is None or queries.shape[2] == 1):
            out = self._plan_step(queries, keys, values, attention_mask, scaling, sparse_meta_data, kwargs.get("layer_idx"), only_hides)
        if out is not None:
            return out, None
        try:
            mask_shape = (queries.shape[0], queries.shape[1], queries.shape[2], keys.shape[2])
            mask = Mask.create_empty_mask(mask_shape, dtype=queries.dtype, device=queries.device)
            if self.maskers:
                # size the row buffers once for the whole chain so no masker has to grow them
                dims = self.maskers[0]._extract_tensor_dimensions(keys, queries)
                planned = self._planned_capacity(dims)
                if planned is not None and planned > 0:
                    rows = NativeRows(mask_shape[0] * mask_shape[1] * mask_shape[2], mask_shape[3], planned, queries.device)
                    mask = _EmptyRowsMask(mask_shape, rows, queries.dtype)

            maskers = self.maskers
            if (len(maskers) >= 2 and type(maskers[0]) is SinkMasker and type(maskers[1]) is LocalMasker
                    and not mask.is_full_mask()):
                # Sink directly followed by Local on a still-empty mask: one fused launch writes both ranges
                mask = fused_sink_local(maskers[0], maskers[1], keys, queries, mask)
                maskers = maskers[2:]

            # per-call scratch the maskers may share (e.g. the QK score keys of one scoring pass)
            call_scratch: Dict[str, Any] = {}
            for masker in maskers:
                mask = masker.add_mask(
                    keys=keys,
                    queries=queries,
                    values=values,
                    attention_mask=attention_mask,
                    scaling=scaling,
                    dropout=dropout,
                    sparse_meta_data=sparse_meta_data,
                    previous_mask=mask,
                    _call_scratch=call_scratch,
                    **kwargs,
                )

            if want_density:
                # active fraction of the (B, Hq, Lq, Lk) mask, from the per-row counts (reference :121-126)
                metrics.log("research_attention_density", mask.get_density(), metadata={"layer_idx": kwargs["layer_idx"]})

            s_aux_raw: Any = kwargs.pop("s_aux", None)
            s_aux: Optional[torch.Tensor] = s_aux_raw if isinstance(s_aux_raw, torch.Tensor) else None
            weights: Optional[torch.Tensor] = None
            # a masker of this call scored every key exactly (OracleTopK, AdaptiveSampling): the attention takes its
            # logits from those scores instead of reading K again
            kwargs["_score_keys"] = (call_scratch.get("qk_score_keys"), call_scratch.get("qk_score_resid"))
            if self.return_attention_weights:
                out, weights = get_masked_attention_output(
                    module=module, queries=queries, keys=keys, values=values, attention_mask=attention_mask,
                    sinks=s_aux, scaling=scaling, dropout=dropout, sparse_attention_mask=mask,
                    return_attention_weights=True, **kwargs,
                )
            else:
                out = get_masked_attention_output(
                    module=module, queries=queries, keys=keys, values=values, attention_mask=attention_mask,
                    sinks=s_aux, scaling=scaling, dropout=dropout, sparse_attention_mask=mask,
                    return_attention_weights=False, **kwargs,
                )
            if want_error:
                # relative distance to dense attention over all keys, by the same kernel in dense mode (reference :150-168)
                true_out, _ = get_true_attention_output(module, queries, keys, values, attention_mask, scaling, dropout, **kwargs)
                error = torch.norm(true_out.float() - out.float()) / torch.norm(true_out.float())
                metrics.log("research_attention_output_error", float(error.item()), metadata={"layer_idx": kwargs["layer_idx"]})
            return out, weights
        finally:
            if question is not None:
                self._mask_facts.take(question, sparse_meta_data)

    def _under_mask(self, queries: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, attention_mask: torch.Tensor,
                    scaling: float, sparse_meta_data: Dict[Any, Any], layer_idx: Optional[int], plannable: bool):
        """(the mask that counts, does it only hide columns, the step's output if it has been made, a question still open).

        An additive mask of zeros (HuggingFace's eager mask of an unpadded decode step) adds nothing anywhere and is left out;
        one that only hides columns has a faster way. Which it is, is established once per mask tensor, i.e. once per forward
        pass, not per layer, and the first layer does not wait for the answer with nothing under way: a decode step's mask is
        taken to be like the session's last step's, the step is launched and the answer read; a step launched on a wrong guess is
        launched again (what it adds to the caches does not depend on the mask). A mask of several queries, all but always
        nonzero, is taken as it is, which is right whatever it holds."""
        am = attention_mask
        facts = self._mask_facts
        flags = facts.known(am)  # (of the layers behind the first, the usual call)
        shape = am.shape
        if (len(shape) != 4 or shape[3] < keys.shape[2]
                or flags is None and am.dtype not in (torch.float32, torch.bfloat16, torch.float16)):
            return am, False, None, None
        same_type = am.dtype == queries.dtype  # (a lowest value of another type is none of the queries')
        if flags is None:
            guess = facts.guess(shape[2] == 1, sparse_meta_data)
            question = MaskQuestion(am)
            q_shape = queries.shape
            # (a mask that does not cover the call has to be zero, or is refused)
            covers = shape[2] == q_shape[2] and shape[0] in (1, q_shape[0]) and shape[1] in (1, q_shape[1])
            if plannable and covers and guess is not None and (guess == 0 or q_shape[2] == 1):
                hides = not guess & _native.AMASK_GENERAL and same_type
                out, error = None, None
                try:
                    out = self._plan_step(queries, keys, values, am if guess else None, scaling, sparse_meta_data, layer_idx, hides,
                                          guessed=True)
                except Exception as e:
                    error = e
                flags = facts.take(question, sparse_meta_data)
                # the error of a right guess is the call's own (memory may have been short for buffers that only a guess needs)
                if error is not None and flags == guess and not isinstance(error, torch.OutOfMemoryError):
                    raise error
                error = None
                if out is not None and (flags == guess or (guess and not (hides and flags & _native.AMASK_GENERAL))):
                    return am, hides, out, None
            elif shape[2] > 1 and guess != 0 and covers:
                return am, False, None, question
            else:
                flags = facts.take(question, sparse_meta_data)
        if flags == 0:
            return None, False, None, None
        return am, not flags & _native.AMASK_GENERAL and same_type, None, None

    def _plan_step(self, queries: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, attention_mask: Optional[torch.Tensor],
                   scaling: float, sparse_meta_data: Dict[Any, Any], layer_idx: Optional[int], only_hides: bool,
                   guessed: bool = False) -> Optional[torch.Tensor]:
        """One step through the cached plan of its geometry, or None where the plan does not cover it. `guessed`: launched as if
        its mask were zero, or only hid columns, before the answer is there."""
        _native.require_device(queries, "queries")
        masked = attention_mask is not None
        # A masked step's buffers belong to the stream and thread of their plan, as those of the masker-by-masker path
        # belong to the call: a step on another stream is not ordered with the ones that use them. So do those of a step whose
        # mask is guessed to be zero: it may turn out to be a masked one. A captured step's belong to its graph alone: what its
        # plan clears is clear when the graph runs, not now; and its mask is what the buffer holds then, which may be anything.
        device = queries.device
        stream = _native.stream_ptr(device)
        owner = (stream, threading.get_ident()) if masked or guessed else None
        capturing = torch.cuda.is_current_stream_capturing() if masked else None
        if capturing:
            plan, only_hides = DecodePlan(self.maskers, self._plan_kind, queries, keys, True), False
        else:
            key = (device, queries.dtype, queries.shape, keys.shape[1], masked, None if masked else owner)
            plan = self._plans.get(key)
            if plan is None or plan.owner != owner:
                if guessed and not masked:
                    guesses = [k for k, p in list(self._plans.items()) if p.owner is not None and not p.masked]
                    if len(guesses) >= _GUESSED_PLANS:
                        self._plans.pop(guesses[0], None)
                plan = self._plans[key] = DecodePlan(self.maskers, self._plan_kind, queries, keys, masked, owner)
        return plan.run(queries, keys, values, scaling, sparse_meta_data, layer_idx, attention_mask, only_hides, guessed, capturing, stream)

    @classmethod
    def create_from_config(cls, config: SparseAttentionConfig) -> "ResearchAttention":
        if not isinstance(config, ResearchAttentionConfig):
            raise TypeError(f"Expected ResearchAttentionConfig, got {type(config)}")
        maskers = [ResearchMasker.create_masker_from_config(c) for c in config.masker_configs]
        return cls(config, maskers)


class _EmptyRowsMask(Mask):
    """An empty mask that already owns row buffers sized for the chain: it reports
    is_empty (so consumers treat it as "no masking") until a masker fills the rows."""

    def __init__(self, shape, rows: NativeRows, dtype: torch.dtype):
        super().__init__(shape=shape, dtype=dtype, device=rows.device, is_empty=True)
        self._planned_rows = rows

    def to_rows(self, extra: int = 0, weighted: Optional[bool] = None) -> NativeRows:
        rows = self._planned_rows
        rows.reserve(extra)
        if weighted:
            rows.zero_if_fresh()
            rows.make_weighted()
        return rows
