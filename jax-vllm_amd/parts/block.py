"""Pre-norm residual arrangement of one layer.  Reference: ``jllm/model/common.py:140-147``:

    h = h + mixer(norm_1(h));   h = h + feed_forward(norm_2(h))

(the norm part is a parameter: an RMS norm or a layer norm).  The residual stream ``h`` is float.  Each sublayer's output is not added at once:
it is handed on as ``delta`` and added inside the next norm's kernel (one pass over
``h`` instead of two), so a block takes and returns ``(h, delta)``.

With ``residual_scale`` m every sublayer's output joins the stream times that constant,
``h = h + m * mixer(norm_1(h))``: the output travels as a ``K.PendingNorm`` without a weight and
the next norm's kernel multiplies in float while it adds.  ``has_feed_forward`` False: the
first line only.
"""
from __future__ import annotations

import torch

from ..ops import kernels as K
from .spec import BLOCK_STATE, PartSpec, StateSpec, TensorSpec, build_part, is_replayable, register_part


# Up to this width one or two rows go from product to product as parts; wider ones, whose splits a launch merges in any case, through the stream.  Microseconds a
# layer by parts / through the stream, one row and two: 2,560 with 9,728 columns in the feed-forward 64.1 / 60.3, 64.1 / 61.3, 4,096 with 12,288 88.4 / 87.9, 90.4 / 88.5.  At
# 2,048 it hangs on the feed-forward: 3,072 33.1 / 32.9, 35.5 / 33.3, 8,192 45.6 / 44.9, 47.7 / 45.5, but 12,288 54.0 / 56.6, 56.3 / 57.3.  (3,072 and 3,584, and
# widths below 2,048 with these head counts, have no form by parts that both sublayers take.)
MADE_WIDTH = 2048


class PreNormBlock:
    def __init__(self, norm: PartSpec, mixer_norm_name: str = "input_layernorm",
                 feed_forward_norm_name: str = "post_attention_layernorm", residual_scale: float = 1.0,
                 has_feed_forward: bool = True):
        self.has_feed_forward = bool(has_feed_forward)
        self.residual_scale = float(residual_scale)
        self.mixer_norm = build_part("norm", norm)
        self.feed_forward_norm = build_part("norm", norm) if self.has_feed_forward else None
        self.names = (mixer_norm_name, feed_forward_norm_name) if self.has_feed_forward else (mixer_norm_name,)
        self.norms = (self.mixer_norm, self.feed_forward_norm) if self.has_feed_forward else (self.mixer_norm,)

    @property
    def replayable(self) -> bool:
        return all(is_replayable(n) for n in self.norms)

    def tensors(self) -> dict:
        out = {}
        for name, part in zip(self.names, self.norms):
            for k, v in part.tensors().items():
                out[f"{name}.{k}"] = v
        return out

    def bind(self, tensors: dict, dtype: torch.dtype) -> None:
        for name, part in zip(self.names, self.norms):
            part.bind({k[len(name) + 1:]: v for k, v in tensors.items() if k.startswith(name + ".")}, dtype)

    def _share(self, out):
        """What a sublayer returned, as the next norm takes it."""
        if isinstance(out, K.PendingPair):                             # two outputs under norms of their own
            if self.residual_scale != 1.0:
                raise ValueError("a residual constant on a pair of normed outputs belongs into their norms' weights")
            return out
        if self.residual_scale != 1.0 or isinstance(out, tuple):       # a pair (rows, float shares) is added there too
            return K.pending_scale(out, self.residual_scale)
        return out.settled() if isinstance(out, K.BiasedOutput) else out

    def _made_by_readers(self, h, delta, mixer, feed_forward, ctx, mem) -> bool:
        """Whether the products behind both norms make their rows themselves (one or two rows of a decode step): both or neither, as the stream
        goes to a second buffer and back."""
        n = h.shape[0]
        if n > K.MADE_MAX_ROWS or not self.has_feed_forward or self.residual_scale != 1.0 or not all(hasattr(p, "pending") for p in self.norms):
            return False
        if delta is not None and not _float_parts(delta):
            return False
        ask = [getattr(p, "takes_pending_rows", None) for p in (mixer, feed_forward)]
        return all(a is not None for a in ask) and ask[0](n, ctx, mem) and ask[1](n)

    takes_products = True      # ``forward`` takes a ``K.PendingProduct`` as ``delta``

    def _through_stream(self, n: int, mixer, feed_forward) -> bool:
        """Whether both sublayers' last products join the stream in their own launch (few rows of a step): their first products read
        ``K.StreamRows``."""
        return (self.has_feed_forward and self.residual_scale == 1.0 and all(hasattr(p, "into_stream") for p in self.norms)
                and all(hasattr(p, "leaves_product") and p.leaves_product(n) and p.takes_stream_rows(n) for p in (mixer, feed_forward)))

    def forward(self, h, delta, mixer, feed_forward, ctx, mem):
        n = h.shape[0]
        # one or two rows of narrow models are made by the products that read them, which then merge the attention's splits too
        narrow = n <= K.MADE_MAX_ROWS and h.shape[1] <= MADE_WIDTH and not isinstance(delta, K.PendingProduct) and self._made_by_readers(h, delta, mixer, feed_forward, ctx, mem)
        if n <= K.SKINNY_AUTO_ROWS and not narrow and self._through_stream(n, mixer, feed_forward):
            x = self.mixer_norm.into_stream(h, delta) if isinstance(delta, K.PendingProduct) else _add_norm(self.mixer_norm, h, delta, mixer, n)
            y = self.feed_forward_norm.into_stream(h, mixer.forward(x, ctx, mem, leave_product=True))
            return feed_forward.forward(y, ctx, leave_product=True)
        if isinstance(delta, K.PendingProduct):
            delta = delta.linear()
        if narrow or n <= K.MADE_MAX_ROWS and self._made_by_readers(h, delta, mixer, feed_forward, ctx, mem):
            between = torch.empty_like(h)                              # the stream between the two sublayers: a product's blocks all read the old one
            a = self._share(mixer.forward(self.mixer_norm.pending(h, delta, between), ctx, mem))
            if _float_parts(a):
                return self._share(feed_forward.forward(self.feed_forward_norm.pending(between, a, h), ctx))
            y = _add_norm(self.feed_forward_norm, between, a, feed_forward, n)
            h.copy_(between)
            return self._share(feed_forward.forward(y, ctx))
        x = _add_norm(self.mixer_norm, h, delta, mixer, n)
        a = self._share(mixer.forward(x, ctx, mem))
        if not self.has_feed_forward:
            return a
        y = _add_norm(self.feed_forward_norm, h, a, feed_forward, n)
        return self._share(feed_forward.forward(y, ctx))


def _float_parts(delta) -> bool:
    """Whether a sublayer's output is a stack of at most four float partial products."""
    return isinstance(delta, torch.Tensor) and delta.dim() == 3 and delta.dtype == torch.float32 and delta.shape[0] <= 4


def _add_norm(norm, h, delta, reader, n_rows: int):
    """``norm.add_norm(h, delta)``.  Only where both sides have said so, the norm may hand on
    ``K.UnscaledRows``: a norm part declares ``may_leave_scale = True`` (its ``add_norm`` takes
    ``unscaled_ok``), a reader part answers ``takes_unscaled_rows(rows)``.  Parts that declare
    neither see the plain interface."""
    ask = getattr(reader, "takes_unscaled_rows", None)
    if (getattr(norm, "may_leave_scale", False) and ask is not None and not isinstance(delta, K.PendingNorm)
            and ask(n_rows)):
        return norm.add_norm(h, delta, unscaled_ok=True)
    if n_rows > 32 and getattr(norm, "dtype", None) == torch.float32 and getattr(norm, "may_leave_terms", False) and not isinstance(delta, K.PendingNorm):
        ask = getattr(reader, "takes_terms", None)
        layout = ask(n_rows) if ask is not None else None
        if layout is not None:
            return norm.add_norm(h, delta, terms=layout)
    return norm.add_norm(h, delta)


class SandwichBlock:
    """Every sublayer between two norms:

        h = h + norm_1b(mixer(norm_1(h)));   h = h + norm_2b(feed_forward(norm_2(h)))

    (the second line only for a layer that has a feed-forward).  A sublayer's output is handed on as a
    ``K.PendingNorm`` (the output and the norm weight that belongs to it): the next norm's kernel norms it,
    adds it to the stream and norms the stream in one pass, also across the border of two layers and
    before the head.

    With ``input_taps`` what a sublayer reads is its normed input plus a causal filter of it over time per channel,
    u + F(u), F(u)_t = sum_j w[:, j] u_(t - taps + 1 + j) (zeros before the sequence's start): the last taps - 1 inputs
    are state of the block's own, in the request's slot.  A step of one token a request filters in the norm's kernel."""

    def __init__(self, norm: PartSpec, has_feed_forward: bool = True,
                 names=("norm1", "norm1b", "norm2", "norm2b"), input_taps: int | None = None, hidden_size: int | None = None,
                 filter_names=("canon1", "canon2")):
        self.has_feed_forward = bool(has_feed_forward)
        self.names = tuple(names) if self.has_feed_forward else tuple(names[:2])
        self.norms = [build_part("norm", norm) for _ in self.names]
        self.taps = int(input_taps) if input_taps else 0
        self.hidden_size = int(hidden_size) if hidden_size else None
        if self.taps and not self.hidden_size:
            raise ValueError("a filter on the sublayers' inputs needs the width")
        self.filter_names = tuple(filter_names[:2 if self.has_feed_forward else 1]) if self.taps else ()

    @property
    def replayable(self) -> bool:
        return all(is_replayable(n) for n in self.norms)

    def tensors(self) -> dict:
        out = {}
        for name, part in zip(self.names, self.norms):
            for k, v in part.tensors().items():
                out[f"{name}.{k}"] = v
        for name in self.filter_names:
            out[f"{name}.weight"] = TensorSpec((self.hidden_size, self.taps), role="vector", init="small")
        return out

    def state_spec(self):
        return tuple(StateSpec((self.taps - 1, self.hidden_size), "float32", name) for name in self.filter_names) or None

    def bind(self, tensors: dict, dtype: torch.dtype) -> None:
        for name, part in zip(self.names, self.norms):
            part.bind({k[len(name) + 1:]: v for k, v in tensors.items() if k.startswith(name + ".")}, dtype)
        self.dtype = dtype
        self.filters = [tensors[f"{name}.weight"].t().contiguous() for name in self.filter_names]     # [taps, width]

    def _input(self, i: int, h, delta, ctx, mem):
        """What sublayer i reads; ``h`` takes what ``delta`` still owes the stream."""
        norm = self.norms[2 * i]
        if not self.taps:
            return norm.add_norm(h, delta)
        state = mem.states[BLOCK_STATE + self.filter_names[i]]
        if (ctx.decode_only and K.norm_filter_possible(self.hidden_size)
                and (delta is None or isinstance(delta, K.PendingNorm) and delta.weight is not None and delta.bias is None)):
            return K.norm_filter(h, delta, norm.weight, norm.eps, self.filters[i], state, ctx.slot_ids, self.dtype)
        return K.token_filter(norm.add_norm(h, delta), self.filters[i], state, ctx.slot_ids, ctx.cu_seqlens, ctx.max_q_len)

    def forward(self, h, delta, mixer, feed_forward, ctx, mem):
        x = self._input(0, h, delta, ctx, mem)
        a = mixer.forward(x, ctx, mem)
        pending = K.pending_norm(a, self.norms[1].weight, self.norms[1].eps)
        if not self.has_feed_forward:
            return pending
        y = self._input(1, h, pending, ctx, mem)
        f = feed_forward.forward(y, ctx)
        return K.pending_norm(f, self.norms[3].weight, self.norms[3].eps)


class OutputNormBlock:
    """A norm on every sublayer's OUTPUT only; the sublayers read the stream itself:

        h = h + norm_1(mixer(h));   h = h + norm_2(feed_forward(h))

    (the second line only for a layer that has a feed-forward; a constant factor on the sublayer's share is the
    norm part's ``gain``).  A sublayer's output is handed on as a ``K.PendingNorm``; the kernel that norms it and adds
    it to the float stream also hands the next reader the stream in the activation type."""

    def __init__(self, norm: PartSpec, has_feed_forward: bool = True, names=("norm1", "norm2")):
        self.has_feed_forward = bool(has_feed_forward)
        self.names = tuple(names) if self.has_feed_forward else tuple(names[:1])
        self.norms = [build_part("norm", norm) for _ in self.names]

    @property
    def replayable(self) -> bool:
        return all(is_replayable(n) for n in self.norms)

    def tensors(self) -> dict:
        out = {}
        for name, part in zip(self.names, self.norms):
            for k, v in part.tensors().items():
                out[f"{name}.{k}"] = v
        return out

    def bind(self, tensors: dict, dtype: torch.dtype) -> None:
        self.dtype = dtype
        for name, part in zip(self.names, self.norms):
            part.bind({k[len(name) + 1:]: v for k, v in tensors.items() if k.startswith(name + ".")}, dtype)

    def _stream(self, h, delta):
        """h += (what ``delta`` still owes the stream); returns h in the activation type."""
        from ..ops import kernels as K

        if delta is None:
            return K.cast_rows(h, self.dtype)
        if not isinstance(delta, K.PendingNorm):
            raise TypeError("this arrangement follows layers that hand on a sublayer's output with its norm")
        out = torch.empty(h.shape, dtype=self.dtype, device=h.device)
        K.postnorm_add_rmsnorm(h, delta.y, delta.parts, delta.weight, delta.eps, None, out, bias=delta.bias,
                               plain_scale=delta.scale)
        return out

    def forward(self, h, delta, mixer, feed_forward, ctx, mem):
        from ..ops import kernels as K

        a = mixer.forward(self._stream(h, delta), ctx, mem)
        pending = K.pending_norm(a, self.norms[0].weight, self.norms[0].eps)
        if not self.has_feed_forward:
            return pending
        f = feed_forward.forward(self._stream(h, pending), ctx)
        return K.pending_norm(f, self.norms[1].weight, self.norms[1].eps)


class ParallelBlock:
    """One norm whose output both sublayers read, their outputs joining the stream together, and an optional
    per-layer token input behind them (``parts/token_input.py``):

        u = norm_1(h);   h = h + (mixer(u) + feed_forward(u));   h = h + norm_t(token_input(h))

    (the feed-forward and the token input are optional).  The sublayers' outputs are added to the float stream by
    one kernel that also hands the token input the stream in the activation type; the token input's output is
    handed on as a ``K.PendingNorm`` with its own norm weight (a plain RMS norm), so the next layer's norm (or the
    final one) does both norms and the residual step in one pass."""

    def __init__(self, norm: PartSpec, has_feed_forward: bool = True, token_input: PartSpec | None = None,
                 norm_name: str = "norm1", token_input_prefix: str = "side."):
        self.has_feed_forward = bool(has_feed_forward)
        self.norm = build_part("norm", norm)
        self.norm_name, self.token_prefix = norm_name, token_input_prefix
        self.token_input = build_part("token_input", token_input) if token_input is not None else None

    @property
    def replayable(self) -> bool:
        return is_replayable(self.norm) and (self.token_input is None or is_replayable(self.token_input))

    def tensors(self) -> dict:
        out = {f"{self.norm_name}.{k}": v for k, v in self.norm.tensors().items()}
        if self.token_input is not None:
            out.update({self.token_prefix + k: v for k, v in self.token_input.tensors().items()})
        return out

    def bind(self, tensors: dict, dtype: torch.dtype) -> None:
        self.dtype = dtype
        name = self.norm_name + "."
        self.norm.bind({k[len(name):]: v for k, v in tensors.items() if k.startswith(name)}, dtype)
        if self.token_input is not None:
            p = self.token_prefix
            self.token_input.bind({k[len(p):]: v for k, v in tensors.items() if k.startswith(p)}, dtype)

    def forward(self, h, delta, mixer, feed_forward, ctx, mem):
        u = self.norm.add_norm(h, delta)
        a = mixer.forward(u, ctx, mem)
        f = feed_forward.forward(u, ctx) if self.has_feed_forward else None
        if self.token_input is None:
            K.add_outputs(h, a, f)
            return None
        x = K.add_outputs(h, a, f, out_dtype=self.dtype)
        y = self.token_input.forward(x, ctx)
        return K.pending_norm(y, self.token_input.norm_weight, self.token_input.eps)


register_part("block", "prenorm", PreNormBlock)
register_part("block", "parallel", ParallelBlock)
register_part("block", "output_norm", OutputNormBlock)
register_part("block", "sandwich", SandwichBlock)
