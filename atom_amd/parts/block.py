"""The pre-norm residual block: norm, mixer, norm, feed-forward, with the residual sum
folded into the norm that follows it (atom/models/qwen3.py:240-258): the block hands
on its feed-forward output and the residual stream, and the next norm adds them."""

from __future__ import annotations

import torch

from .base import BLOCKS, FEED_FORWARDS, MIXERS, NORMS, Block, ParamSpec, PartChoice, PendingPost, PendingSum, ScaledSum, StreamUpdate


class PreNormBlock(Block):
    def __init__(self, mixer: PartChoice, feed_forward: PartChoice | None, norm: PartChoice, prefix: str = "",
                 names: dict[str, str] | None = None):
        super().__init__(prefix)
        n = {"mixer_norm": "input_layernorm", "mixer": "self_attn", "ffn_norm": "post_attention_layernorm",
             "ffn": "mlp", **(names or {})}
        sub = lambda name: f"{prefix}.{n[name]}" if prefix else n[name]  # noqa: E731
        self.mixer_norm = norm.build(NORMS, prefix=sub("mixer_norm"))
        self._mixer = mixer.build(MIXERS, prefix=sub("mixer"))
        # ``feed_forward`` None: the layer is its mixer alone, and hands on the mixer's output
        self.ffn = feed_forward.build(FEED_FORWARDS, prefix=sub("ffn")) if feed_forward is not None else None
        self.ffn_norm = norm.build(NORMS, prefix=sub("ffn_norm")) if self.ffn is not None else None

    @property
    def mixer(self):
        return self._mixer

    def children(self):
        return [self.mixer_norm, self._mixer] + ([self.ffn_norm, self.ffn] if self.ffn is not None else [])

    def forward(self, ctx, hidden, residual, cache):
        if not self.mixer_norm.accepts_deferred:
            hidden = ctx.ops.materialize(hidden)
        hidden, residual = self.mixer_norm.forward_residual(ctx, hidden, residual)
        if not self._mixer.accepts_deferred:
            hidden = ctx.ops.materialize(hidden)
        hidden = self._mixer.forward(ctx, hidden, cache)
        if self.ffn is None:
            return hidden, residual
        if not self.ffn_norm.accepts_deferred:
            hidden = ctx.ops.materialize(hidden)
        hidden, residual = self.ffn_norm.forward_residual(ctx, hidden, residual)
        if not self.ffn.accepts_deferred:
            hidden = ctx.ops.materialize(hidden)
        hidden = self.ffn.forward(ctx, hidden)
        return hidden, residual


class SandwichBlock(Block):
    """Norms before and after each sublayer: ``x += post1(mixer(pre1(x)))``, then ``x += post2(ffn(pre2(x)))``;
    ``feed_forward`` None leaves the second sublayer out.  As in the pre-norm block, the block hands on its last
    summand (not yet added) beside the stream, and the norm that follows adds it.  The sum of a sublayer's normed output
    and the norm before the next sublayer are one kernel where the norm offers ``forward_post``: within the block, and from
    one block to the next through a ``PendingPost`` (two kernels of 5.0 and 4.0 us in a step of 4 rows of 2,048, one of
    4.1 so)."""

    accepts_pending = (PendingPost,)

    def __init__(self, mixer: PartChoice, feed_forward: PartChoice | None, norm: PartChoice, prefix: str = "",
                 names: dict[str, str] | None = None):
        super().__init__(prefix)
        n = {"mixer_pre": "norm1", "mixer": "mix", "mixer_post": "norm1b", "ffn_pre": "norm2", "ffn": "mlp",
             "ffn_post": "norm2b", **(names or {})}
        sub = lambda name: f"{prefix}.{n[name]}" if prefix else n[name]  # noqa: E731
        self.mixer_pre = norm.build(NORMS, prefix=sub("mixer_pre"))
        self._mixer = mixer.build(MIXERS, prefix=sub("mixer"))
        self.mixer_post = norm.build(NORMS, prefix=sub("mixer_post"))
        self.ffn = feed_forward.build(FEED_FORWARDS, prefix=sub("ffn")) if feed_forward is not None else None
        self.ffn_pre = norm.build(NORMS, prefix=sub("ffn_pre")) if self.ffn is not None else None
        self.ffn_post = norm.build(NORMS, prefix=sub("ffn_post")) if self.ffn is not None else None

    @property
    def mixer(self):
        return self._mixer

    def children(self):
        parts = [self.mixer_pre, self._mixer, self.mixer_post]
        if self.ffn is not None:
            parts += [self.ffn_pre, self.ffn, self.ffn_post]
        return parts

    def forward(self, ctx, hidden, residual, cache):
        ops = ctx.ops
        if (isinstance(hidden, PendingPost) and residual is not None and type(self.mixer_pre) is type(hidden.norm)
                and hidden.norm.eps == self.mixer_pre.eps):
            hidden = hidden.norm.forward_post(ctx, hidden.x, residual, self.mixer_pre)
        else:
            if isinstance(hidden, PendingPost):
                hidden = hidden.resolve(ctx)
            if not self.mixer_pre.accepts_deferred:
                hidden = ops.materialize(hidden)
            hidden, residual = self.mixer_pre.forward_residual(ctx, hidden, residual)
        if not self._mixer.accepts_deferred:
            hidden = ops.materialize(hidden)
        mixed = ops.materialize(self._mixer.forward(ctx, hidden, cache))
        if self.ffn is None:
            return self.mixer_post.forward(ctx, mixed, out_dtype=torch.float32), residual
        post = getattr(self.mixer_post, "forward_post", None)
        if post is not None:
            hidden = post(ctx, mixed, residual, self.ffn_pre)
        else:
            hidden, residual = self.ffn_pre.forward_residual(ctx, self.mixer_post.forward(ctx, mixed), residual)
        if not self.ffn.accepts_deferred:
            hidden = ops.materialize(hidden)
        out = ops.materialize(self.ffn.forward(ctx, hidden))
        if post is not None:
            return PendingPost(out, self.ffn_post), residual
        return self.ffn_post.forward(ctx, out, out_dtype=torch.float32), residual


class PostNormBlock(Block):
    """Norms on the sublayers' outputs only: ``x += norm1(mixer(x))``, then ``x += norm2(ffn(x))``
    (``feed_forward`` None leaves it out), then, where the layer has one, a ``side`` part (kind from the
    FEED_FORWARDS registry) that is handed the stream and adds to it itself.  The sublayers read the stream, which
    is float32; the block keeps it whole (nothing pending) and hands it on as ``hidden`` with no residual.  A
    copy of the stream in the step's type, for the products that read it, comes out of the kernel that adds to
    it."""

    def __init__(self, mixer: PartChoice, feed_forward: PartChoice | None, norm: PartChoice,
                 side: PartChoice | None = None, prefix: str = "", names: dict[str, str] | None = None):
        super().__init__(prefix)
        n = {"mixer": "mix", "mixer_post": "norm1", "ffn": "mlp", "ffn_post": "norm2", "side": "side", **(names or {})}
        sub = lambda name: f"{prefix}.{n[name]}" if prefix else n[name]  # noqa: E731
        self._mixer = mixer.build(MIXERS, prefix=sub("mixer"))
        self.mixer_post = norm.build(NORMS, prefix=sub("mixer_post"))
        self.ffn = feed_forward.build(FEED_FORWARDS, prefix=sub("ffn")) if feed_forward is not None else None
        self.ffn_post = norm.build(NORMS, prefix=sub("ffn_post")) if self.ffn is not None else None
        self.side = side.build(FEED_FORWARDS, prefix=sub("side")) if side is not None else None
        for post in (self.mixer_post, self.ffn_post):
            if post is not None and not hasattr(post, "forward_post"):
                raise ValueError(f"{type(post).__name__} cannot add its output to the stream (no forward_post)")

    @property
    def mixer(self):
        return self._mixer

    def children(self):
        parts = [self._mixer, self.mixer_post]
        if self.ffn is not None:
            parts += [self.ffn, self.ffn_post]
        if self.side is not None:
            parts.append(self.side)
        return parts

    def forward(self, ctx, hidden, residual, cache):
        ops = ctx.ops
        if residual is not None:
            raise ValueError("this block takes the whole stream, with nothing pending beside it")
        stream = ops.materialize(hidden)
        if stream.dtype != torch.float32:
            raise ValueError("this block keeps a float32 stream: the embedding before it must write float32")
        # the stream in the step's type, as the products read it: left by the block before this one, or made now
        reads = ctx.memo.pop(("stream copy", stream.data_ptr()), None)
        if reads is None:
            reads = stream if ctx.dtype == torch.float32 else ops.cast_rows(stream, ctx.dtype)
        mixed = ops.materialize(self._mixer.forward(ctx, reads, cache))
        reads = self.mixer_post.forward_post(ctx, mixed, stream)
        if self.ffn is not None:
            out = ops.materialize(self.ffn.forward(ctx, reads))
            reads = self.ffn_post.forward_post(ctx, out, stream)
        if self.side is not None:
            reads = self.side.forward_stream(ctx, reads, stream)
        ctx.memo[("stream copy", stream.data_ptr())] = reads
        return stream, None


class NormedSumBlock(Block):
    """The norm comes after the sum and its result is the stream: ``x <- norm1(alpha x + mixer(x))``, then
    ``x <- norm2(alpha x + ffn(x))`` (``feed_forward`` None leaves the second step out).  The sublayers read the
    stream, which is float32 and kept whole (nothing pending); its rows in the step's type, for the products that
    read them, come out of the kernel that norms it.  A mixer with ``reads_stream`` is handed the float32 rows.
    ``names["mixer"]`` may be empty: the mixer then takes the layer's own prefix.  A checkpoint that holds the second
    norm's weight for a layer without feed-forward gets the second step with nothing added: ``x <- norm2(alpha x)``.
    In steps of single tokens the last norm may be left to the next block (a ``PendingSum``), whose mixer can take the sum
    and the norm into its own first kernel (``forward_pending``)."""

    accepts_pending = (PendingSum,)

    def __init__(self, mixer: PartChoice, feed_forward: PartChoice | None, norm: PartChoice, alpha: float = 1.0,
                 prefix: str = "", names: dict[str, str] | None = None):
        super().__init__(prefix)
        n = {"mixer": "mix", "mixer_norm": "norm1", "ffn": "mlp", "ffn_norm": "norm2", **(names or {})}
        sub = lambda name: (f"{prefix}.{n[name]}" if prefix else n[name]) if n[name] else prefix  # noqa: E731
        self._norm_choice, self._ffn_norm_prefix, self._ffn_norm_name = norm, sub("ffn_norm"), n["ffn_norm"]
        self.alpha = float(alpha)
        self._mixer = mixer.build(MIXERS, prefix=sub("mixer"))
        self.mixer_norm = norm.build(NORMS, prefix=sub("mixer_norm"))
        self.ffn = feed_forward.build(FEED_FORWARDS, prefix=sub("ffn")) if feed_forward is not None else None
        self.ffn_norm = norm.build(NORMS, prefix=sub("ffn_norm")) if self.ffn is not None else None
        for post in (self.mixer_norm, self.ffn_norm):
            if post is not None and not hasattr(post, "forward_sum"):
                raise ValueError(f"{type(post).__name__} cannot norm a sum into the stream (no forward_sum)")

    @property
    def mixer(self):
        return self._mixer

    def children(self):
        return ([self._mixer, self.mixer_norm] + ([self.ffn] if self.ffn is not None else [])
                + ([self.ffn_norm] if self.ffn_norm is not None else []))

    def adopt_shapes(self, shape_of):
        named = shape_of(self._ffn_norm_name) is not None or shape_of(f"{self._ffn_norm_name}.weight") is not None
        if self.ffn is None and self.ffn_norm is None and named:
            self.ffn_norm = self._norm_choice.build(NORMS, prefix=self._ffn_norm_prefix)

    @staticmethod
    def _summands(ops, y):
        if isinstance(y, ScaledSum):
            return [ops.materialize(t) for t in y.terms], y.scales
        return [ops.materialize(y)], [1.0]

    def forward(self, ctx, hidden, residual, cache):
        ops = ctx.ops
        if residual is not None:
            raise ValueError("this block takes the whole stream, with nothing pending beside it")
        mixed = None
        if isinstance(hidden, PendingSum):
            stream, ahead = hidden.stream, getattr(self._mixer, "forward_pending", None)
            mixed = ahead(ctx, hidden, cache) if ahead is not None else None
            if mixed is None:
                hidden.resolve(ctx)
        else:
            stream = ops.materialize(hidden)
        if stream.dtype != torch.float32:
            raise ValueError("this block keeps a float32 stream: the embedding before it must write float32")
        if mixed is None:
            reads = ctx.memo.pop(("stream copy", stream.data_ptr()), None)
            if self._mixer.reads_stream:
                reads = stream
            elif reads is None:
                reads = stream if ctx.dtype == torch.float32 else ops.cast_rows(stream, ctx.dtype)
            mixed = self._mixer.forward(ctx, reads, cache)
        terms, scales = self._summands(ops, mixed)
        # the copy is for the feed-forward, or for the next block's mixer where that reads one
        reads = self.mixer_norm.forward_sum(ctx, terms, scales, stream, self.alpha,
                                            copy=self.ffn is not None or not self._mixer.reads_stream)
        if self.ffn is not None:
            terms, scales = self._summands(ops, self.ffn.forward(ctx, reads))
            if ctx.max_q_len == 1 and hasattr(self._mixer, "forward_pending") and hasattr(ops, "sum_norm_shift"):
                return PendingSum(stream, self.alpha, terms, scales, self.ffn_norm, not self._mixer.reads_stream), None
            reads = self.ffn_norm.forward_sum(ctx, terms, scales, stream, self.alpha, copy=not self._mixer.reads_stream)
        elif self.ffn_norm is not None:
            reads = self.ffn_norm.forward_sum(ctx, [], [], stream, self.alpha, copy=not self._mixer.reads_stream)
        if reads is not stream:
            ctx.memo[("stream copy", stream.data_ptr())] = reads
        return stream, None


class StreamsBlock(Block):
    """Pre-norm sublayers over a residual of ``streams`` float32 streams side by side.  Sublayer q (1: mixer, 2:
    feed-forward; ``feed_forward`` None leaves it out) reads the norm of ``u = sum_s in_q[s] x_s``, and its result y, times
    a scale per entry where ``layer_scale`` is set, joins them: ``x_t <- sum_s mix_q[s, t] x_s + out_q[t] y`` (the matrix
    is indexed [from, to]).  The block hands on its last sublayer's ``StreamUpdate`` beside the streams, and the norm that
    follows applies it.  All streams start as the rows of the embedding."""

    def __init__(self, mixer: PartChoice, feed_forward: PartChoice | None, norm: PartChoice, streams: int,
                 layer_scale: bool = True, prefix: str = "", names: dict[str, str] | None = None):
        super().__init__(prefix)
        n = {"mixer": "mix", "mixer_norm": "norm1", "mixer_scale": "ls1", "mixer_streams": "hc1", "ffn": "mlp",
             "ffn_norm": "norm2", "ffn_scale": "ls2", "ffn_streams": "hc2", "in": "in", "out": "out", "mix": "mix",
             **(names or {})}
        sub = lambda name: f"{prefix}.{n[name]}" if prefix else n[name]  # noqa: E731
        if streams < 1:
            raise ValueError("a residual has at least one stream")
        self.names, self.streams, self.layer_scale = n, int(streams), bool(layer_scale)
        self._mixer = mixer.build(MIXERS, prefix=sub("mixer"))
        self.mixer_norm = norm.build(NORMS, prefix=sub("mixer_norm"))
        self.ffn = feed_forward.build(FEED_FORWARDS, prefix=sub("ffn")) if feed_forward is not None else None
        self.ffn_norm = norm.build(NORMS, prefix=sub("ffn_norm")) if self.ffn is not None else None
        self.size = self.mixer_norm.size
        if not hasattr(self.mixer_norm, "forward_streams"):
            raise ValueError(f"{type(self.mixer_norm).__name__} cannot norm a sum of streams (no forward_streams)")

    @property
    def mixer(self):
        return self._mixer

    def children(self):
        return [self._mixer, self.mixer_norm] + ([self.ffn, self.ffn_norm] if self.ffn is not None else [])

    def param_specs(self):
        n, S, specs = self.names, self.streams, {}
        for q in ("mixer",) + (("ffn",) if self.ffn is not None else ()):
            hc = n[f"{q}_streams"]
            specs[f"{q}.in"] = ParamSpec.single(f"{hc}.{n['in']}", (S,), kind="vector", init="one_plus_normal")
            specs[f"{q}.out"] = ParamSpec.single(f"{hc}.{n['out']}", (S,), kind="vector", init="one_plus_normal")
            specs[f"{q}.mix"] = ParamSpec.single(f"{hc}.{n['mix']}", (S, S), kind="vector")
            if self.layer_scale:
                specs[f"{q}.scale"] = ParamSpec.single(n[f"{q}_scale"], (self.size,), kind="vector", init="one_plus_normal")
        return specs

    def _sublayer(self, ctx, q, norm, run, accepts_deferred, hidden, streams):
        x, streams = norm.forward_streams(ctx, hidden, streams, self.params[f"{q}.in"], self.streams)
        y = run(x if accepts_deferred else ctx.ops.materialize(x))
        return StreamUpdate(y, self.p(f"{q}.scale"), self.params[f"{q}.out"], self.params[f"{q}.mix"]), streams

    def forward(self, ctx, hidden, residual, cache):
        hidden, residual = self._sublayer(ctx, "mixer", self.mixer_norm, lambda x: self._mixer.forward(ctx, x, cache),
                                          self._mixer.accepts_deferred, hidden, residual)
        if self.ffn is not None:
            hidden, residual = self._sublayer(ctx, "ffn", self.ffn_norm, lambda x: self.ffn.forward(ctx, x),
                                              self.ffn.accepts_deferred, hidden, residual)
        return hidden, residual


BLOCKS.register("streams", StreamsBlock)
BLOCKS.register("prenorm", PreNormBlock)
BLOCKS.register("normed_sum", NormedSumBlock)
BLOCKS.register("sandwich", SandwichBlock)
BLOCKS.register("postnorm", PostNormBlock)
