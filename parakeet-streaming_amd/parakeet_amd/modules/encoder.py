"""Drop-in for the streaming parts of ``parakeet.modules.encoder``
(parakeet/modules/encoder.py).

* ``init_streaming_state`` builds the paged :class:`ModelCache`
  (encoder.py:140-165);
* ``_create_streaming_masks`` is one HIP launch for the whole batch instead of
  a per-stream Python loop with two device->host syncs per stream
  (encoder.py:167-227);
* ``forward`` keeps the layer loop and the state advance (encoder.py:229-267);
  the attention of every layer runs on the paged cache;
* ``EncoderStepGraph`` replays a recorded step for a fixed batch: the 9 to 14
  launches per layer that ``forward`` issues from Python (15 to 17 where the layer
  runs module by module) become one HIP graph replay, with the host page work and
  one upload per step left outside it.

The parameters are torch modules with the reference's names (encoder.py:11-81,
feedforward.py:4-26).  In 16 bits without gradients, a layer's products run on
``pk_linear``: SiLU in the first feed-forward product, the convolution module's
GLU and depthwise conv in its first pointwise product with each stream's conv
state updated in place (convolution.py:107-162, cache.py:47-53), its LayerNorm
and SiLU ahead of the second, and for few rows each residual update and LayerNorm
in the product that reads it.  Every other case (fp32, gradients, hooks, other
sizes) runs the modules, with the conv step as one HIP launch.  ``pre_encode`` is the batched convolution subsampling of
``modules/frontend.py`` (one HIP launch for the 8x stack), built from the same
constructor arguments as the reference's (encoder.py:105-112), so a reference
checkpoint loads strictly and ``ModelRunner`` finds ``encoder.pre_encode``
(model_runner.py:44,221).
"""

from __future__ import annotations

import torch
from torch import Tensor, nn
from torch.nn import functional as F

from .. import ops
from .attention import ConformerAttention, PositionalEncoding
from .cache import ConvCacheRef, ModelCache, StreamingState
from .frontend import ConvSubsampling


class ConformerFeedForward(nn.Module):
    def __init__(self, hidden_size: int, d_ff: int, dropout: float, use_bias: bool = True):
        super().__init__()
        self.d_model = hidden_size
        self.d_ff = d_ff
        self.use_bias = use_bias
        self.linear1 = nn.Linear(hidden_size, d_ff, bias=use_bias)
        self.activation = nn.SiLU()
        self.linear2 = nn.Linear(d_ff, hidden_size, bias=use_bias)
        self.dropout = nn.Dropout(dropout)

    def forward(self, x: Tensor) -> Tensor:
        if not torch.jit.is_scripting():
            y = self._launched(x)
            if y is not None:
                return y
        return self.linear2(self.dropout(self.activation(self.linear1(x))))

    def _launched(self, x: Tensor):
        """The block with linear1 and its SiLU as one launch, or None where the
        modules have to run (what :func:`ops.linear_applies` and :meth:`_fused`
        leave to them; a traced stand-in for x touches no parameter here)."""
        l1, l2 = self.linear1, self.linear2
        if type(x) not in (Tensor, nn.Parameter) or not self._fused(l1):
            return None
        w1, b1 = l1.weight, l1.bias
        if not ops.linear_applies(x, w1, b1, silu=True):
            return None
        if ops.plain_module(l2, nn.Linear):
            w2, b2 = l2.weight, l2.bias
            if w2.shape[1:] == w1.shape[:1] and ops.layer_applies(x.dtype, x.device, x.numel() // x.shape[-1], w2, b2):
                return ops._feed_forward(x, w1, b1, w2, b2)
        return l2(ops.linear(x, w1, b1, silu=True))

    def _fused(self, linear1: nn.Module | None = None) -> bool:
        drop = self.dropout
        return (
            ops.plain_module(self.linear1 if linear1 is None else linear1, nn.Linear)
            and ops.plain_module(self.activation, nn.SiLU)
            and ops.plain_module(drop, nn.Dropout)
            and not (drop.training and drop.p > 0.0)
        )


class CausalConv1d(nn.Conv1d):
    """Depthwise conv whose left context comes from a per-stream cache of
    kernel_size-1 frames (parakeet/modules/convolution.py:8-52); holds the
    parameters, the step itself runs in ConformerConvolution."""

    def __init__(self, in_channels, out_channels, kernel_size, stride=1, padding=(0, 0), dilation=1, groups=1, bias=True):
        self._left_padding = padding[0]
        self._right_padding = padding[1]
        super().__init__(in_channels, out_channels, kernel_size, stride=stride, padding=0, dilation=dilation, groups=groups, bias=bias)


class ConformerConvolution(nn.Module):
    """pointwise conv -> [GLU -> pad mask -> causal depthwise conv with the
    stream's cache -> LayerNorm -> SiLU] -> pointwise conv
    (parakeet/modules/convolution.py:107-162).  The bracket is one HIP launch
    (``pk_conv_step``); the pointwise convolutions (kernel size 1) are matrix
    products.  ``cache`` is the reference's [B, D, kernel-1] state (a new state is
    returned), None (zeros), or a ``ConvCacheRef`` from ``ModelCache.conv_ref``
    (the batch's state is updated in place and None is returned)."""

    def __init__(self, hidden_size, kernel_size, use_bias=False):
        super().__init__()
        self.d_model = hidden_size
        self.kernel_size = kernel_size
        self.pointwise_conv1 = nn.Conv1d(hidden_size, hidden_size * 2, kernel_size=1, bias=use_bias)
        self.depthwise_conv = CausalConv1d(
            hidden_size, hidden_size, kernel_size, groups=hidden_size, padding=(kernel_size - 1, 0), bias=use_bias
        )
        self.batch_norm = nn.LayerNorm(hidden_size)
        self.activation = nn.SiLU()
        self.pointwise_conv2 = nn.Conv1d(hidden_size, hidden_size, kernel_size=1, bias=use_bias)

    def _middle(self, h: Tensor, pad_mask: Tensor | None, frames: Tensor, layer: int = 0, slots=None) -> Tensor:
        dw = self.depthwise_conv
        return ops.conv_step(
            h,
            frames,
            dw.weight,
            self.batch_norm.weight,
            self.batch_norm.bias,
            layer=layer,
            slots=slots,
            pad_mask=pad_mask,
            dw_bias=dw.bias,
            eps=self.batch_norm.eps,
        )

    def forward(self, x: Tensor, pad_mask: Tensor, cache=None):
        return self.after_pointwise1(
            ops.functional_linear(x, self.pointwise_conv1.weight.squeeze(-1), self.pointwise_conv1.bias), pad_mask, cache
        )

    def after_pointwise1(self, h: Tensor, pad_mask: Tensor, cache=None):
        """:meth:`forward` from the first pointwise convolution's output [B, T, 2 D]."""
        if isinstance(cache, ConvCacheRef):
            bn, dw = self.batch_norm, self.depthwise_conv
            y = cache.cache.conv_step(cache.layer_idx, h, pad_mask, dw.weight, dw.bias, bn.weight, bn.bias, bn.eps)
            new_cache = None
        else:
            B, K = h.shape[0], self.kernel_size
            if cache is None:
                frames = torch.zeros((B, 1, K - 1, self.d_model), dtype=h.dtype, device=h.device)
            else:
                frames = cache.transpose(1, 2).unsqueeze(1).contiguous()
            y = self._middle(h, pad_mask, frames)
            new_cache = frames[:, 0].transpose(1, 2)
        out = ops.functional_linear(y, self.pointwise_conv2.weight.squeeze(-1), self.pointwise_conv2.bias)
        return out, new_cache


class ConformerLayer(nn.Module):
    """FF/2 -> rel-pos MHA -> conv -> FF/2 -> LN (parakeet/modules/encoder.py:11-81)."""

    def __init__(self, layer_idx, hidden_size, d_ff, num_heads, dropout, conv_kernel_size, use_bias):
        super().__init__()
        self.layer_idx = layer_idx
        self.hidden_size = hidden_size
        self.norm_feed_forward1 = nn.LayerNorm(hidden_size)
        self.feed_forward1 = ConformerFeedForward(hidden_size, d_ff, dropout, use_bias)
        self.norm_conv = nn.LayerNorm(hidden_size)
        self.conv = ConformerConvolution(hidden_size, conv_kernel_size)
        self.norm_self_att = nn.LayerNorm(hidden_size)
        self.self_attn = ConformerAttention(layer_idx=layer_idx, hidden_size=hidden_size, num_heads=num_heads, use_bias=use_bias)
        self.norm_feed_forward2 = nn.LayerNorm(hidden_size)
        self.feed_forward2 = ConformerFeedForward(hidden_size, d_ff, dropout, use_bias)
        self.norm_out = nn.LayerNorm(hidden_size)

    def forward(self, x: Tensor, pos_emb: Tensor, pad_mask: Tensor, attn_mask: Tensor, cache: ModelCache):
        if self.fuses(x, cache):
            return self.finish(self.fused_step(x, pos_emb, pad_mask, attn_mask, cache))
        # each residual update and the LayerNorm that reads it are one step
        # (``residual_norm``); the layer's input is not modified
        residual, h = self.residual_norm(x, self.feed_forward1(self.norm_feed_forward1(x)), self.norm_self_att, 0.5)
        attn = self.self_attn(h, pos_emb, attn_mask=attn_mask, cache=cache)
        residual, h = self.residual_norm(residual, attn, self.norm_conv, 1.0, in_place=True)
        conv_out, conv_cache = self.conv(h, pad_mask=pad_mask, cache=cache.conv_ref(self.layer_idx))
        cache.update_conv_cache(self.layer_idx, conv_cache)
        residual, h = self.residual_norm(residual, conv_out, self.norm_feed_forward2, 1.0, in_place=True)
        _, out = self.residual_norm(residual, self.feed_forward2(h), self.norm_out, 0.5, in_place=True)
        return out

    def fuses(self, x: Tensor, cache) -> bool:
        """Whether :meth:`fused_step` is this layer's step on ``x``: every module
        of it is the class's own (no subclass, hook, replaced forward or active
        dropout that the fused launches would pass by) on one 16-bit dtype, and
        no gradient is asked for.  The line is where the first pointwise product
        stops taking the convolution with it (2,146 rows at d_model 1024, 8,583 at
        512): past it nothing is kept in fp32 between the two, and the modules one
        by one are faster.  us a layer in a recorded step, one by one and fused, mean
        of fp16 and bf16: 1024 wide, 2,100 rows 278 271, 2,296 278 280, 3,584 328
        338; 512 wide, 3,600 rows 240 239, 4,096 247 248, 5,200 312 315, 6,400 347
        351, 8,400 429 436."""
        attn, conv = self.self_attn, self.conv
        return (
            isinstance(cache, ModelCache)
            and self.residual_norm is ConformerLayer.residual_norm
            and x.is_contiguous()
            and ops.plain_module(attn, ConformerAttention)
            and ops.plain_module(attn.qkv, nn.Linear)
            and ops.plain_module(conv, ConformerConvolution)
            and ops.plain_module(conv.pointwise_conv1, nn.Conv1d)
            and all(
                ops.plain_module(ff, ConformerFeedForward) and ff._fused() and ops.linear_applies(x, ff.linear1.weight, ff.linear1.bias, silu=True)
                for ff in (self.feed_forward1, self.feed_forward2)
            )
            and all(
                ops.norm_applies(n, x)
                for n in (self.norm_feed_forward1, self.norm_self_att, self.norm_conv, self.norm_feed_forward2, self.norm_out)
            )
            and attn.qkv.weight.dtype == conv.pointwise_conv1.weight.dtype == x.dtype
            and x.numel() // x.shape[-1] * conv.pointwise_conv1.weight.numel() <= ops._LINEAR_PRODUCTS
        )

    def fused_step(self, x, pos_emb: Tensor, pad_mask: Tensor, attn_mask: Tensor, cache: ModelCache) -> ops.Pending:
        """The layer's step up to its last residual update and norm, which the
        next reader's launch takes with it (or :meth:`residual_norm`).  ``x``: the
        layer's input, or the layer before's :class:`ops.Pending` one."""
        ff1, ff2, attn, conv = self.feed_forward1, self.feed_forward2, self.self_attn, self.conv
        own = isinstance(x, ops.Pending)  # then the residual is this step's own buffer
        x, h = ops.norm_linear(x, self.norm_feed_forward1, ff1.linear1.weight, ff1.linear1.bias, silu=True)
        r, qkv = ops.norm_linear(
            x, self.norm_self_att, attn.qkv.weight, attn.qkv.bias, branch=ops.module_linear(h, ff1.linear2), alpha=0.5, in_place=own
        )
        a = attn.attend(qkv, pos_emb, attn_mask, cache)
        p1, p2, dw, bn = conv.pointwise_conv1, conv.pointwise_conv2, conv.depthwise_conv, conv.batch_norm
        w1, w2 = p1.weight.squeeze(-1), p2.weight.squeeze(-1)
        if ops.glu_conv_applies(r, w1, p1.bias, w2, p2.bias, dw, bn) and cache.takes_glu_conv(r):
            r, y = cache.glu_conv(self.layer_idx, r, a, self.norm_conv, w1, p1.bias, dw.weight, dw.bias, pad_mask)
            c = ops.norm_silu_linear(y, bn, w2, p2.bias)
        else:
            r, h = ops.norm_linear(r, self.norm_conv, w1, p1.bias, branch=a, in_place=True)
            c, state = conv.after_pointwise1(h, pad_mask=pad_mask, cache=cache.conv_ref(self.layer_idx))
            cache.update_conv_cache(self.layer_idx, state)
        r, h = ops.norm_linear(r, self.norm_feed_forward2, ff2.linear1.weight, ff2.linear1.bias, branch=c, silu=True, in_place=True)
        return ops.Pending(r, ops.module_linear(h, ff2.linear2), self.norm_out, 0.5)

    @staticmethod
    def finish(p: ops.Pending) -> Tensor:
        """The update and norm that :meth:`fused_step` left."""
        return ConformerLayer.residual_norm(p.x, p.branch, p.norm, p.alpha, in_place=True)[1]

    @staticmethod
    def residual_norm(residual: Tensor, branch: Tensor, norm: nn.LayerNorm, alpha: float, in_place: bool = False):
        """``residual += alpha * branch`` and ``norm(residual)`` (encoder.py:61-80),
        one HIP launch: returns the updated residual (``residual`` itself when
        ``in_place``) and its norm."""
        return ops.residual_norm(residual, branch, norm.weight, norm.bias, alpha=alpha, eps=norm.eps, in_place=in_place)


class ConformerEncoder(nn.Module):
    """Streaming FastConformer encoder stack on the paged cache
    (parakeet/modules/encoder.py:84-267); same constructor arguments."""

    def __init__(
        self,
        feat_in: int,
        hidden_size,
        ff_expansion_factor: int,
        num_layers: int,
        num_heads: int,
        subsampling_factor: int,
        pos_emb_max_len: int,
        conv_kernel_size: int,
        att_context_size,
        subsampling_conv_channels: int,
        use_bias: bool,
        pre_encode_cache_size: list | tuple = (0, 9),
        drop_extra_pre_encoded: int = 2,
        page_size: int = 16,
    ):
        super().__init__()
        self.embed_dim = hidden_size
        self.feat_in = feat_in
        self.subsampling_factor = subsampling_factor
        self.pre_encode = ConvSubsampling(
            hidden_size=hidden_size,
            subsampling_conv_channels=subsampling_conv_channels,
            feat_in=feat_in,
            subsampling_factor=subsampling_factor,
            stride=2,
            kernel_size=3,
        )
        self.pos_enc = PositionalEncoding(hidden_size=hidden_size, dropout_rate_emb=0.0, max_len=pos_emb_max_len, dropout=0.0)
        self.layers = nn.ModuleList(
            ConformerLayer(i, hidden_size, hidden_size * ff_expansion_factor, num_heads, 0.0, conv_kernel_size, use_bias)
            for i in range(num_layers)
        )
        self.pos_enc.extend_pe(pos_emb_max_len, device=next(self.parameters()).device)
        self.att_context_size = list(att_context_size)
        self.conv_kernel_size = conv_kernel_size
        self.pre_encode_cache_size = pre_encode_cache_size
        self.drop_extra_pre_encoded = drop_extra_pre_encoded
        self.page_size = page_size

    def init_streaming_state(
        self,
        batch_size: int = 1,
        device: torch.device | None = None,
        dtype: torch.dtype | None = None,
        **cache_kwargs,
    ) -> StreamingState:
        if device is None:
            device = next(self.parameters()).device
        if dtype is None:
            dtype = next(self.parameters()).dtype
        cache_kwargs.setdefault("page_size", self.page_size)
        cache = ModelCache(
            num_layers=len(self.layers),
            attn_context_size=self.att_context_size,
            embed_dim=self.embed_dim,
            conv_kernel_size=self.conv_kernel_size,
            batch_size=batch_size,
            device=device,
            dtype=dtype,
            **cache_kwargs,
        )
        return StreamingState(
            cache=cache,
            processed_frames=torch.zeros(batch_size, dtype=torch.int64, device=device),
            cache_lengths=torch.zeros(batch_size, dtype=torch.int64, device=device),
        )

    def _create_streaming_masks(
        self,
        current_len: int,
        cache_lengths: Tensor,
        processed_frames: Tensor,
        device: torch.device,
        lengths: Tensor | int,
    ):
        """(pad_mask [B, T], att_mask [B, T, left+T]) from one kernel launch."""
        batch = cache_lengths.shape[0]

        def as_state(v):
            if isinstance(v, Tensor):
                return v.to(device=device, dtype=torch.int64).contiguous()
            return torch.full((batch,), int(v), dtype=torch.int64, device=device)

        if lengths is None:
            raise ValueError("lengths is required (the reference compares against it, encoder.py:204)")
        lengths = as_state(lengths) if isinstance(lengths, Tensor) else int(lengths)
        return ops.streaming_mask(
            as_state(processed_frames),
            as_state(cache_lengths),
            lengths,
            chunk=current_len,
            left=self.att_context_size[0],
            chunk_size=self.att_context_size[1] + 1,
        )

    def forward(self, x: Tensor, state: StreamingState, length: Tensor | None = None, bypass_pre_encode: bool = False):
        cache_lengths = state.cache_lengths
        if not isinstance(cache_lengths, Tensor):
            cache_lengths = torch.full((x.size(0),), int(cache_lengths), dtype=torch.int64, device=x.device)
        processed = state.processed_frames
        if not isinstance(processed, Tensor):
            processed = torch.full((x.size(0),), int(processed), dtype=torch.int64, device=x.device)
        x, pos_emb = self.pos_enc(x, cache_len=self.att_context_size[0])
        pad_mask, att_mask = self._create_streaming_masks(
            current_len=x.size(1),
            cache_lengths=cache_lengths,
            processed_frames=processed,
            device=x.device,
            lengths=length,
        )
        # a layer's last residual update and norm run in the next layer's first launch
        pend = None
        for layer in self.layers:
            y = x if pend is None else pend.x
            if ops.plain_module(layer, ConformerLayer) and layer.fuses(y, state.cache):
                pend = layer.fused_step(x if pend is None else pend, pos_emb, pad_mask, att_mask, state.cache)
                continue
            if pend is not None:
                x, pend = ConformerLayer.finish(pend), None
            x = layer(x, pos_emb=pos_emb, pad_mask=pad_mask, attn_mask=att_mask, cache=state.cache)
        if pend is not None:
            x = ConformerLayer.finish(pend)
        if isinstance(length, Tensor):
            state.processed_frames.add_(length)
            state.cache_lengths.add_(length)
            state.cache_lengths.clamp_(max=self.att_context_size[0])
        else:
            state.processed_frames += x.size(1)
            state.cache_lengths = min(int(state.cache_lengths) + x.size(1), self.att_context_size[0])
        return x.transpose(1, 2), state


class EncoderStepGraph:
    """``encoder(x, state, length)`` for a fixed batch, recorded once in a HIP
    graph and replayed every step (the call ModelRunner._encode_step makes,
    parakeet/engine/model_runner.py:285-291, with whole chunks).

    Every launch of a step reads the same device memory each step: the page
    pools, the batch's block-table rows, the state counters, the conv state, the
    position table and the weights; only their contents change.  A call runs
    ``state.cache.open_step()`` (the host page work and the one upload of the
    batch's rows), copies ``x`` into a fixed input buffer and replays.  The first
    call runs the step eagerly -- its real work, which also initialises the
    libraries' handles -- and then records the step without running it.

    ``length`` is the per-stream frame count of every step ([B] int64; the engine
    feeds whole chunks, parakeet/engine/sequence.py:137-146).  The returned
    [B, D, T] tensor is a fixed buffer that the next call overwrites.
    """

    def __init__(self, encoder: ConformerEncoder, state: StreamingState, length: Tensor):
        cache = state.cache
        if not isinstance(cache, ModelCache):
            raise TypeError("state.cache must be the paged ModelCache")
        for name in ("processed_frames", "cache_lengths"):
            if not isinstance(getattr(state, name), Tensor):
                raise TypeError(f"state.{name} must be a device tensor (a recorded step advances it on the device)")
        B = cache.batch_size
        dev = cache.k_pages.device
        if not isinstance(length, Tensor) or tuple(length.shape) != (B,):
            raise ValueError(f"length must be a [{B}] tensor")
        self.encoder = encoder
        self.state = state
        self.length = length.to(device=dev, dtype=torch.int64).clone()
        self.shape = (B, cache.chunk, encoder.embed_dim)
        self.x: Tensor | None = None
        self.out: Tensor | None = None
        self.graph: torch.cuda.CUDAGraph | None = None

    def __call__(self, x: Tensor) -> Tensor:
        if tuple(x.shape) != self.shape:
            raise ValueError(f"x must be {self.shape}, got {tuple(x.shape)}")
        cache = self.state.cache
        cache.open_step()
        if self.graph is None:
            self.x = x.detach().clone()
            out, _ = self.encoder(self.x, self.state, length=self.length)
            graph = torch.cuda.CUDAGraph()
            with cache.recording(), torch.cuda.graph(graph):
                self.out, _ = self.encoder(self.x, self.state, length=self.length)
            self.graph = graph
            return out
        self.x.copy_(x)
        for layer in self.encoder.layers:  # the recording reads the kept position projections
            layer.self_attn.refresh_projected_pos()
        self.graph.replay()
        return self.out


__all__ = [
    "ConformerEncoder",
    "ConformerLayer",
    "ConformerConvolution",
    "ConformerFeedForward",
    "CausalConv1d",
    "EncoderStepGraph",
]
