"""pk_linear and the layers that take it against float64 (feedforward.py:20-26,
attention.py:92,122, convolution.py:152,158).

The bound: operands are exact 16-bit values, products accumulate in fp32 (K
terms: relative 2^-24 sqrt(K) of the sum of magnitudes, far below one rounding),
and each output is rounded once, relative 2^-11 (fp16) or 2^-8 (bf16).  Held at
1.05 roundings of the value plus the accumulation's 2^-24 K |x||w|.  SiLU adds
the fp32 exponential's few 2^-23."""

import math

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from parakeet_amd import ops
from parakeet_amd.modules.encoder import ConformerFeedForward

EPS = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}
TINY = {torch.float16: 2.0**-24, torch.bfloat16: 2.0**-130}


def _check(got, x, w, b, dtype, silu):
    y = x.double() @ w.double().T + (b.double() if b is not None else 0.0)
    mag = x.double().abs() @ w.double().abs().T
    ref = F.silu(y) if silu else y
    bar = 1.05 * EPS[dtype] * ref.abs() + 2.0**-22 * mag + TINY[dtype]
    err = (got.double() - ref).abs()
    assert bool((err <= bar).all()), (tuple(x.shape), tuple(w.shape), float((err - bar).max()))


# every form of the launch rule, its edges: one row, a row short of and past a
# tile, several tiles a CU; K of one stage and of many
CASES = [
    (1, 64, 512), (16, 512, 512), (17, 2048, 512), (2, 512, 2048), (33, 1024, 4096), (63, 1536, 768),
    (65, 4096, 1024), (129, 512, 256), (255, 3072, 1024), (480, 1024, 4096), (840, 1024, 1024), (841, 2048, 1024),
    (840, 4096, 1024), (1793, 1024, 1024), (4095, 512, 512), (1000, 64, 256), (4097, 2048, 512), (3600, 4096, 1024),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k", CASES)
def test_linear_matches_float64(cuda, dtype, rows, n, k):
    print(f"\n[linear] {dtype} rows={rows} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + n + k)
    x = torch.randn(rows, k, generator=g, device=cuda).to(dtype)
    w = (torch.randn(n, k, generator=g, device=cuda) / math.sqrt(k)).to(dtype)
    b = torch.randn(n, generator=g, device=cuda).to(dtype)
    for bias, silu in ((None, False), (b, True), (b, False)):
        _check(ops.linear(x, w, bias, silu=silu), x, w, bias, dtype, silu)


@pytest.mark.gpu
def test_linear_reads_strided_weights_and_odd_views(cuda):
    g = torch.Generator(device="cuda").manual_seed(1)
    big = (torch.randn(128, 1024, generator=g, device=cuda) / 16).half()
    w = big[:, 256:768]  # rows 1024 apart
    x = torch.randn(3, 5, 1024, generator=g, device=cuda).half()[..., 1:513]  # neither contiguous nor aligned
    assert ops.linear_applies(x, w, None)
    _check(ops.linear(x, w).reshape(15, 128), x.reshape(15, 512), w, None, torch.float16, False)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(1, 1), (64, 2), (60, 14), (2100, 4)])
def test_feed_forward_block(cuda, rows):
    d, dtype = 512, torch.float16
    print(f"\n[ff] {rows}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    with torch.device(cuda):
        ff = ConformerFeedForward(d, 4 * d, 0.1, use_bias=True).to(dtype).eval().requires_grad_(False)
    x = torch.randn(*rows, d, generator=g, device=cuda).to(dtype)
    with torch.no_grad():
        got = ff(x)
    h = F.silu(F.linear(x.double(), ff.linear1.weight.double(), ff.linear1.bias.double()))
    ref = F.linear(h, ff.linear2.weight.double(), ff.linear2.bias.double())
    mag = h.abs() @ ff.linear2.weight.double().abs().T
    # the hidden layer's rounding adds at most 2^-11 of each product's magnitude
    assert bool(((got.double() - ref).abs() <= EPS[dtype] * (1.05 * ref.abs() + 1.1 * mag)).all())


@pytest.mark.gpu
def test_feed_forward_keeps_gradients_hooks_dropout_and_autocast(cuda):
    """What a kernel call would pass by keeps torch's own path."""
    with torch.device(cuda):
        ff = ConformerFeedForward(512, 2048, 0.5).half()
    x = torch.randn(4, 2, 512, device=cuda).half()
    ff.train()
    y = ff(x.requires_grad_())  # gradients
    y.float().sum().backward()
    assert x.grad is not None and ff.linear1.weight.grad is not None
    with torch.no_grad():
        assert not torch.equal(ff(x), ff(x))  # dropout draws
        ff.eval()
        seen = []
        hook = ff.linear1.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        a = ff(x)
        hook.remove()
        assert seen == [torch.Size([4, 2, 2048])]
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert ff(x.float()).dtype == torch.bfloat16 and ff(x).dtype == torch.bfloat16
        b = torch.func.vmap(ff)(x)
        c = ff(x)
        for t in (b, c):
            assert float((t - a).abs().max()) <= 2.0**-8 * float(a.abs().max())
        ff.linear2 = nn.Sequential(ff.linear2)
        assert torch.equal(ff(x), ff.linear2(ops.linear(x, ff.linear1.weight, ff.linear1.bias, silu=True)))
        f32 = ConformerFeedForward(512, 2048, 0.0).to(cuda).eval()
        assert f32(x.float()).dtype == torch.float32


def _norm(D, dtype, device, g):
    n = nn.LayerNorm(D).to(device=device, dtype=dtype).requires_grad_(False)
    n.weight.copy_(1.0 + 0.2 * torch.randn(D, generator=g, device=device))
    n.bias.copy_(0.2 * torch.randn(D, generator=g, device=device))
    return n


# rows of one tile and a remainder, one tile a CU with 32, 64 and 128 outputs,
# and past them (the separate launches)
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k", [(1, 2048, 512), (17, 1536, 512), (100, 2048, 512), (250, 2048, 512), (700, 2048, 512),
                                      (2, 4096, 1024), (33, 3072, 1024), (64, 4096, 1024), (120, 4096, 1024), (300, 2048, 1024)])
def test_norm_linear_matches_its_parts(cuda, dtype, rows, n, k):
    """The residual is torch's own bit for bit; the product reads a norm that is
    within one rounding of the fp32 LayerNorm (statistics in another order), so
    outputs differ from the product of that norm by at most the sum of the
    operand's roundings (relative 2 eps of each product) and their own."""
    print(f"\n[norm-linear] {dtype} rows={rows} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + n + k)
    x = (2.0 * torch.randn(rows, k, generator=g, device=cuda) + 0.5).to(dtype)
    br = torch.randn(rows, k, generator=g, device=cuda).to(dtype)
    w = (torch.randn(n, k, generator=g, device=cuda) / math.sqrt(k)).to(dtype)
    n0, n1 = _norm(k, dtype, cuda, g), _norm(k, dtype, cuda, g)

    def ln(v, m):
        return F.layer_norm(v.double(), (k,), m.weight.double(), m.bias.double(), m.eps)

    def check(out, h, silu):
        y = h @ w.double().T
        mag = h.abs() @ w.double().abs().T
        ref = F.silu(y) if silu else y
        err = (out.double() - ref).abs()
        bar = 1.05 * EPS[dtype] * ref.abs() + (1.1 * EPS[dtype] * (2 * mag) if silu else EPS[dtype] * 2 * mag) + TINY[dtype]
        assert bool((err <= bar).all()), float((err - bar).max())
        # the roundings are independent: their sum grows as the root of their number
        rms = float((err.square().mean() / ref.square().mean()).sqrt())
        assert rms <= 2.0 * EPS[dtype], rms

    with torch.no_grad():
        r, out = ops.norm_linear(x, n1, w, None, silu=True)
        assert r is x
        check(out, ln(x, n1), True)
        want = x + br * 0.5
        for silu in (False, True):
            r, out = ops.norm_linear(x, n1, w, None, branch=br, alpha=0.5, silu=silu)
            assert torch.equal(r, want)
            check(out, ln(want, n1), silu)
        r, out = ops.norm_linear(ops.Pending(x, br, n0, 1.0), n1, w, None, silu=True)
        y, _ = ops.residual_norm2(ops.Pending(x, br, n0, 1.0), n1)
        assert float((r.double() - ln(x + br, n0)).abs().max()) <= 4 * EPS[dtype] * 4.0
        assert float((r - y).abs().float().max()) <= 8 * EPS[dtype]
        check(out, ln(r, n1), True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D,rows", [(torch.float16, 512, 5), (torch.bfloat16, 1024, 257), (torch.float32, 176, 3)])
def test_residual_norm2_is_two_norms(cuda, dtype, D, rows):
    g = torch.Generator(device="cuda").manual_seed(D)
    x, br = (torch.randn(rows, D, generator=g, device=cuda).to(dtype) for _ in range(2))
    n0, n1 = _norm(D, dtype, cuda, g), _norm(D, dtype, cuda, g)
    y, z = ops.residual_norm2(ops.Pending(x, br, n0, 0.5), n1)
    r, want = ops.residual_norm(x, br, n0.weight, n0.bias, alpha=0.5, eps=n0.eps)
    _, want2 = ops.residual_norm(want, torch.zeros_like(want), n1.weight, n1.bias, eps=n1.eps)
    assert torch.equal(y, want) and torch.equal(z, want2)


@pytest.mark.gpu
@pytest.mark.parametrize("streams", [3, 200])
def test_encoder_fused_layers_match_module_by_module(cuda, streams):
    """The fused step of the layers against the same encoder run module by module
    (a forward hook on a layer's submodule keeps its torch call), over several steps."""
    from parakeet_amd.modules.encoder import ConformerEncoder

    torch.manual_seed(streams)
    with torch.device(cuda):
        enc = ConformerEncoder(
            feat_in=80, hidden_size=512, ff_expansion_factor=4, num_layers=3, num_heads=8, subsampling_factor=8,
            pos_emb_max_len=500, conv_kernel_size=9, att_context_size=[70, 1], subsampling_conv_channels=256, use_bias=False,
        )
    for layer in enc.layers:
        layer.self_attn.pos_bias_u.data.normal_(std=0.02)
        layer.self_attn.pos_bias_v.data.normal_(std=0.02)
    enc = enc.half().eval().requires_grad_(False)
    states = [enc.init_streaming_state(batch_size=streams, device=cuda, dtype=torch.float16) for _ in range(3)]
    length = torch.full((streams,), 2, dtype=torch.int64, device=cuda)
    with torch.no_grad():
        for step in range(4):
            x = torch.randn(streams, 2, 512, device=cuda).half()
            assert enc.layers[0].fuses(x, states[0].cache)
            a, _ = enc(x, states[0], length=length)
            hooks = [m.register_forward_hook(lambda *_: None) for m in (enc.layers[1].feed_forward1.linear1, enc.layers[2].norm_conv)]
            assert not enc.layers[1].fuses(x, states[1].cache) and not enc.layers[2].fuses(x, states[1].cache)
            b, _ = enc(x, states[1], length=length)
            hooks += [enc.layers[0].self_attn.register_forward_hook(lambda *_: None)]
            c, _ = enc(x, states[2], length=length)
            for h in hooks:
                h.remove()
            for t in (b, c):  # three layers of independent fp16 roundings
                assert float((t.float() - a.float()).norm() / a.float().norm()) <= 4e-3


# streams of 1, 2, 3, 14 and 16 frames: several streams a tile and a remainder, a
# tile of 16 rows not filled; few rows (the norm form) and the tile forms
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T,D", [(1, 2, 512), (5, 3, 512), (70, 2, 512), (40, 1, 512), (7, 14, 1024), (3, 16, 512), (33, 2, 1024),
                                   (60, 14, 1024), (300, 2, 512), (700, 3, 512), (1025, 2, 512), (900, 1, 1024)])
def test_glu_conv_matches_its_parts(cuda, dtype, B, T, D):
    """pk_linear with the depthwise convolution, then with the norm and SiLU,
    against float64 and pk_conv_step over two steps: shuffled slots, one padded
    frame.  The cache holds GLU outputs rounded once (fused: from fp32 values and
    gates; parts: from values rounded first), so the two agree within the
    roundings of value and gate: 3 roundings of max(1, |value|)."""
    print(f"\n[glu-conv] {dtype} B={B} T={T} D={D}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B * 31 + T)
    Ly, layer, S, eps = 2, 1, B + 3, EPS[dtype]
    w1 = (torch.randn(2 * D, D, generator=g, device=cuda) / math.sqrt(D)).to(dtype)
    b1 = (0.1 * torch.randn(2 * D, generator=g, device=cuda)).to(dtype)
    w2 = (torch.randn(D, D, generator=g, device=cuda) / math.sqrt(D)).to(dtype)
    dw = (torch.randn(D, 1, 9, generator=g, device=cuda) / 3).to(dtype)
    db = (0.1 * torch.randn(D, generator=g, device=cuda)).to(dtype)
    norm, bn = _norm(D, dtype, cuda, g), _norm(D, dtype, cuda, g)
    slots = torch.randperm(S, generator=g, device=cuda)[:B].to(torch.int32)
    cache = torch.randn(S, Ly, 8, D, generator=g, device=cuda).to(dtype)
    pad = torch.zeros(B, T, dtype=torch.bool, device=cuda)
    pad[B // 2, T - 1] = True
    for step in range(2):
        x = torch.randn(B, T, D, generator=g, device=cuda).to(dtype)
        br = torch.randn(B, T, D, generator=g, device=cuda).to(dtype)
        mine, parts = cache.clone(), cache.clone()
        want_r = x + br
        r, y = ops.glu_conv(x.clone(), br, norm, w1, b1, dw, db, mine, layer, slots, pad)
        assert torch.equal(r, want_r) and y.dtype == torch.float32
        # float64 from this step's cache and the module's own roundings of the norm
        h = F.layer_norm(want_r.double(), (D,), norm.weight.double(), norm.bias.double(), norm.eps)
        v, ga = (h.to(dtype).double() @ w1.double().T + b1.double()).chunk(2, -1)
        glu = (v * torch.sigmoid(ga)).masked_fill(pad[..., None], 0.0)
        win = torch.cat([cache[slots.long(), layer].double(), glu], 1)
        ref = sum(win[:, k : k + T] * dw[:, 0, k].double() for k in range(9)) + db.double()
        assert float((y.double() - ref).norm() / ref.norm()) <= 2 * eps
        new = mine[slots.long(), layer]
        assert bool(((new.double() - win[:, -8:]).abs() <= 3 * eps * win[:, -8:].abs().clamp(min=1.0)).all())
        others = torch.ones(S, dtype=torch.bool, device=cuda)
        others[slots.long()] = False
        assert torch.equal(mine[others], cache[others]) and torch.equal(mine[:, 0], cache[:, 0])
        if T < 8:  # rows that only move keep their bits
            assert torch.equal(new[:, : 8 - T], cache[slots.long(), layer][:, T:])
        assert bool((new[B // 2, -1] == 0).all())
        # against the separate launches
        _, hh = ops.residual_norm(x, br, norm.weight, norm.bias, eps=norm.eps)
        z = ops.conv_step(ops.linear(hh, w1, b1), parts, dw, bn.weight, bn.bias, layer=layer, slots=slots, pad_mask=pad, dw_bias=db, eps=bn.eps)
        out = ops.norm_silu_linear(y, bn, w2, None)
        sep = ops.linear(z, w2, None)
        exact = F.silu(F.layer_norm(ref, (D,), bn.weight.double(), bn.bias.double(), bn.eps)) @ w2.double().T
        e_new, e_old = (float((t.double() - exact).norm() / exact.norm()) for t in (out, sep))
        print(f"  error against float64: fused {e_new:.2e}, parts {e_old:.2e}", flush=True)
        assert e_new <= 1.05 * e_old + 0.1 * eps
        cache = mine


@pytest.mark.gpu
def test_feed_forward_under_transforms_of_its_weights(cuda):
    """functional_call under vmap and grad over the weights, and a symbolic trace,
    keep torch's path: 3 fp16 roundings of values below the output's maximum."""
    from torch.func import functional_call, grad, vmap

    torch.manual_seed(4)
    with torch.device(cuda):
        ff = ConformerFeedForward(256, 512, 0.0).half().eval().requires_grad_(False)
    x = torch.randn(4, 2, 256, device=cuda).half()
    p = dict(ff.named_parameters())
    with torch.no_grad():
        want = ff(x)
        y = vmap(lambda q: functional_call(ff, q, (x,)))({k: torch.stack([v, v]) for k, v in p.items()})
        traced = torch.fx.symbolic_trace(ff)(x)
    bar = 3 * EPS[torch.float16] * float(want.abs().max())
    assert float((y[1] - want).abs().max()) <= bar and float((traced - want).abs().max()) <= bar
    g = grad(lambda q: functional_call(ff, q, (x,)).float().square().sum())(p)
    assert all(v.dtype == torch.float16 and float(v.abs().sum()) > 0 for v in g.values())


@pytest.mark.gpu
def test_linear_with_more_column_tiles_than_a_grid_holds(cuda):
    """8 row tiles by 65,537 column tiles: the block split over the XCDs would be a
    grid of 8 x 1 x 65,537 (limit 65,535); the linear tile order takes it."""
    rows, n, k, dtype = 449, 64 * 65537, 256, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(rows, k, generator=g, device=cuda).to(dtype)
    w = torch.randn(n, k, generator=g, device=cuda, dtype=dtype) / 16
    y = ops.linear(x, w)
    for c in (slice(0, 128), slice(n // 2, n // 2 + 128), slice(n - 128, n)):
        _check(y[:, c], x, w[c], None, dtype, False)


@pytest.mark.gpu
def test_encoder_refuses_what_its_launches_do_not_fit(cuda):
    """A hooked linear2 or linear_out that returns another dtype or shape, and a
    cache built for another kernel size: the errors of the separate launches,
    raised on the host; the encoder steps on afterwards."""
    from parakeet_amd.modules.encoder import ConformerEncoder

    torch.manual_seed(6)

    def build(kernel):
        with torch.device(cuda):
            enc = ConformerEncoder(
                feat_in=80, hidden_size=512, ff_expansion_factor=4, num_layers=2, num_heads=8, subsampling_factor=8,
                pos_emb_max_len=500, conv_kernel_size=kernel, att_context_size=[70, 1], subsampling_conv_channels=256, use_bias=False,
            )
        for layer in enc.layers:
            layer.self_attn.pos_bias_u.data.normal_(std=0.02)
            layer.self_attn.pos_bias_v.data.normal_(std=0.02)
        return enc.half().eval().requires_grad_(False)

    enc, B = build(9), 3
    length = torch.full((B,), 2, dtype=torch.int64, device=cuda)
    x = torch.randn(B, 2, 512, device=cuda).half()

    def state(of):
        return of.init_streaming_state(batch_size=B, device=cuda, dtype=torch.float16)

    with torch.no_grad():
        assert enc.layers[0].fuses(x, state(enc).cache)
        want, _ = enc(x, state(enc), length=length)
        for module in (enc.layers[0].feed_forward1.linear2, enc.layers[1].self_attn.linear_out, enc.layers[1].feed_forward2.linear2):
            for change in (lambda o: o.float(), lambda o: o[:1], lambda o: o.mean(1, keepdim=True)):
                hook = module.register_forward_hook(lambda m, i, o: change(o))
                with pytest.raises(ValueError, match="must match"):
                    enc(x, state(enc), length=length)
                hook.remove()
        for kernel in (5, 15):
            with pytest.raises(ValueError, match="dw_weight"):
                enc(x, state(build(kernel)), length=length)
        got, _ = enc(x, state(enc), length=length)
        assert torch.equal(got, want)
        torch.set_default_device(cuda)
        try:
            assert enc.layers[0].fuses(x, state(enc).cache)
        finally:
            torch.set_default_device(None)
