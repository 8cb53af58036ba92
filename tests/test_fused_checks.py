"""What the fused encoder launches refuse or leave to the modules, on the CPU: a
pointer that reaches a kernel is read by its dtype and stride alone, so every
shape, dtype and device the launch assumes is checked before it.  The library is
replaced by one that accepts the few-row forms and fails the test on a launch."""

import types

import pytest
import torch
from torch import nn

from parakeet_amd import ops


@pytest.fixture
def no_launch(monkeypatch):
    def launched(*_):
        pytest.fail("the native call was reached")

    stub = types.SimpleNamespace(pk_linear_takes_norm=lambda *_: 1, pk_linear=launched, pk_residual_norm=launched)
    monkeypatch.setattr(ops, "lib", lambda: stub)
    monkeypatch.setattr(ops, "_stream", lambda dev: None)
    return stub


def _half(*shape):
    return torch.zeros(*shape, dtype=torch.float16)


def _ln(D):
    return nn.LayerNorm(D).half().requires_grad_(False)


BRANCHES = {
    "fp32": lambda: torch.zeros(2, 2, 512),
    "broadcast": lambda: _half(1, 1, 512),
    "fewer rows": lambda: _half(2, 1, 512),
    "narrower": lambda: _half(2, 2, 256),
}


@pytest.mark.parametrize("branch", list(BRANCHES))
@pytest.mark.parametrize("entry", ["norm_linear", "norm_linear pending", "residual_norm2", "glu_conv"])
def test_branch_must_match_the_residual(no_launch, entry, branch):
    """A replaced or hooked linear2 / linear_out may return anything; the separate
    residual update refused what does not match, and so does every fused one."""
    x, br, n, w = _half(2, 2, 512), BRANCHES[branch](), _ln(512), _half(1024, 512)
    with pytest.raises(ValueError, match="must match"):
        if entry == "norm_linear":
            ops.norm_linear(x, n, w, None, branch=br, alpha=0.5)
        elif entry == "norm_linear pending":
            ops.norm_linear(ops.Pending(x, br, n, 0.5), n, w, None, silu=True)
        elif entry == "residual_norm2":
            ops.residual_norm2(ops.Pending(x, br, n, 0.5), n)
        else:
            ops.glu_conv(x, br, n, w, None, _half(512, 1, 9), None, _half(2, 1, 8, 512), 0, None, None)


def _conv_args(cache=(2, 1, 8, 512), dw=(512, 1, 9), db=(512,), layer=0, slots=None, weight=(1024, 512)):
    return (_half(*weight), None, _half(*dw), None if db is None else _half(*db), _half(*cache), layer, slots, None)


BAD_CONV = {
    "a cache of 4 rows": (dict(cache=(2, 1, 4, 512)), ValueError, "dw_weight"),
    "a cache of 10 rows": (dict(cache=(2, 1, 10, 512)), ValueError, "dw_weight"),
    "a narrower cache": (dict(cache=(2, 1, 8, 256)), ValueError, "cache must be"),
    "a cache of 3 dimensions": (dict(cache=(2, 8, 512)), ValueError, "cache must be"),
    "fewer slots than streams": (dict(cache=(1, 1, 8, 512)), ValueError, "slots"),
    "a layer past the cache": (dict(layer=1), IndexError, "out of range"),
    "a slot map of int64": (dict(slots=torch.zeros(2, dtype=torch.int64)), ValueError, "int32"),
    "a shorter slot map": (dict(slots=torch.zeros(1, dtype=torch.int32)), ValueError, "int32"),
    "a shorter depthwise bias": (dict(db=(256,)), ValueError, "dw_bias"),
    "fewer taps": (dict(dw=(512, 1, 5)), ValueError, "dw_weight"),
    "a narrower product": (dict(weight=(1024, 256)), ValueError, "weight must be"),
}


@pytest.mark.parametrize("what", list(BAD_CONV))
def test_glu_conv_refuses_a_state_that_does_not_fit(no_launch, monkeypatch, what):
    """The kernel indexes the state as [slot][layer][8][D]: what conv_step refuses,
    the launch that replaces it refuses too."""
    kw, error, match = BAD_CONV[what]
    monkeypatch.setattr(ops, "_require_device", lambda *t: t[0].device)
    x = _half(2, 2, 512)
    with pytest.raises(error, match=match):
        ops.glu_conv(x, x, _ln(512), *_conv_args(**kw))


@pytest.mark.parametrize("shape,dtype,takes", [((2, 1, 8, 512), torch.float16, True), ((2, 1, 4, 512), torch.float16, False),
                                               ((2, 1, 8, 1024), torch.float16, False), ((2, 1, 8, 512), torch.float32, False)])
def test_conv_state_of_another_shape_takes_the_conv_step(shape, dtype, takes):
    from parakeet_amd.modules.cache import ModelCache

    cache = object.__new__(ModelCache)
    cache.conv_frames = torch.zeros(shape, dtype=dtype)
    assert cache.takes_glu_conv(_half(2, 2, 512)) is takes


def test_glu_conv_applies_looks_at_the_depthwise_parameters():
    w1, w2, n = _half(1024, 512), _half(512, 512), _ln(512)
    x = _half(2, 2, 512)

    def applies(**kw):
        dw = nn.Conv1d(512, 512, 9, groups=512).half().requires_grad_(False)
        for k, v in kw.items():
            setattr(dw, k, v)
        return ops.glu_conv_applies(x, w1, None, w2, None, dw, n)

    assert applies() and applies(bias=None)
    assert not applies(bias=nn.Parameter(_half(256), requires_grad=False))
    assert not applies(bias=nn.Parameter(torch.zeros(512, device="meta", dtype=torch.float16), requires_grad=False))
    assert not applies(weight=nn.Parameter(_half(512, 1, 9)))  # a gradient is asked for
    assert not applies(bias=nn.Parameter(_half(512)))


@pytest.mark.filterwarnings("ignore:Sparse CSR")
def test_a_parameter_of_another_shape_keeps_torch(no_launch):
    """What torch's own modules broadcast, refuse or take another way is left to
    them: biases that are not [n], sparse weights, norms of another width."""
    w, x = _half(512, 512), _half(2, 2, 512)

    def applies(weight, bias=None):
        return ops.layer_applies(torch.float16, x.device, 4, weight, bias)

    assert applies(w) and applies(w, _half(512))
    assert not applies(w, _half(1)) and not applies(w, _half(256)) and not applies(w, _half(1, 512))
    assert not applies(w.to_sparse_csr()) and not applies(_half(512, 512, 1)) and not applies(_half(512))
    n = _ln(512)
    assert ops.norm_applies(n, x)
    n.weight = nn.Parameter(_half(256), requires_grad=False)
    assert not ops.norm_applies(n, x)
    assert not ops.glu_conv_applies(x, _half(1024, 256), None, w, None, nn.Conv1d(512, 512, 9, groups=512).half().requires_grad_(False), _ln(512))


def test_products_refuse_operands_that_do_not_fit(no_launch):
    x, n = _half(2, 2, 512), _ln(512)
    calls = [
        lambda: ops.linear(x, _half(512, 1024)),
        lambda: ops.linear(x, _half(512, 512).bfloat16()),
        lambda: ops.linear(x, _half(512, 512), _half(256)),
        lambda: ops.linear(x, _half(512, 1024)[:, ::2]),
        lambda: ops.linear(x, _half(512, 512).t()),
        lambda: ops.linear(x, _half(512, 512), _half(1024)[::2]),
        lambda: ops.feed_forward(x, _half(1024, 512), None, _half(512, 512), None),
        lambda: ops.norm_silu_linear(x, n, _half(512, 512), None),
        lambda: ops.norm_silu_linear(x.float(), _ln(256), _half(512, 512), None),
        lambda: ops.norm_linear(x, _ln(256), _half(512, 512), None, silu=True),
    ]
    for f in calls:
        with pytest.raises(ValueError):
            f()
    with pytest.raises(RuntimeError):  # torch's own
        ops.norm_linear(x, n, _half(512, 1024), None, silu=True)


def test_feed_forward_of_unequal_layers_is_refused_by_torch(monkeypatch):
    from parakeet_amd.modules.encoder import ConformerFeedForward

    ff = ConformerFeedForward(512, 1024, 0.0).half().eval().requires_grad_(False)
    ff.linear2 = nn.Linear(2048, 512).half().requires_grad_(False)
    monkeypatch.setattr(ops, "linear_applies", lambda *a, **k: True)
    monkeypatch.setattr(ops, "linear", lambda x, w, b, silu=False: torch.nn.functional.silu(torch.nn.functional.linear(x, w, b)))
    monkeypatch.setattr(ops, "_feed_forward", lambda *a: pytest.fail("the launch would read past the hidden rows"))
    with pytest.raises(RuntimeError):
        ff(_half(2, 2, 512))


def test_a_default_device_is_not_a_transform():
    from torch.overrides import TorchFunctionMode

    class Sees(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x = _half(2, 512)
    assert not ops._transformed(x)
    with torch.device("cpu"):
        assert not ops._transformed(x)
        with Sees():
            assert ops._transformed(x)
    with Sees(), torch.device("cpu"):
        assert ops._transformed(x)
    torch.set_default_device("cpu")
    try:
        assert not ops._transformed(x)
    finally:
        torch.set_default_device(None)


def test_own_conv_methods_of_a_cache_are_called(monkeypatch):
    """A cache that keeps its convolution state another way: the layer's fused step
    takes its conv_ref and hands the new state to its update_conv_cache."""
    from parakeet_amd.modules.cache import ModelCache
    from parakeet_amd.modules.encoder import ConformerLayer

    class Dense(ModelCache):
        def conv_ref(self, layer):
            return ("state of", layer)

        def update_conv_cache(self, layer, state):
            self.new = (layer, state)

    cache = object.__new__(Dense)
    cache.conv_frames = _half(2, 1, 8, 512)
    x = _half(2, 2, 512)
    assert not cache.takes_glu_conv(x)
    plain = object.__new__(ModelCache)
    plain.conv_frames = cache.conv_frames
    assert plain.takes_glu_conv(x)
    plain.conv_step = lambda *a: None
    assert not plain.takes_glu_conv(x)

    layer = ConformerLayer(1, 512, 1024, 8, 0.0, 9, False).half().eval().requires_grad_(False)
    monkeypatch.setattr(ops, "norm_linear", lambda x, norm, w, b, **kw: (x, _half(2, 2, w.shape[0])))
    monkeypatch.setattr(ops, "glu_conv_applies", lambda *a: True)
    monkeypatch.setattr(layer.self_attn, "attend", lambda *a: x)
    got = []
    monkeypatch.setattr(layer.conv, "after_pointwise1", lambda h, pad_mask, cache: (got.append(cache) or x, "next"))
    layer.fused_step(x, None, None, None, cache)
    assert got == [("state of", 1)] and cache.new == (1, "next")


def test_a_layer_with_its_own_residual_norm_runs_its_modules(monkeypatch):
    from parakeet_amd.modules.cache import ModelCache
    from parakeet_amd.modules.encoder import ConformerLayer

    class Own(ConformerLayer):
        @staticmethod
        def residual_norm(residual, branch, norm, alpha, in_place=False):
            return residual, norm(residual)

    monkeypatch.setattr(ops, "linear_applies", lambda *a, **k: True)
    x, cache = _half(2, 2, 512), object.__new__(ModelCache)
    make = lambda cls: cls(0, 512, 1024, 8, 0.0, 9, False).half().eval().requires_grad_(False)
    assert make(ConformerLayer).fuses(x, cache)
    assert not make(Own).fuses(x, cache)
    layer = make(ConformerLayer)
    layer.residual_norm = Own.residual_norm
    assert not layer.fuses(x, cache)
