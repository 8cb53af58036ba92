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
