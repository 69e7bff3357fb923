"""Which native calls the training entries of the operator reach, on the CPU with those calls
replaced: derivatives they must refuse, one arithmetic with and without gradients, and what
they keep for the backward."""

import pytest
import torch
from torch.autograd import forward_ad

from visionhope_amd.models.srnl_core import spatial

HEADS, HEAD_DIM = 2, 16


def _inputs(requires_grad=False):
    gen = torch.Generator().manual_seed(5)

    def randn(*shape):
        return torch.randn(*shape, generator=gen).requires_grad_(requires_grad)

    mems = [randn(4, HEADS, HEAD_DIM, HEAD_DIM) for _ in range(3)] + [randn(4, HEADS, HEAD_DIM) for _ in range(2)]
    channels = HEADS * HEAD_DIM
    x, q = randn(1, 3, 5, channels), randn(1, 3, 5, channels)
    return mems, x, q, randn(HEADS, HEAD_DIM), randn(4, channels), (5, 5, 3, 3)


@pytest.fixture
def calls(monkeypatch):
    """The native forward replaced by x, its calls recorded."""
    seen = []

    def forward(memories, x, *_):
        seen.append("training")
        return x.detach().clone(), torch.zeros(1)

    monkeypatch.setattr(spatial, "srnl_spatial_training_forward", forward)
    if hasattr(spatial, "srnl_spatial_inference"):
        monkeypatch.setattr(spatial, "srnl_spatial_inference", lambda s, x, *_: seen.append("inference") or x.clone())
    return seen


@pytest.mark.parametrize("tangent", ["x", "q", "memory", "d_skip", "weights"])
@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_derivatives_are_refused(calls, tangent, grad):
    """No native call carries a tangent, so a dual input raises whether or not gradients are
    recorded; an output without its tangent would be a wrong derivative."""
    mems, x, q, skip, weights, chunks = _inputs()
    with forward_ad.dual_level(), torch.set_grad_enabled(grad):
        def dual(t, name):
            return forward_ad.make_dual(t, torch.ones_like(t)) if name == tangent else t

        mems[1] = dual(mems[1], "memory")
        with pytest.raises(NotImplementedError):
            spatial.srnl_spatial(mems, dual(x, "x"), dual(q, "q"), dual(skip, "d_skip"), dual(weights, "weights"), chunks)


def test_one_forward_with_and_without_gradients(calls):
    """Activation checkpointing runs the forward without gradients and again with them, and
    both must be the same kernels."""
    for requires_grad in (True, False):
        args = _inputs(requires_grad)
        with torch.no_grad():
            assert not spatial.srnl_spatial(*args).requires_grad
        assert spatial.srnl_spatial(*args).requires_grad == requires_grad
    assert calls == ["training"] * 4
