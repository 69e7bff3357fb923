"""Which native calls the training entries of the operator reach, on the CPU with those calls
replaced: derivatives they must refuse, one arithmetic with and without gradients, and what
they keep for the backward."""

import pytest
import torch
from torch.autograd import forward_ad

from visionhope_amd.models import VisionHOPEOperator, operator as operator_module
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


@pytest.fixture
def operator(monkeypatch):
    """An operator whose spatial training entries return x and record their map and queries."""
    seen = []
    monkeypatch.setattr(operator_module, "spatial_training_supported", lambda *_: True)
    monkeypatch.setattr(operator_module, "projected_training_supported", lambda *_: True)
    monkeypatch.setattr(operator_module, "srnl_spatial",
                        lambda m, x, q, *_: seen.append(("module", x, q)) or x.float().clone())
    monkeypatch.setattr(operator_module, "srnl_spatial_projected",
                        lambda m, x, *_: seen.append(("projected", x, None)) or x.float().clone())
    op = VisionHOPEOperator(HEADS * HEAD_DIM, HEAD_DIM).train()
    op.seen = seen
    return op


def _channels_last():
    return torch.randn(2, HEADS * HEAD_DIM, 3, 5).contiguous(memory_format=torch.channels_last)


def test_query_projection_may_be_any_module(operator):
    """``W_q`` replaced by a module without a ``weight`` of its own (an adapter around the
    Linear, say): the call goes through, and the map kept for the backward is a copy, since
    no Linear is known to keep it."""
    operator.W_q = torch.nn.Sequential(operator.W_q, torch.nn.Identity())
    x = _channels_last()
    operator(x)
    (route, kept, q), = operator.seen
    assert route == "module" and kept.data_ptr() != x.data_ptr()
    assert torch.equal(q, operator.W_q(x.permute(0, 2, 3, 1)))


@pytest.mark.parametrize("frozen", [True, False])
def test_projection_route_does_not_depend_on_gradients(operator, frozen):
    """The same projection with and without gradients, and no copy of the map where nothing
    is kept for a backward."""
    operator.W_q.requires_grad_(not frozen)
    x = _channels_last()
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            operator(x)
    (route, without, _), (route_grad, _, _) = operator.seen
    assert route == route_grad == ("module" if frozen else "projected")
    assert without.data_ptr() == x.data_ptr()


class _Recorder:
    """A native library that runs nothing and records the pointers of each call."""

    def __init__(self):
        self.pointers = {}

    def __getattr__(self, name):
        def call(*args):
            self.pointers[name] = args
            return 4096 if name.endswith("_bytes") else 0
        return call


def test_backward_takes_saved_tensors_of_any_strides(monkeypatch):
    """Saved-tensor hooks may hand tensors back with other strides than they were saved with;
    kernels that read them by pointer get contiguous copies."""
    lib = _Recorder()
    monkeypatch.setattr(spatial.hip, "load_library", lambda *_: lib)
    monkeypatch.setattr(spatial.hip, "stream_of", lambda _: 0)
    mems, x, q, skip, weights, chunks = _inputs()
    gains = torch.zeros(64, 2)[:, 0]
    spatial.srnl_spatial_backward(mems, x, q, skip, weights, chunks, gains, torch.ones_like(x))
    assert gains.data_ptr() not in lib.pointers["vh_srnl_spatial_backward"]
    x = torch.zeros(*x.shape, 2)[..., 0]
    operands = torch.zeros(66, 32, 2)[..., 0]
    dq = torch.zeros(1, 3, 5, 32)
    spatial.project_queries_backward(x, operands, dq, dq, True, True)
    assert x.data_ptr() not in lib.pointers["vh_linear_weight_grad"]
    first, last = operands.data_ptr(), operands.data_ptr() + 4 * operands.numel()
    assert not any(isinstance(p, int) and first <= p < last for p in lib.pointers["vh_pointwise_conv_nhwc_forward"])


@pytest.mark.parametrize("chunk,kept", [(7, True), (6, False)])
def test_large_gains_are_not_kept(monkeypatch, chunk, kept):
    """A step keeps its chunk gains up to a size in proportion to the map; beyond that the
    backward forms them again."""
    gains = torch.zeros(4 * 3 * -(-168 // chunk) * 32 * 32)   # 4 directions, 3 heads of 32, 168 tokens
    monkeypatch.setattr(spatial, "srnl_spatial_training_forward", lambda m, x, *_: (x.detach().clone(), gains))
    seen = []
    monkeypatch.setattr(spatial, "srnl_spatial_backward", lambda m, x, q, s, w, c, gains, dout: seen.append(gains) or (
        *m, x, q, s, w))
    mems = [torch.zeros(4, 3, 32, 32) for _ in range(3)] + [torch.zeros(4, 3, 32) for _ in range(2)]
    x = torch.zeros(1, 8, 21, 96, requires_grad=True)
    spatial.srnl_spatial(mems, x, x.detach(), torch.zeros(96), torch.ones(4, 96), (chunk,) * 4).sum().backward()
    assert len(seen) == 1 and (seen[0] is not None) == kept
