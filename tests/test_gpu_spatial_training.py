"""GPU parity of the operator's training path on channels-last maps (the spatial forward and
``vh_srnl_spatial_backward`` as one autograd Function): against the float64 oracle, and
against the packed path (serialized scans, then the fusion) over the inputs both take."""

import pytest
import torch

from tests.helpers import assert_close, memories, randn

pytestmark = pytest.mark.gpu

_NAMES = ("dM_m", "dM_v", "dM_k", "dM_eta", "dM_alpha", "dx", "dq", "d_skip", "d_weights")


def _oracle(x, q, mems, skip, weights, chunks, dout, head_dim):
    """Output and gradients of the operator on NHWC maps, float64 on the CPU."""
    from oracle.oracle_torch import direction_fusion_torch, sequence_forward_torch
    from visionhope_amd.models.operator import scan_orders

    batch, height, width, channels = x.shape
    heads = channels // head_dim
    leaves = [torch.from_numpy(m).double().requires_grad_() for m in mems]
    leaves += [t.double().requires_grad_() for t in (x, q, skip, weights)]
    xs = scan_orders(leaves[5].reshape(batch, -1, channels), height, width)
    xs = xs.reshape(batch, 4, height * width, heads, head_dim).transpose(2, 3)
    qs = scan_orders(leaves[6].reshape(batch, -1, channels), height, width)
    y = sequence_forward_torch(xs, qs, leaves[:5], chunks)
    out = direction_fusion_torch(y, xs, leaves[7], leaves[8], height, width)
    (out * dout.double().permute(0, 3, 1, 2)).sum().backward()
    return out.detach(), [t.grad.numpy() for t in leaves]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,head_dim,chunks,per_direction,offset", [
    ((2, 5, 7, 32), 16, None, False, 0), ((1, 16, 17, 48), 16, None, True, 1), ((1, 3, 33, 96), 32, None, True, 0),
    ((2, 1, 9, 16), 16, None, False, 3), ((1, 6, 6, 32), 32, (7, 7, 7, 7), False, 0),
    ((1, 2, 70, 16), 16, None, False, 0),
    ((32, 2, 35, 32), 16, None, False, 0), ((33, 2, 35, 32), 16, None, False, 0),        # 256 lines: spare waves; 264
    ((64, 17, 3, 32), 32, None, False, 0), ((65, 17, 3, 32), 32, None, False, 0)])
def test_spatial_backward_matches_oracle(device, shape, head_dim, chunks, per_direction, offset, dtype):
    """Odd and single-row maps, several blocks per row, explicit chunk lengths, both skip
    layouts, tensors that start at an odd element.  FP32: the roundings of at most one
    chunk's products and, for the parameters, of the sum over pixels; 16-bit: one rounding
    per direction and one of the sum."""
    from visionhope_amd.models.srnl_core.spatial import srnl_spatial

    batch, height, width, channels = shape
    chunks = chunks or (width, width, height, height)
    heads = channels // head_dim

    def place(t):
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        flat[offset:] = t.reshape(-1).to(device)
        return flat[offset:].view(t.shape).requires_grad_()

    mems = memories(4, heads, head_dim, kind="perturbed", seed=channels)
    x, q = (randn(*shape, seed=s).to(dtype) for s in (301, 302))
    skip = randn(*((4, heads, head_dim) if per_direction else (heads, head_dim)), seed=303)
    weights = 1.0 + 0.3 * randn(4, channels, seed=304)
    dout = randn(*shape, seed=305)
    out_want, want = _oracle(x.float(), q.float(), mems, skip, weights, chunks, dout, head_dim)
    leaves = [torch.from_numpy(m).to(device).requires_grad_() for m in mems] + [place(t) for t in (x, q, skip, weights)]
    out = srnl_spatial(leaves[:5], leaves[5], leaves[6], leaves[7], leaves[8], chunks)
    got = torch.autograd.grad(out, leaves, dout.to(device))
    assert_close(out.detach().permute(0, 3, 1, 2).double().cpu().numpy(), out_want.numpy(), 2e-5, "output")
    tol = 2.0 ** -23 * (max(chunks) + 4 * head_dim)
    rounding = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    for name, g, w, leaf in zip(_NAMES, got, want, leaves):
        assert g.shape == leaf.shape and g.dtype == leaf.dtype, name
        assert_close(g.double().cpu().numpy(), w, tol + (rounding if name in ("dx", "dq") else 0.0), name)


def _train(op, x, dout, autocast, packed):
    """Output and gradients of one training step, with the packed path forced by a hook."""
    handle = op.srnl.register_forward_hook(lambda *_: None) if packed else None
    try:
        with torch.autocast("cuda", dtype=autocast or torch.bfloat16, enabled=autocast is not None):
            y = op(x)
        return [y] + list(torch.autograd.grad(y, [x] + list(op.parameters()), dout))
    finally:
        if handle is not None:
            handle.remove()


@pytest.mark.parametrize("merge", ["scale", "softmax", "sum"])
@pytest.mark.parametrize("layout", ["nchw", "channels_last", "sliced"])
@pytest.mark.parametrize("dim,head_dim,chunk,autocast", [
    (32, 16, None, None), (64, 32, None, torch.bfloat16), (48, 16, 9, None), (32, 16, None, torch.float16),
    (16, 8, None, None), (32, 16, 300, None)])
def test_training_step_matches_packed_path(device, dim, head_dim, chunk, autocast, layout, merge):
    """The module's training step against the packed path on the same inputs: NCHW and
    channels-last storage, a channel slice of a larger map, every merge mode, explicit
    chunk lengths, autocast; head_dim 8 and chunks above 256 take the packed path either
    way (the latter without gradients)."""
    from visionhope_amd.models import VisionHOPEOperator

    torch.manual_seed(dim)
    op = VisionHOPEOperator(dim, head_dim, chunk, merge, merge != "softmax").to(device).train()
    with torch.no_grad():
        for name, p in op.named_parameters():
            p.add_(torch.randn_like(p) * (0.05 if "M_" in name else 0.2))
    height, width = 11, 6
    dtype = autocast or torch.float32
    x = randn(2, dim, height, width, seed=311).to(device, dtype)
    if layout == "channels_last":
        x = x.contiguous(memory_format=torch.channels_last)
    elif layout == "sliced":
        x = randn(2, height, width, 2 * dim, seed=311).to(device, dtype).permute(0, 3, 1, 2)[:, dim // 2:dim // 2 + dim]
    x = x.detach().requires_grad_()
    dout = randn(2, dim, height, width, seed=312).to(device)
    if chunk == 300:
        with torch.no_grad():
            assert op(x).shape == x.shape
        with pytest.raises(NotImplementedError):
            op(x).sum().backward()
        return
    got, want = (_train(op, x, dout, autocast, packed) for packed in (False, True))
    # 16 bits: y and each direction's gradients are rounded at other places
    tol = {None: 2e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}[autocast]
    assert got[0].is_contiguous(memory_format=torch.channels_last) == want[0].is_contiguous(
        memory_format=torch.channels_last)
    names = ["y", "dx"] + [n for n, _ in op.named_parameters()]
    for name, g, w in zip(names, got, want):
        assert g.dtype == w.dtype and g.shape == w.shape, name
        assert_close(g.detach().double().cpu().numpy(), w.detach().double().cpu().numpy(), tol, f"{layout} {merge} {name}")


def test_input_overwritten_after_the_call(device):
    """With a frozen query projection nothing else keeps x for the backward: overwriting it
    after the call changes no gradient."""
    from visionhope_amd.models import VisionHOPEOperator

    torch.manual_seed(3)
    op = VisionHOPEOperator(32, 16).to(device).train()
    op.W_q.requires_grad_(False)
    x = randn(1, 5, 8, 32, seed=321).to(device).permute(0, 3, 1, 2)
    dout = randn(1, 32, 5, 8, seed=322).to(device)
    params = [p for p in op.parameters() if p.requires_grad]
    want = torch.autograd.grad(op(x), params, dout)
    y = op(x)
    x.zero_()
    for g, w in zip(torch.autograd.grad(y, params, dout), want):
        assert torch.equal(g, w)
