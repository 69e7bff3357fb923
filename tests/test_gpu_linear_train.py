"""The query projection of a training step: operands, weight gradients and the fused
autograd Function, against float64 and against the step that calls the ``W_q`` module."""

import pytest
import torch

from tests.helpers import memories, randn, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 257, 1000, 5003])
@pytest.mark.parametrize("n,k", [(16, 16), (32, 48), (128, 128), (144, 272)])
def test_weight_gradient(device, tokens, n, k):
    """Widths inside, at and over a workgroup's 128 channels; tokens around a step and a
    workgroup's share.  Products of bf16 are exact in FP32, so the error is that of a sum
    of ``tokens`` FP32 terms: each rounding at most 2^-23 of the terms' absolute sum."""
    from visionhope_amd.utils import hip

    dy, x = (randn(tokens, w, seed=tokens + w).to(torch.bfloat16).to(device) for w in (n, k))
    dw, db = torch.empty(n, k, device=device), torch.empty(n, device=device)
    lib = hip.load_library()
    ws = hip.workspace(lib.vh_linear_weight_grad_workspace_bytes(tokens, n, k), device)
    hip.check(lib.vh_linear_weight_grad(dy.data_ptr(), x.data_ptr(), tokens, n, k, dw.data_ptr(), db.data_ptr(),
                                        ws.data_ptr(), ws.numel() * 4, hip.stream_of(x)), "vh_linear_weight_grad")
    dy, x = dy.cpu().double(), x.cpu().double()
    bound = (tokens + 16) * 2.0 ** -23
    for got, want, size in ((dw, dy.T @ x, dy.abs().T @ x.abs()), (db, dy.sum(0), dy.abs().sum(0))):
        assert ((got.cpu().double() - want).abs() <= bound * size).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k", [(1, 1), (16, 48), (96, 32)])
def test_operands(device, n, k, dtype):
    from visionhope_amd.utils import hip

    w, b = randn(n, k, seed=1).to(dtype).to(device), randn(n, seed=2).to(dtype).to(device)
    w16, wt16 = (torch.empty(s, device=device, dtype=torch.bfloat16) for s in ((n, k), (k, n)))
    b32 = torch.empty(n, device=device)
    hip.check(hip.load_library().vh_linear_operands(
        w.data_ptr(), b.data_ptr(), hip.dtype_code(dtype), n, k, w16.data_ptr(), wt16.data_ptr(), b32.data_ptr(),
        hip.stream_of(w)), "vh_linear_operands")
    assert torch.equal(w16, w.to(torch.bfloat16)) and torch.equal(wt16, w16.T)
    assert torch.equal(b32, b.to(torch.bfloat16).float())


@pytest.mark.parametrize("layout", ["nchw", "channels_last", "offset"])
@pytest.mark.parametrize("frozen", [None, "x", "W_q.bias"])
@pytest.mark.parametrize("shape,head_dim", [((2, 32, 7, 9), 16), ((1, 160, 5, 3), 32), ((3, 96, 16, 17), 16)])
def test_projected_step_matches_module_call(device, shape, head_dim, frozen, layout):
    """The step with the projection inside the Function against the step that a hook on
    ``W_q`` makes call the module.  Both round the queries, the map gradient's two terms and
    (the module only) the weight gradients to bf16: half an ulp, 2^-9 of a value, on either
    side."""
    from visionhope_amd.models import VisionHOPEOperator

    batch, dim, height, width = shape
    op = VisionHOPEOperator(dim, head_dim=head_dim).to(device)
    with torch.no_grad():
        for p, m in zip(op.srnl.initial_memories, memories(4, dim // head_dim, head_dim, kind="perturbed", seed=dim)):
            p.copy_(torch.from_numpy(m))
        op.W_q.bias.copy_(randn(dim, seed=4, scale=0.1))
        op.W_q.weight.copy_(randn(dim, dim, seed=5, scale=dim ** -0.5))
        op.d_skip.copy_(randn(*op.d_skip.shape, seed=6, scale=0.3))
    x = randn(batch, height, width, dim, seed=7).to(torch.bfloat16).to(device)
    if layout == "offset":
        x = torch.empty(x.numel() + 1, dtype=x.dtype, device=device)[1:].view(x.shape).copy_(x)
    x = x.permute(0, 3, 1, 2)
    x = (x.contiguous() if layout == "nchw" else x).detach().requires_grad_(frozen != "x")
    op.W_q.bias.requires_grad_(frozen != "W_q.bias")
    leaves = [t for t in (x, *op.parameters()) if t.requires_grad]
    dout = randn(*shape, seed=8).to(device)

    def step(module_call):
        handle = op.W_q.register_forward_hook(lambda *_: None) if module_call else None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = op(x)
        if handle is not None:
            handle.remove()
        return y, torch.autograd.grad(y, leaves, dout)

    (y, got), (y_ref, want) = step(False), step(True)
    for g, w, leaf in zip((y, *got), (y_ref, *want), (y_ref, *leaves)):
        assert g.dtype == w.dtype == leaf.dtype and g.shape == w.shape
        assert rel_err(g.detach().float().cpu().numpy(), w.detach().float().cpu().numpy()) <= 2.0 ** -8


@pytest.mark.parametrize("dim,head_dim,layout", [(32, 16, "channels_last"), (96, 32, "nchw"), (48, 16, "nchw"),
                                                 (128, 16, "offset")])
@pytest.mark.parametrize("bias", [True, False])
def test_inference_projection(device, dim, head_dim, layout, bias):
    """The operator's queries in inference under bf16 autocast against float64: one rounding
    of W and b (2^-9 each of their terms) and one of q."""
    from visionhope_amd.models import VisionHOPEOperator
    from visionhope_amd.models.srnl_core import fused

    op = VisionHOPEOperator(dim, head_dim=head_dim, fast_inference=True).to(device).eval()
    with torch.no_grad():
        op.W_q.weight.copy_(randn(dim, dim, seed=5, scale=dim ** -0.5))
        op.W_q.bias.copy_(randn(dim, seed=4, scale=0.1))
    if not bias:
        op.W_q.bias = None
    x = randn(2, 5, 7, dim, seed=7).to(torch.bfloat16).to(device)
    if layout == "offset":
        x = torch.empty(x.numel() + 1, dtype=x.dtype, device=device)[1:].view(x.shape).copy_(x)
    x = x.permute(0, 3, 1, 2)
    x = x.contiguous() if layout == "nchw" else x
    seen, real = [], fused.srnl_spatial_inference
    fused.srnl_spatial_inference = lambda m, xs, q, *rest: seen.append(q) or real(m, xs, q, *rest)
    try:
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            op(x)
    finally:
        fused.srnl_spatial_inference = real
    q, = seen
    x64, w64 = x.permute(0, 2, 3, 1).double(), op.W_q.weight.detach().double()
    b64 = op.W_q.bias.detach().double() if bias else torch.zeros(dim, device=device, dtype=torch.float64)
    bound = 2.0 ** -8 * (x64.abs() @ w64.abs().T + b64.abs())
    assert q.dtype == torch.bfloat16 and ((q.double() - (x64 @ w64.T + b64)).abs() <= bound).all()
