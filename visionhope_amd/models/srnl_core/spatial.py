"""The four-direction operator on channels-last maps, with autograd.

``srnl_spatial`` is what a training step of the operator runs where the spatial kernels
apply: a scan in FP32 products that keeps the chunk gains (``vh_srnl_spatial_gains``), the
fused readout of the inference path, and a backward (``vh_srnl_spatial_backward``) that
starts from those gains, all reading and writing maps at their pixels; the four directions'
gradients are summed in one pass.  The packed path it replaces serialises x and the queries into
four scan orders, scans, reads out, restores and fuses in separate passes (reference
``operator.py:88-145``), each with its transposed pass in the backward.
"""

import torch

from .chunk import BACKWARD_MAX_CHUNK, _float_memories, srnl_consts
from .fused import srnl_spatial_inference, srnl_spatial_readout, srnl_spatial_workspace
from ...utils import hip
from ...utils.cuda import on_tensor_device

# Head dims of the block-form backward.
SPATIAL_BACKWARD_HEAD_DIMS = (16, 32)


def spatial_training_supported(x, q, head_dim, chunks):
    """Whether ``srnl_spatial`` takes an NCHW map x and queries q of its dtype."""
    return (x.is_cuda and q.device == x.device and q.dtype == x.dtype
            and x.dtype in (torch.float16, torch.bfloat16, torch.float32)
            and min(x.shape) > 0 and x.shape[2] * x.shape[3] < (1 << 24)
            and head_dim in SPATIAL_BACKWARD_HEAD_DIMS and max(chunks) <= BACKWARD_MAX_CHUNK)


class SpatialSRNLFunction(torch.autograd.Function):
    """``[B, H, W, C]`` FP32 = sum_r w_r (y_r + skip_r x) from x, q ``[B, H, W, C]``; FP32
    d_skip (C or 4 C values) and weights ``[4, C]``; one chunk length per direction."""

    @staticmethod
    def forward(ctx, M_m_0, M_v_0, M_k_0, M_eta_0, M_alpha_0, x, q, d_skip, weights, chunks):
        if torch.jit.is_tracing():
            raise RuntimeError("SRNL TorchScript tracing is unsupported; use eager or CUDA Graph inference.")
        memories = (M_m_0, M_v_0, M_k_0, M_eta_0, M_alpha_0)
        out, gains = srnl_spatial_training_forward(memories, x, q, d_skip, weights, chunks)
        ctx.save_for_backward(*memories, x, q, d_skip, weights, gains)
        ctx.chunks = chunks
        return out

    @staticmethod
    def backward(ctx, dout):
        *memories, x, q, d_skip, weights, gains = ctx.saved_tensors
        return (*srnl_spatial_backward(memories, x, q, d_skip, weights, ctx.chunks, gains, dout), None)


@on_tensor_device
def srnl_spatial_training_forward(memories, x, q, d_skip, weights, chunks):
    """The operator's output ``[B, H, W, C]`` FP32 and the gains its backward starts from."""
    batch, height, width, channels = x.shape
    head_dim = memories[0].shape[-1]
    heads = channels // head_dim
    states, _ = _float_memories(memories, 4, heads, head_dim, batch * 4 * heads)
    x_c = x.contiguous()
    lib = hip.load_library()
    chunk_ptr, _keep = hip.int64_array(chunks)
    gains = hip.workspace(lib.vh_srnl_spatial_gains_bytes(batch, height, width, channels, head_dim, chunk_ptr), x.device)
    ws = srnl_spatial_workspace(x_c, head_dim, chunks)
    hip.check(lib.vh_srnl_spatial_gains(
        hip.ptr(x_c), hip.dtype_code(x.dtype), *[hip.ptr(m) for m in states], batch, height, width, channels, head_dim,
        chunk_ptr, srnl_consts(), hip.ptr(gains), gains.numel() * 4, hip.ptr(ws), ws.numel() * 4,
        hip.stream_of(x_c)), "vh_srnl_spatial_gains")
    return srnl_spatial_readout(ws, x_c, q, d_skip, weights, chunks, head_dim), gains


@on_tensor_device
def srnl_spatial_backward(memories, x, q, d_skip, weights, chunks, gains, dout):
    """Gradients of ``SpatialSRNLFunction`` for the output gradient ``dout [B, H, W, C]`` and
    the ``gains`` of its forward: the five memories, x, q, d_skip and the weights, each
    shaped and typed like its input."""
    batch, height, width, channels = x.shape
    head_dim = memories[0].shape[-1]
    heads = channels // head_dim
    states, _ = _float_memories(memories, 4, heads, head_dim, batch * 4 * heads)
    x_c, q_c = x.contiguous(), q.contiguous()
    g = dout.float().contiguous()
    skip = d_skip.detach().float().contiguous()
    wts = weights.detach().float().contiguous()
    dx, dq = torch.empty_like(x_c), torch.empty_like(q_c)
    dmem = [torch.empty_like(m) for m in states]
    dskip, dweights = torch.empty_like(skip), torch.empty_like(wts)
    lib = hip.load_library()
    chunk_ptr, _keep = hip.int64_array(chunks)
    io = hip.dtype_code(x.dtype)
    nbytes = lib.vh_srnl_spatial_backward_workspace_bytes(batch, height, width, channels, head_dim, io, chunk_ptr)
    if nbytes == 0:
        raise ValueError(f"spatial SRNL backward does not cover head_dim={head_dim} with chunks {tuple(chunks)}")
    ws = hip.workspace(nbytes, x.device)
    hip.check(lib.vh_srnl_spatial_backward(
        hip.ptr(x_c), hip.ptr(q_c), io, hip.ptr(g), *[hip.ptr(m) for m in states], hip.ptr(skip),
        int(skip.numel() == 4 * channels), hip.ptr(wts), hip.ptr(gains), hip.ptr(dx), hip.ptr(dq), *[hip.ptr(m) for m in dmem],
        hip.ptr(dskip), hip.ptr(dweights), batch, height, width, channels, head_dim, chunk_ptr, srnl_consts(),
        hip.ptr(ws), ws.numel() * 4, hip.stream_of(x_c)), "vh_srnl_spatial_backward")
    grads = [d.view(m.shape).to(m.dtype) for d, m in zip(dmem, memories)]
    return (*grads, dx, dq, dskip.view(d_skip.shape).to(d_skip.dtype), dweights.view(weights.shape).to(weights.dtype))


def srnl_spatial(memories, x_nhwc, q_nhwc, d_skip, weights, chunks):
    """Differentiable spatial operator (``spatial_training_supported``)."""
    if weights.shape != (4, x_nhwc.shape[-1]) or d_skip.numel() not in (weights.numel(), x_nhwc.shape[-1]):
        raise RuntimeError("d_skip must contain C or 4*C values and the direction weights 4*C")
    if not (torch.is_grad_enabled() and any(t.requires_grad for t in (*memories, x_nhwc, q_nhwc, d_skip, weights))):
        # nothing to differentiate: the inference scan, which keeps nothing
        if torch.jit.is_tracing():
            raise RuntimeError("SRNL TorchScript tracing is unsupported; use eager or CUDA Graph inference.")
        return srnl_spatial_inference(memories, x_nhwc, q_nhwc, d_skip, weights, chunks)
    return SpatialSRNLFunction.apply(*memories, x_nhwc, q_nhwc, d_skip, weights, tuple(int(c) for c in chunks))
