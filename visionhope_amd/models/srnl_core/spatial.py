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

from .chunk import BACKWARD_MAX_CHUNK, srnl_consts
from .fused import srnl_spatial_readout, srnl_spatial_workspace
from ...utils import hip
from ...utils.cached_params import as_fp32
from ...utils.cuda import on_tensor_device
from ...utils.pointwise import EPI_ADD, EPI_BIAS

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
        ctx.save_for_backward(*memories, x, q, d_skip, weights, gains if keeps_gains(x, gains) else None)
        ctx.chunks = chunks
        return out

    @staticmethod
    def backward(ctx, dout):
        *memories, x, q, d_skip, weights, gains = ctx.saved_tensors
        return (*srnl_spatial_backward(memories, x, q, d_skip, weights, ctx.chunks, gains, dout), None)


# Bytes of chunk gains per map element that a step keeps for its backward, at most.  A chunk of
# c tokens leaves 16 d / c (four directions, d x d FP32 per head), so this covers chunks from 4
# tokens at head_dim 16 and 7 at head_dim 32, the smallest maps of the backbones.  What would be
# more (512 bytes for single-token chunks at head_dim 32, against 4 of a bf16 map and its
# queries) the backward forms again: 6 x 6 x 256 maps, batch 128, d = 32, 101 MB of gains, 277
# -> 374 us.
KEPT_GAIN_BYTES = 80


def keeps_gains(x, gains):
    return gains.numel() * 4 <= KEPT_GAIN_BYTES * x.numel()


@on_tensor_device
def srnl_spatial_gains(memories, x, chunks):
    """The products of the chunk gains that the backward starts from, and the workspace that
    ``srnl_spatial_readout`` reads (the content memories at the chunk starts)."""
    batch, height, width, channels = x.shape
    head_dim = memories[0].shape[-1]
    states = [as_fp32(m) for m in memories]
    x_c = x.contiguous()
    lib = hip.load_library()
    chunk_ptr, _keep = hip.int64_array(chunks)
    gains = hip.workspace(lib.vh_srnl_spatial_gains_bytes(batch, height, width, channels, head_dim, chunk_ptr), x.device)
    ws = srnl_spatial_workspace(x_c, head_dim, chunks)
    hip.check(lib.vh_srnl_spatial_gains(
        x_c.data_ptr(), hip.dtype_code(x.dtype), *[m.data_ptr() for m in states], batch, height, width, channels,
        head_dim, chunk_ptr, srnl_consts(), gains.data_ptr(), gains.numel() * 4, ws.data_ptr(), ws.numel() * 4,
        hip.stream_of(x_c)), "vh_srnl_spatial_gains")
    return gains, ws


def srnl_spatial_training_forward(memories, x, q, d_skip, weights, chunks):
    """The operator's output ``[B, H, W, C]`` FP32 and the gains its backward starts from."""
    gains, ws = srnl_spatial_gains(memories, x, chunks)
    return srnl_spatial_readout(ws, x, q, d_skip, weights, chunks, memories[0].shape[-1]), gains


@on_tensor_device
def srnl_spatial_backward(memories, x, q, d_skip, weights, chunks, gains, dout):
    """Gradients of ``SpatialSRNLFunction`` for the output gradient ``dout [B, H, W, C]`` and
    the ``gains`` of its forward (None: formed again): the five memories, x, q, d_skip and the
    weights, each shaped and typed like its input."""
    batch, height, width, channels = x.shape
    head_dim = memories[0].shape[-1]
    states = [as_fp32(m) for m in memories]
    if gains is None:
        gains = srnl_spatial_gains(memories, x, chunks)[0]
    # saved tensors come back from hooks with whatever strides those give them
    x_c, q_c, g, gains = x.contiguous(), q.contiguous(), as_fp32(dout), gains.contiguous()
    skip, wts = as_fp32(d_skip), as_fp32(weights)
    dx, dq = torch.empty_like(x_c), torch.empty_like(q_c)
    grads = [torch.empty_like(t) for t in (*states, skip, wts)]
    lib = hip.load_library()
    chunk_ptr, _keep = hip.int64_array(chunks)
    io = hip.dtype_code(x.dtype)
    nbytes = lib.vh_srnl_spatial_backward_workspace_bytes(batch, height, width, channels, head_dim, io, chunk_ptr)
    if nbytes == 0:
        raise ValueError(f"spatial SRNL backward does not cover head_dim={head_dim} with chunks {tuple(chunks)}")
    ws = hip.workspace(nbytes, x.device)
    hip.check(lib.vh_srnl_spatial_backward(
        x_c.data_ptr(), q_c.data_ptr(), io, g.data_ptr(), *[m.data_ptr() for m in states], skip.data_ptr(),
        int(skip.numel() == 4 * channels), wts.data_ptr(), gains.data_ptr(), dx.data_ptr(), dq.data_ptr(),
        *[d.data_ptr() for d in grads], batch, height, width, channels, head_dim, chunk_ptr, srnl_consts(),
        ws.data_ptr(), ws.numel() * 4, hip.stream_of(x_c)), "vh_srnl_spatial_backward")
    grads = [d.view(t.shape).to(t.dtype) for d, t in zip(grads, (*memories, d_skip, weights))]
    return (*grads[:5], dx, dq, *grads[5:])


def projected_training_supported(x_nhwc, linear):
    """Whether ``srnl_spatial_projected`` takes x and the query projection ``linear``: what
    bf16 autocast makes of an FP32 Linear, at the widths of the 1x1 convolution kernel."""
    w, b = linear.weight, linear.bias
    return (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16
            and x_nhwc.dtype == torch.bfloat16 and (x_nhwc.data_ptr() % 16 == 0 or not x_nhwc.is_contiguous())
            and type(w) is torch.nn.Parameter and type(b) is torch.nn.Parameter
            and w.dtype == b.dtype == torch.float32 and w.device == b.device == x_nhwc.device
            and w.shape == (x_nhwc.shape[-1],) * 2 and b.shape == w.shape[:1] and x_nhwc.shape[-1] % 32 == 0)


class ProjectedSpatialSRNLFunction(torch.autograd.Function):
    """``SpatialSRNLFunction`` of q = x W^T + b under bf16 autocast, x ``[B, H, W, C]``
    contiguous bf16 (``projected_training_supported``), with the projection's own gradients:
    dx gains dq W in the product's epilogue, dW and db come from one pass over the maps.

    Autocast's linear rounds W, b and q to bf16, and so does this; its weight gradients are
    FP32 sums rounded to bf16 on the way, these are not."""

    @staticmethod
    def forward(ctx, M_m_0, M_v_0, M_k_0, M_eta_0, M_alpha_0, x, w, b, d_skip, weights, chunks):
        if torch.jit.is_tracing():
            raise RuntimeError("SRNL TorchScript tracing is unsupported; use eager or CUDA Graph inference.")
        memories = (M_m_0, M_v_0, M_k_0, M_eta_0, M_alpha_0)
        operands, q = project_queries(x, w, b)
        out, gains = srnl_spatial_training_forward(memories, x, q, d_skip, weights, chunks)
        ctx.save_for_backward(*memories, x, q, operands, d_skip, weights, gains if keeps_gains(x, gains) else None)
        ctx.chunks = chunks
        return out

    @staticmethod
    def backward(ctx, dout):
        *memories, x, q, operands, d_skip, weights, gains = ctx.saved_tensors
        *dmem, dx, dq, dskip, dweights = srnl_spatial_backward(memories, x, q, d_skip, weights, ctx.chunks, gains, dout)
        needs = ctx.needs_input_grad
        dx, dw, db = project_queries_backward(x, operands, dx, dq, needs[5], needs[6] or needs[7])
        return (*dmem, dx, dw, db, dskip, dweights, None)


@on_tensor_device
def project_queries(x, w, b):
    """The projection's bf16 operands (W, W^T and b, in one buffer) and the queries."""
    channels = x.shape[-1]
    w, b = as_fp32(w), as_fp32(b)
    operands = torch.empty((2 * channels + 2, channels), device=x.device, dtype=torch.bfloat16)
    q = torch.empty_like(x)
    lib, base, half = hip.load_library(), operands.data_ptr(), 2 * channels * channels
    stream = hip.stream_of(x)
    hip.check(lib.vh_linear_operands(w.data_ptr(), b.data_ptr(), hip.VH_DTYPE_F32, channels, channels, base, base + half,
                                     base + 2 * half, stream), "vh_linear_operands")
    hip.check(lib.vh_pointwise_conv_nhwc_forward(
        x.data_ptr(), hip.VH_DTYPE_BF16, base, base + 2 * half, EPI_BIAS, None, None, None, 0, q.data_ptr(),
        x.numel() // channels, channels, channels, stream), "vh_pointwise_conv_nhwc_forward")
    return operands, q


@on_tensor_device
def project_queries_backward(x, operands, dx, dq, need_dx, need_params):
    """dx + dq W (or None), dW and db (or None) of ``project_queries``."""
    channels = x.shape[-1]
    x, operands = x.contiguous(), operands.contiguous()
    tokens, lib, stream = x.numel() // channels, hip.load_library(), hip.stream_of(x)
    total = dw = db = None
    if need_dx:
        total = torch.empty_like(x)
        hip.check(lib.vh_pointwise_conv_nhwc_forward(
            dq.data_ptr(), hip.VH_DTYPE_BF16, operands.data_ptr() + 2 * channels * channels, None, EPI_ADD,
            dx.data_ptr(), None, None, 0, total.data_ptr(), tokens, channels, channels, stream),
            "vh_pointwise_conv_nhwc_forward")
    if need_params:
        dw = torch.empty((channels, channels), device=x.device, dtype=torch.float32)
        db = torch.empty(channels, device=x.device, dtype=torch.float32)
        ws = hip.workspace(lib.vh_linear_weight_grad_workspace_bytes(tokens, channels, channels), x.device)
        hip.check(lib.vh_linear_weight_grad(dq.data_ptr(), x.data_ptr(), tokens, channels, channels, dw.data_ptr(),
                                            db.data_ptr(), ws.data_ptr(), ws.numel() * 4, stream),
                  "vh_linear_weight_grad")
    return total, dw, db


def _check_merge(x_nhwc, d_skip, weights):
    if weights.shape != (4, x_nhwc.shape[-1]) or d_skip.numel() not in (weights.numel(), x_nhwc.shape[-1]):
        raise RuntimeError("d_skip must contain C or 4*C values and the direction weights 4*C")


def srnl_spatial(memories, x_nhwc, q_nhwc, d_skip, weights, chunks):
    """Differentiable spatial operator (``spatial_training_supported``).  The Function runs
    without gradients too: it is what refuses tracing and forward-mode derivatives, and a
    checkpointed step repeats its forward with the same kernels."""
    _check_merge(x_nhwc, d_skip, weights)
    return SpatialSRNLFunction.apply(*memories, x_nhwc, q_nhwc, d_skip, weights, tuple(int(c) for c in chunks))


def srnl_spatial_projected(memories, x_nhwc, linear, d_skip, weights, chunks):
    """``srnl_spatial`` of the queries ``linear(x_nhwc)`` (``projected_training_supported``)."""
    _check_merge(x_nhwc, d_skip, weights)
    return ProjectedSpatialSRNLFunction.apply(*memories, x_nhwc, linear.weight, linear.bias, d_skip, weights,
                                              tuple(int(c) for c in chunks))
