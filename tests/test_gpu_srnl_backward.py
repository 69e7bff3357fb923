"""GPU parity of the SRNL backward (vh_srnl_backward) against autograd of the float64
PyTorch oracle (itself pinned by finite differences in test_oracle_backward.py)."""

import numpy as np
import pytest
import torch

from tests.helpers import assert_close, memories, randn

pytestmark = pytest.mark.gpu

GRAD_TOL = 2e-3   # fp32 recurrence and reductions against float64, relative to each gradient's scale


def _oracle_grads(x, q, mems, chunks, dy, q_raw):
    from oracle.oracle_torch import sequence_forward_torch

    xs = x.double().requires_grad_()
    qs = q.double().requires_grad_()
    ms = [torch.from_numpy(m).double().requires_grad_() for m in mems]
    y = sequence_forward_torch(xs, qs, ms, chunks, q_raw=q_raw)
    (y * dy.double()).sum().backward()
    return [m.grad.numpy() for m in ms] + [xs.grad.numpy(), qs.grad.numpy()]


def _check(got, want, what, tol=GRAD_TOL):
    names = ["dM_m", "dM_v", "dM_k", "dM_eta", "dM_alpha", "dx", "dq"]
    for name, g, w in zip(names, got, want):
        assert g.shape == w.shape, f"{what} {name} shape"
        assert_close(g.detach().double().cpu().numpy(), w, tol, f"{what} {name}")


@pytest.mark.parametrize("head_dim", [4, 8, 16, 32])
@pytest.mark.parametrize("q_raw", [True, False])
@pytest.mark.parametrize("kind", ["perturbed", "strong"])
def test_srnl_backward_matches_oracle(device, head_dim, q_raw, kind):
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads, length = 2, 4, 2, 23
    chunks = [5, 7, 4, 9]                   # ragged last chunks, one length per direction
    mems = memories(directions, heads, head_dim, kind=kind, seed=head_dim + (7 if q_raw else 0))
    x = randn(batch, directions, heads, length, head_dim, seed=3)
    if q_raw:
        q = randn(batch, directions, length, heads * head_dim, seed=4)
    else:
        q = randn(batch, directions, heads, length, head_dim, seed=4)
        q = q / q.norm(dim=-1, keepdim=True)
    dy = randn(batch, directions, heads, length, head_dim, seed=5)
    want = _oracle_grads(x, q, mems, chunks, dy, q_raw)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=q_raw)
    _check(got, want, f"d={head_dim} q_raw={q_raw} {kind}")


@pytest.mark.parametrize("heads", [4, 8])
@pytest.mark.parametrize("head_dim", [4, 8, 16])
@pytest.mark.parametrize("q_raw", [True, False])
def test_srnl_backward_packed_lines_match_oracle(device, heads, head_dim, q_raw):
    """Head counts divisible by 4 run the variant that packs 4 lines (consecutive heads of
    one image and direction) into a workgroup for head_dim 4, 8 and 16 with chunks of 64
    or less; raw and normalised queries, ragged chunks, perturbed memories."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, length = 2, 4, 21
    chunks = [6, 4, 8, 5]
    mems = memories(directions, heads, head_dim, kind="perturbed", seed=100 + heads + head_dim)
    x = randn(batch, directions, heads, length, head_dim, seed=31)
    if q_raw:
        q = randn(batch, directions, length, heads * head_dim, seed=32)
    else:
        q = randn(batch, directions, heads, length, head_dim, seed=32)
        q = q / q.norm(dim=-1, keepdim=True)
    dy = randn(batch, directions, heads, length, head_dim, seed=33)
    want = _oracle_grads(x, q, mems, chunks, dy, q_raw)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=q_raw)
    _check(got, want, f"heads={heads} d={head_dim} q_raw={q_raw}")


def test_srnl_backward_tiny_stage3_shape(device):
    """The Tiny stage-3 operator shape the packed variant trains on: 8 heads of d = 16 on
    a 14 x 14 map (196-token lines, chunks of 14), one image, raw queries."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads, length, d = 1, 4, 8, 196, 16
    chunks = [14, 14, 14, 14]
    mems = memories(directions, heads, d, kind="perturbed", seed=77)
    x = randn(batch, directions, heads, length, d, seed=34)
    q = randn(batch, directions, length, heads * d, seed=35)
    dy = randn(batch, directions, heads, length, d, seed=36)
    want = _oracle_grads(x, q, mems, chunks, dy, True)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=True)
    _check(got, want, "Tiny stage 3")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_srnl_backward_low_precision_inputs(device, dtype):
    """bf16 / fp16 x and raw q: the kernel reads the rounded values and computes in fp32;
    the oracle differentiates at the same rounded values."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads, length, d = 2, 4, 2, 30, 16
    chunks = [6, 6, 10, 10]
    mems = memories(directions, heads, d, kind="perturbed", seed=21)
    x = randn(batch, directions, heads, length, d, seed=22).to(dtype)
    q = randn(batch, directions, length, heads * d, seed=23).to(dtype)
    dy = randn(batch, directions, heads, length, d, seed=24)
    want = _oracle_grads(x.float(), q.float(), mems, chunks, dy, True)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=True)
    assert got[5].dtype == dtype and got[6].dtype == dtype
    _check([g.float() for g in got], want, f"{dtype}", tol=1e-2)   # dx, dq returned rounded to the input dtype


def test_srnl_backward_per_line_memories(device):
    """5-D memories (one state per line): the per-line gradients are not summed."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads, length, d = 2, 4, 1, 17, 8
    chunks = [4, 4, 4, 4]
    shared = memories(directions, heads, d, kind="strong", seed=31)
    gen = np.random.default_rng(32)
    mems = tuple(np.ascontiguousarray(np.stack([m + 0.05 * gen.standard_normal(m.shape).astype(np.float32)
                                                for _ in range(batch)]), dtype=np.float32) for m in shared)
    x = randn(batch, directions, heads, length, d, seed=33)
    q = randn(batch, directions, length, heads * d, seed=34)
    dy = randn(batch, directions, heads, length, d, seed=35)
    # oracle: per-line states as lines of one batch each
    from oracle.oracle_torch import srnl_lines_torch
    n = batch * directions * heads
    xs = x.double().requires_grad_()
    qs = q.double().requires_grad_()
    ms = [torch.from_numpy(m).double().requires_grad_() for m in mems]
    q_lines = qs.reshape(batch, directions, length, heads, d).permute(0, 1, 3, 2, 4).reshape(n, length, d)
    y = srnl_lines_torch(xs.reshape(n, length, d), q_lines,
                         [m.reshape((n,) + tuple(m.shape[3:])) for m in ms], list(range(n)), [4] * n)
    (y.reshape(dy.shape) * dy.double()).sum().backward()
    want = [m.grad.numpy() for m in ms] + [xs.grad.numpy(), qs.grad.numpy()]
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=True)
    _check(got, want, "per-line memories")


def test_srnl_raw_query_function_backward(device):
    """Through the autograd Function (the module's ordinary path): gradients land on the
    parameters and inputs with their shapes and dtypes."""
    from visionhope_amd.models.srnl_core.chunk import srnl_raw_query

    batch, heads, length, d = 2, 2, 20, 16
    mems = [torch.from_numpy(m).to(device).requires_grad_() for m in memories(4, heads, d, kind="perturbed", seed=41)]
    x = randn(batch, 4, heads, length, d, seed=42).to(device).requires_grad_()
    q = randn(batch, 4, length, heads * d, seed=43).to(device).requires_grad_()
    y = srnl_raw_query(*mems, x, q, 6, heads, d)
    dy = randn(*y.shape, seed=44).to(device)
    (y * dy).sum().backward()
    want = _oracle_grads(x.detach().cpu(), q.detach().cpu(), [m.detach().cpu().numpy() for m in mems], [6] * 4,
                         dy.cpu(), True)
    _check([m.grad for m in mems] + [x.grad, q.grad], want, "autograd Function")


def test_srnl_backward_rejects(device):
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    mems = tuple(torch.from_numpy(m).to(device) for m in memories(4, 1, 16, seed=51))
    x = torch.zeros(1, 4, 1, 270, 16, device=device)
    q = torch.zeros(1, 4, 270, 16, device=device)
    with pytest.raises(ValueError):
        srnl_packed_backward(mems, x, q, [257, 8, 8, 8], torch.zeros_like(x), q_raw=True)   # chunk > 256


@pytest.mark.parametrize("head_dim,chunks,length", [(16, [100, 100, 65, 65], 230), (32, [128, 128, 128, 128], 300),
                                                    (8, [256, 3, 256, 3], 260)])
def test_srnl_backward_long_chunks(device, head_dim, chunks, length):
    """Chunks of 65 to 256 tokens (the long-line range; 256-token LDS buffers), mixed with
    short chunks in other directions, ragged last chunks."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads = 1, 4, 2
    mems = memories(directions, heads, head_dim, kind="perturbed", seed=head_dim + 61)
    x = randn(batch, directions, heads, length, head_dim, seed=62, scale=0.5)
    q = randn(batch, directions, length, heads * head_dim, seed=63)
    dy = randn(batch, directions, heads, length, head_dim, seed=64)
    want = _oracle_grads(x, q, mems, chunks, dy, True)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=True)
    _check(got, want, f"d={head_dim} chunks={chunks}")


def test_srnl_long_chunk_function_backward(device):
    """Through the long-chunk autograd Function (chunk 96 > 64)."""
    from visionhope_amd.models.srnl_core.lines import srnl_long_chunk

    batch, heads, length, d = 1, 2, 200, 16
    mems = [torch.from_numpy(m).to(device).requires_grad_() for m in memories(4, heads, d, kind="perturbed", seed=71)]
    x = randn(batch, 4, heads, length, d, seed=72, scale=0.5).to(device).requires_grad_()
    q = randn(batch, 4, length, heads * d, seed=73).to(device).requires_grad_()
    y = srnl_long_chunk(*mems, x, q, 96, heads, d)
    dy = randn(*y.shape, seed=74).to(device)
    (y * dy).sum().backward()
    want = _oracle_grads(x.detach().cpu(), q.detach().cpu(), [m.detach().cpu().numpy() for m in mems], [96] * 4,
                         dy.cpu(), True)
    _check([m.grad for m in mems] + [x.grad, q.grad], want, "long-chunk Function")


@pytest.mark.parametrize("head_dim", [4, 8, 16])
@pytest.mark.parametrize("heads", [2, 4, 8])
@pytest.mark.parametrize("q_raw", [True, False])
def test_srnl_backward_lines_per_workgroup(device, head_dim, heads, q_raw):
    """Both launch shapes of the backward: heads % 4 == 0 packs 4 lines (consecutive heads of
    one image and direction) into a workgroup at d <= 16, otherwise 1 line per workgroup.
    Ragged last chunks, one length per direction."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, length = 2, 4, 19
    chunks = [6, 4, 7, 5]
    mems = memories(directions, heads, head_dim, kind="perturbed", seed=100 + heads * head_dim)
    x = randn(batch, directions, heads, length, head_dim, seed=101)
    if q_raw:
        q = randn(batch, directions, length, heads * head_dim, seed=102)
    else:
        q = randn(batch, directions, heads, length, head_dim, seed=102)
        q = q / q.norm(dim=-1, keepdim=True)
    dy = randn(batch, directions, heads, length, head_dim, seed=103)
    want = _oracle_grads(x, q, mems, chunks, dy, q_raw)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               chunks, dy.to(device), q_raw=q_raw)
    _check(got, want, f"d={head_dim} heads={heads} q_raw={q_raw}")


def test_srnl_backward_tiny_stage3_shape(device):
    """The Tiny stage-3 operator's lines (8 heads of 16, 14x14 map, chunks of 14: the shape
    the packed variant trains on), at batch 2, bf16 inputs as under autocast."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    batch, directions, heads, d, length = 2, 4, 8, 16, 196
    mems = memories(directions, heads, d, kind="perturbed", seed=111)
    x = randn(batch, directions, heads, length, d, seed=112).bfloat16()
    q = randn(batch, directions, length, heads * d, seed=113).bfloat16()
    dy = randn(batch, directions, heads, length, d, seed=114)
    want = _oracle_grads(x.float(), q.float(), mems, [14] * 4, dy, True)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                               [14] * 4, dy.to(device), q_raw=True)
    _check([g.float() for g in got], want, "Tiny stage 3", tol=1e-2)


def _block_form_case(device, head_dim, chunks, length, *, heads=1, batch=1, dtype=torch.float32, kind="perturbed",
                     gate_scale=1.0, offset=0, q_raw=True):
    """Gradients of random lines and the tolerance for them: every gradient is a sum of
    products along at most one chunk (the gains never expand), so an FP32 evaluation is
    within (chunk + 4 d) roundings of 2^-24, doubled, of the gradient's scale; 16-bit inputs
    round the returned dx and dq once more (2^-8 for bf16, 2^-11 for fp16)."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_backward

    def place(t):
        """t on the GPU, starting ``offset`` elements into its storage."""
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        flat[offset:] = t.reshape(-1).to(device)
        return flat[offset:].view(t.shape)

    directions = len(chunks)
    mems = list(memories(directions, heads, head_dim, kind=kind, seed=head_dim + 201))
    mems[3:] = [m * gate_scale for m in mems[3:]]
    x = randn(batch, directions, heads, length, head_dim, seed=202).to(dtype)
    q = (randn(batch, directions, length, heads * head_dim, seed=203).to(dtype) if q_raw else
         torch.nn.functional.normalize(randn(batch, directions, heads, length, head_dim, seed=203), dim=-1))
    dy = randn(batch, directions, heads, length, head_dim, seed=204)
    want = _oracle_grads(x.float(), q.float(), mems, chunks, dy, q_raw)
    got = srnl_packed_backward(tuple(torch.from_numpy(m).to(device) for m in mems), place(x), place(q), chunks,
                               place(dy), q_raw=q_raw)
    tol = 2.0 ** -23 * (max(chunks) + 4 * head_dim)
    rounding = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    what = f"d={head_dim} chunks={chunks} {dtype}"
    _check(got[:5], want[:5], what, tol)
    for name, g, w in zip(("dx", "dq"), got[5:], want[5:]):
        assert_close(g.double().cpu().numpy(), w, tol + rounding, f"{what} {name}")


@pytest.mark.parametrize("head_dim,chunks,length", [
    (16, [1, 2, 15, 16], 35), (16, [17, 31, 32, 33], 70), (16, [63, 64, 65, 3], 140), (16, [127, 128, 129, 16], 290),
    (16, [256, 200, 255, 130], 530), (16, [39, 40, 64, 128], 40), (32, [1, 15, 16, 7], 33), (32, [17, 32, 33, 48], 100),
    (32, [64, 65, 100, 128], 210), (32, [256, 129, 192, 16], 520)])
def test_srnl_backward_block_edges(device, head_dim, chunks, length):
    """The block-form kernels (head_dim 16 and 32) around their tile, wave-count and segment
    edges: 1, 2, 4 or 8 waves, chunks of one slot to several segments, ragged last chunks,
    directions with fewer blocks than waves, and lines of a single chunk."""
    _block_form_case(device, head_dim, chunks, length, heads=2)


@pytest.mark.parametrize("head_dim,chunks,length", [(16, [97, 112, 96, 81], 230), (16, [65, 80, 33, 48], 170),
                                                    (32, [33, 48, 32, 17], 100)])
def test_srnl_backward_spare_waves(device, head_dim, chunks, length):
    """7, 6, 5 and 3 blocks on 8 waves, 3 and 2 on 4: few spare waves leave the readout's
    gradients to the waves of their blocks, more of them take them all."""
    _block_form_case(device, head_dim, chunks, length, heads=2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim,directions", [(16, 1), (32, 2)])
def test_srnl_backward_block_inputs(device, head_dim, directions, dtype):
    """Every activation type, tensors that start at an odd element of their storage, one and
    two directions, and saturated gates with strong memories (retentions down to the clamp)."""
    chunks = [19, 40][:directions]
    _block_form_case(device, head_dim, chunks, 90, heads=3, batch=2, dtype=dtype, offset=1)
    _block_form_case(device, head_dim, chunks, 90, dtype=dtype, kind="strong", gate_scale=4.0, offset=3, q_raw=False)


@pytest.mark.parametrize("head_dim", [16, 32])
def test_retention_products_of_saturated_gates(device, head_dim):
    """The gain of a chunk of 16 tokens whose keys are zero is the product of its retentions
    times the identity: 2^-100 here, in every entry within the roundings of 16 gates (three
    each: the exponential, the sum and the reciprocal) and of the five products.  As a
    difference of sums of logarithms it would carry 2^-24 of 100."""
    from visionhope_amd.models.srnl_core import chunk
    from visionhope_amd.models.srnl_core.spatial import srnl_spatial_training_forward

    heads, tokens, batch = 4, 16, 8
    channels = heads * head_dim
    gen = torch.Generator().manual_seed(head_dim)
    gates = -7.0 + torch.rand(4, heads, head_dim, generator=gen)
    mats = [torch.randn(4, heads, head_dim, head_dim, generator=gen), *torch.zeros(2, 4, heads, head_dim, head_dim)]
    # token t of a row selects gate entry perm[t]; two rows, so that a second chunk exists
    perms = torch.stack([torch.randperm(head_dim, generator=gen)[:tokens] for _ in range(batch * heads)])
    x = torch.zeros(batch, 2, tokens, heads, head_dim)
    for i, perm in enumerate(perms):
        x[i // heads, :, torch.arange(tokens), i % heads, perm] = 1.0
    x = x.reshape(batch, 2, tokens, channels)
    mems = [m.to(device) for m in (*mats, torch.zeros_like(gates), gates)]
    _, gains = srnl_spatial_training_forward(mems, x.to(device), x.to(device), torch.zeros(channels, device=device),
                                             torch.ones(4, channels, device=device), (tokens,) * 4)
    gains = gains.cpu()[:batch * 4 * heads * 2 * head_dim ** 2].double()
    got = gains.reshape(batch, 4, heads, 2, head_dim, head_dim)[:, 0, :, 1]
    bias = np.float32(chunk.RETENTION_BIAS)
    for i, perm in enumerate(perms):
        pre = (gates[0, i % heads, perm].numpy() + bias).astype(np.float64)
        retention = chunk.MIN_RETENTION + (1 - chunk.MIN_RETENTION) / (1 + np.exp(-pre))
        want = torch.eye(head_dim, dtype=torch.float64) * retention.prod()
        bound = (3 * tokens + 5) * 2.0 ** -24 * retention.prod()
        assert (got[i // heads, i % heads] - want).abs().max() <= bound
