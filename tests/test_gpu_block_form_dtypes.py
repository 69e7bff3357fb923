"""The block-form scans (srnl_ut.hip, srnl_utw.hip, srnl_utw32.hip) on fp16 and FP32
activations, through the spatial operator (``vh_srnl_spatial_forward``, FP32 output) and
the sequence entry, against the C oracle on the same inputs.

Each shape runs the library's own dispatch: one workgroup per line with a chunk's blocks over
1 or 2 waves (head_dim 16: chunks of one block, or few lines), the packed one-wave form (longer
chunks from 2,048 lines, unaligned rows) and the head_dim-32 form with chunks of 14 and 56
tokens (1 and 4 waves).  fp16 values are exact as bf16 hi + lo
operands and FP32 values enter within 2^-16 of their value, so both are held to the bound of
the bf16 block form, 2e-5 (about one hi + lo rounding of the output, five times inside the
FP32 contract of 1e-4; observed on MI355X: 5e-8 normwise with default-scale memories, up to
9e-7 elementwise with strong ones).  The observed errors are printed (``pytest -s``).
"""

import pytest
import torch

from tests.helpers import max_rel_err, memories, randn, rel_err

pytestmark = pytest.mark.gpu

BLOCK_TOL = 2e-5     # FP32 output: the block form's own arithmetic
FP32_TOL = 1e-4      # the FP32 parity contract (the stepped and wide kernels under an override)
FP16_OUT_TOL = 2e-3  # fp16 output of the sequence entry: one fp16 rounding (2^-11) on top

# (batch, H = W, heads, head_dim): kernel chosen by the default dispatch
SHAPES = [
    (64, 14, 16, 16),   # 4096 lines, one block per chunk
    (32, 14, 8, 16),    # 1024 lines, one block per chunk
    (4, 28, 4, 16),     # 64 lines, chunks of 28: few-line form, 2 waves per line
    (8, 14, 4, 32),     # head_dim 32, chunks of 14: one wave per line
    (2, 56, 2, 32),     # head_dim 32, chunks of 56: four waves per line
]


def _spatial_case(batch, hw, heads, d, dtype, kind):
    channels = heads * d
    seed = batch * 1000 + hw * 10 + heads + d
    mems = memories(4, heads, d, kind=kind, seed=seed)
    x = randn(batch, hw, hw, channels, seed=seed + 1).to(dtype)
    q = randn(batch, hw, hw, channels, seed=seed + 2).to(dtype)
    skip = randn(channels, seed=seed + 3, scale=0.1)
    wts = 1 + randn(4, channels, seed=seed + 4, scale=0.1)
    return mems, x, q, skip, wts


@pytest.mark.parametrize("batch,hw,heads,d", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["perturbed", "strong"])
def test_block_form_spatial_fp16_fp32(oracle, device, batch, hw, heads, d, dtype, kind):
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    mems, x, q, skip, wts = _spatial_case(batch, hw, heads, d, dtype, kind)
    print(f"\n[case] spatial {dtype} B={batch} {hw}x{hw} heads={heads} d={d} lines={batch * 4 * heads} {kind}",
          flush=True)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                                 skip.to(device), wts.to(device), (hw,) * 4).cpu().numpy()
    expected = oracle.operator_forward(x.float().numpy(), q.float().numpy(), mems, skip.numpy(), wts.numpy(), d)
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    print(f"[err] {dtype} {hw}x{hw} d={d} {kind}: normwise {r:.2e} elementwise {m:.2e}", flush=True)
    assert r <= BLOCK_TOL and m <= BLOCK_TOL, f"{dtype} {hw}x{hw} d={d} {kind}: normwise {r:.3e}, elementwise {m:.3e}"


@pytest.mark.parametrize("head_dim,chunk", [(16, 14), (16, 64), (32, 14), (32, 49)])
@pytest.mark.parametrize("dtype,tol", [(torch.float16, FP16_OUT_TOL), (torch.float32, BLOCK_TOL)])
def test_block_form_sequence_fp16_fp32(oracle, device, head_dim, chunk, dtype, tol):
    """Packed sequences (the SRNL module's inference entry) of 196 tokens, 2 sequences, one
    direction, 2 heads (config 1's shape at head_dim 32), raw queries; y comes back in the
    input dtype (fp16: one rounding, 2^-11 relative, on top of the scan's error)."""
    from visionhope_amd.models.srnl_core.chunk import srnl_packed_forward

    batch, directions, heads, length = 2, 1, 2, 196
    seed = 7 * head_dim + chunk
    mems = memories(directions, heads, head_dim, kind="perturbed", seed=seed)
    x = randn(batch, directions, heads, length, head_dim, seed=seed + 1).to(dtype)
    q = randn(batch, directions, length, heads * head_dim, seed=seed + 2).to(dtype)
    print(f"\n[case] sequence {dtype} d={head_dim} chunk={chunk}", flush=True)
    got = srnl_packed_forward(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                              [chunk], q_raw=True)
    assert got.dtype == dtype
    expected = oracle.sequence_forward(x.float().numpy(), q.float().numpy(), mems, [chunk])
    got = got.float().cpu().numpy()
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    print(f"[err] sequence {dtype} d={head_dim} chunk={chunk}: normwise {r:.2e} elementwise {m:.2e}", flush=True)
    assert r <= tol and m <= tol, f"{dtype} d={head_dim} chunk={chunk}: normwise {r:.3e}, elementwise {m:.3e}"


@pytest.mark.parametrize("batch,hw,heads,d,forced", [
    (32, 14, 8, 16, {"scan_ut": 0}),      # stepped form, 1024 lines
    (4, 28, 4, 16, {"scan_wide": 2}),     # wide scan, 64 lines
    (8, 14, 4, 32, {"scan_utw": 0}),      # head_dim 32: wide scan
])
def test_fp32_forced_stepped_and_wide_forms(oracle, device, dispatch, batch, hw, heads, d, forced):
    """The kernels the block form replaced stay reachable for FP32 maps under an override."""
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    dispatch(**forced)
    mems, x, q, skip, wts = _spatial_case(batch, hw, heads, d, torch.float32, "strong")
    print(f"\n[case] forced {forced} FP32 B={batch} {hw}x{hw} d={d}", flush=True)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                                 skip.to(device), wts.to(device), (hw,) * 4).cpu().numpy()
    expected = oracle.operator_forward(x.numpy(), q.numpy(), mems, skip.numpy(), wts.numpy(), d)
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    print(f"[err] forced {forced}: normwise {r:.2e} elementwise {m:.2e}", flush=True)
    assert r <= FP32_TOL and m <= FP32_TOL, f"{forced}: normwise {r:.3e}, elementwise {m:.3e}"


@pytest.mark.parametrize("batch,height,width,heads", [
    (2, 1, 16, 1), (1, 17, 1, 2), (2, 16, 17, 1), (1, 31, 32, 2), (1, 33, 48, 1), (2, 49, 15, 1), (1, 64, 65, 1),
    (1, 5, 127, 2), (1, 128, 3, 1),      # 1 to 8 blocks per chunk, full, ragged and single-token, fewer blocks than waves
    (128, 16, 16, 4), (128, 17, 5, 4), (127, 17, 5, 4)])    # 2048 lines: one block per chunk, two, and just below
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_line_per_workgroup_scan_edges(oracle, device, batch, height, width, heads, dtype):
    """The one-workgroup-per-line scan at head_dim 16 around its block, wave-count and
    line-count edges, maps of a single row or column included (lines of one chunk)."""
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    channels = 16 * heads
    seed = 1000 * height + width
    mems = memories(4, heads, 16, kind="strong", seed=seed)
    x, q = (randn(batch, height, width, channels, seed=seed + i).to(dtype) for i in (1, 2))
    skip, wts = randn(channels, seed=seed + 3, scale=0.1), 1 + randn(4, channels, seed=seed + 4, scale=0.1)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                                 skip.to(device), wts.to(device), (width, width, height, height)).cpu().numpy()
    expected = oracle.operator_forward(x.float().numpy(), q.float().numpy(), mems, skip.numpy(), wts.numpy(), 16)
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    assert r <= BLOCK_TOL and m <= BLOCK_TOL, f"{dtype} {height}x{width}: normwise {r:.3e}, elementwise {m:.3e}"


@pytest.mark.parametrize("batch,height,width,heads", [
    (2, 1, 16, 1), (1, 17, 1, 2), (2, 16, 17, 1), (1, 31, 32, 2), (1, 33, 48, 1), (2, 49, 15, 1), (1, 64, 65, 1),
    (1, 5, 127, 2), (1, 128, 3, 1), (64, 16, 16, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_line_per_workgroup_scan_edges_wide_heads(oracle, device, batch, height, width, heads, dtype):
    """The same at head_dim 32: 1 to 8 blocks per chunk (fp16 and FP32 maps with more than 4 run
    the stepped and the wide scan), full, ragged and single-token, rows and columns with
    different wave counts."""
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    channels = 32 * heads
    seed = 1000 * height + width
    mems = memories(4, heads, 32, kind="strong", seed=seed)
    x, q = (randn(batch, height, width, channels, seed=seed + i).to(dtype) for i in (1, 2))
    skip, wts = randn(channels, seed=seed + 3, scale=0.1), 1 + randn(4, channels, seed=seed + 4, scale=0.1)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                                 skip.to(device), wts.to(device), (width, width, height, height)).cpu().numpy()
    expected = oracle.operator_forward(x.float().numpy(), q.float().numpy(), mems, skip.numpy(), wts.numpy(), 32)
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    assert r <= BLOCK_TOL and m <= BLOCK_TOL, f"{dtype} {height}x{width}: normwise {r:.3e}, elementwise {m:.3e}"


@pytest.mark.parametrize("batch,height,width,heads", [(1, 65, 65, 2), (1, 100, 80, 2), (1, 128, 128, 1)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_wide_heads_long_chunks_keep_fp32_products(oracle, device, batch, height, width, heads, dtype):
    """head_dim 32, chunks of 65 to 128 tokens of fp16 and FP32 maps, saturated gates: FP32
    products throughout.  The output is two chained sums of 32 FP32 products, so with random
    roundings it is within sqrt(2 x 32) 2^-24 normwise (observed 1.6e-7); operands split into
    bf16 hi + lo gave 7e-7 to 1.1e-6 for the first two maps."""
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    channels = 32 * heads
    seed = 1000 * height + width
    mems = list(memories(4, heads, 32, kind="strong", seed=seed))
    mems[3:] = [4.0 * m for m in mems[3:]]
    x, q = (randn(batch, height, width, channels, seed=7 * height + width + i).to(dtype) for i in (1, 2))
    skip, wts = torch.zeros(channels), torch.ones(4, channels)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), x.to(device), q.to(device),
                                 skip.to(device), wts.to(device), (width, width, height, height)).cpu().numpy()
    expected = oracle.operator_forward(x.float().numpy(), q.float().numpy(), mems, skip.numpy(), wts.numpy(), 32)
    assert rel_err(got, expected) <= 64 ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("batch,height,width,heads,offset", [
    (64, 17, 5, 8, 0), (128, 17, 5, 8, 0), (129, 5, 18, 8, 0), (114, 18, 20, 9, 0), (64, 3, 130, 4, 0),
    (2, 17, 5, 4, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_packed_scan_by_default(oracle, device, batch, height, width, heads, offset, dtype):
    """What the library gives to the packed scan by itself: chunks of more than 16 tokens from
    2,048 lines (one line per wave), from 4,096 with an even and an odd number of heads (two
    lines per wave, one), chunks of more than 128 from 1,024 lines, and rows that are not
    aligned for vector loads."""
    from visionhope_amd.models.srnl_core.fused import srnl_spatial_inference

    channels = 16 * heads
    seed = 1000 * height + width + heads
    mems = memories(4, heads, 16, kind="strong", seed=seed)
    x, q = (randn(batch, height, width, channels, seed=seed + i).to(dtype) for i in (1, 2))
    skip, wts = randn(channels, seed=seed + 3, scale=0.1), 1 + randn(4, channels, seed=seed + 4, scale=0.1)
    xd = torch.empty(x.numel() + offset, dtype=dtype, device=device)[offset:].view(x.shape).copy_(x)
    got = srnl_spatial_inference(tuple(torch.from_numpy(m).to(device) for m in mems), xd, q.to(device),
                                 skip.to(device), wts.to(device), (width, width, height, height)).cpu().numpy()
    expected = oracle.operator_forward(x.float().numpy(), q.float().numpy(), mems, skip.numpy(), wts.numpy(), 16)
    r, m = rel_err(got, expected), max_rel_err(got, expected)
    assert r <= BLOCK_TOL and m <= BLOCK_TOL, f"{dtype} {height}x{width}: normwise {r:.3e}, elementwise {m:.3e}"
