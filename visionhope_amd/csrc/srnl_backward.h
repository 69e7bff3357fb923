// Launch parameters shared by the SRNL backward kernels (srnl_backward.hip and
// srnl_backward_blocks.hip).
#pragma once

#include "vh_common.h"

namespace vh {

constexpr int kBwdMaxChunk = 64;     // small head dims: chunks up to this length use the small-LDS variant
constexpr int kBwdLongChunk = 256;   // longest chunk of the backward (lines.cu:252-760 range)

struct BwdParams {
    const void* x;      // [B, R, heads, N, D] io dtype
    const void* q;      // raw: [B, R, N, heads * D] io dtype; else fp32 [B, R, heads, N, D]
    const float* dy;    // [B, R, heads, N, D]
    const float* m0[5]; // M_m, M_v, M_k [S, D, D]; M_eta, M_alpha [S, D]; S = R * heads, or one per line
    int per_line;       // 1: state s = line; 0: s = line % (R * heads), shared over the batch
    float* dx;          // [B, R, heads, N, D]
    float* dq;          // layout of q, fp32
    float* dline;       // [lines, 3 D^2 + 2 D] per-line gradient of the initial state
    float* states;      // small head dims: [lines, nc, 3 D^2 + 2 D] chunk-start states;
                        // block form: [lines, nc, D^2] products of the chunk gains before each chunk
                        // (from the first chunk on; written by the gains kernel)
    float* gtraj;       // small head dims: [lines, CMAX, D, D] gain trajectory of the current chunk;
                        // block form: [lines, waves, segments, D^2] segment-start gains (chunks of several segments)
    int64_t B, R, heads, N, nc;
    int segs;           // block form: segments of the longest chunk
    int io_dtype, q_raw;
    int chunk[4];
    vh_srnl_consts k;
    // Spatial form (block form only): x, q, dy are channels-last maps [B, H, W, heads * D]
    // (x and q io dtype, dy the FP32 gradient of the fused output), R = 4 scan orders; dx and
    // dq become four planes of such maps in the io dtype, one per direction, and the M_m part
    // of dline the gradient for unit direction weights.
    const float* scale;   // [4, heads * D] direction weights; null: packed lines (backward kernel)
    int64_t H, W;
    float inv_h;
    void *dx_planes, *dq_planes;
    float* content;       // gains kernel: chunk-start M_m for the readout, or null
    int content_split;    // stored as bf16 hi + lo pairs (store_state4)
};

// d(eta^)/d(cap) of eta^ = cap (1 - exp(-u)), u = eta / cap: (1 - e^-u) - u e^-u, by its
// series u^2 (1/2 - u/3 + u^2/8 - u^3/30 + u^4/144) below u = 1e-3 (cancellation).
__device__ __forceinline__ float softcap_dcap(float u, float e_neg) {
    if (u < 1e-3f) return u * u * (0.5f + u * (-1.f / 3.f + u * (1.f / 8.f + u * (-1.f / 30.f + u / 144.f))));
    return -expm1f(-u) - u * e_neg;
}

// Block form (head_dim 16 and 32): waves per line for the longest chunk, and the segments
// of 16 * waves tokens that chunk takes.
int bwd_block_waves(int head_dim, int64_t max_chunk, int64_t lines);
inline int bwd_block_segs(int waves, int64_t max_chunk) { return static_cast<int>((max_chunk + 16 * waves - 1) / (16 * waves)); }
int launch_backward_gains(const BwdParams& p, bool spatial, int head_dim, int waves, int64_t lines, hipStream_t stream);
int launch_backward_blocks(const BwdParams& p, int head_dim, int waves, int64_t lines, hipStream_t stream);

}  // namespace vh
