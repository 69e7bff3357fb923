// SRNL chunk scan for head_dim 16 (bf16, fp16 or FP32 activations) in 16-token blocks, one
// workgroup per line, one wave per block of a chunk (W = the chunk's blocks rounded up to a
// power of two, at most 8): every line count with chunks of one block, fewer than 2,048 lines
// with longer ones (launch_scan in srnl.hip).
//
// With Gamma the product of the gains of the chunks so far, the state is S_0 Gamma (reference
// refresh inference_recurrence.cuh:119-133: M <- M G, e <- G^T e, a <- G^T a), so only the
// 16 x 16 Gamma is carried: z = Gamma x, k~ = M_k z, v = M_v z and the gate pre-activations
// e.z, a.z come from the initial memories, which stay in registers.  For a block of 16 slots
// entered with gain G (D_a, D_e, L: srnl_blocks.h; K the keys, Delta = k - v):
//   G' = a G - R D_e K^T,  R (I + L) = G K D_a + Delta;   as a map  G' = G X + Y,
//   X = a I - K D_a S,  Y = -Delta S,  (I + L) S = D_e K^T.
//   * several blocks per chunk: wave w forms X_w and (Gamma Y_w)^T = -S^T (Gamma Delta)^T;
//     after one barrier wave 0 chains P <- X_w^T P + (Gamma Y_w)^T from P = Gamma^T, which
//     ends as the next chunk's Gamma^T, and hands it out through LDS; the last wave stores
//     the chunk-start content memory M_m Gamma meanwhile;
//   * one block per chunk (W = 1): the right-hand side is multiplied by Gamma before the
//     solve, (I + L^T) (Gamma R)^T = D_a K^T Gamma^T + (Gamma Delta)^T, so Gamma'^T =
//     a Gamma^T - K D_e (Gamma R)^T needs no map.
// Products run on bf16 operands split hi + lo (x exact when it is bf16), which leave the vector
// pipe free while they run; the solves are FP32 (v_mfma_f32_16x16x4_f32), which hold it.
// (Measured: a vector FMA of another wave waits for a 34-cycle FP32 product, not for a bf16
// one; with FP32 products throughout, two waves on a SIMD did not overlap and 8 waves took
// 389 us where the split ones take 296.)  Bound by the dependency chain of a chunk.
//
// Per launch on MI355X, against the form that carried the whole 64 x 16 state and solved
// (I + L) by columns on the vector unit: 96 lines of 16,384 tokens (chunks of 128) 370 -> 288
// us, 64 lines of 600 (30, 20) 64 -> 44, 32 lines of 196 (14) 30 -> 18; against the packed form
// (srnl_ut.hip): 1,024 lines of 3,136 (56) 202 -> 179, 4,096 of 196 (14) 52 -> 44, 8,192 of 49
// (7) 48 -> 40.
#include <algorithm>

#include "srnl_block_form.h"
#include "srnl_blocks.h"

namespace vh {
using namespace blocks;
using blockform::XQuad;

namespace {

// An FP32 tile as bf16 matrix-core operands, |v - hi - lo| <= 2^-16 |v|.
struct Op {
    v4s h, l;
};
__device__ __forceinline__ Op split(v4f v) {
    Op o;
    blockform::split4(v, o.h, o.l);
    return o;
}
// acc + A^T B
__device__ __forceinline__ v4f mm(const Op& a, const Op& b, v4f acc) { return blockform::mma3(a.h, a.l, b.h, b.l, acc); }

__device__ __forceinline__ v4f load4f(const float* p) { return *reinterpret_cast<const v4f*>(p); }

template <int W>
struct Shared {
    Scratch scratch[W];
    float gam[16][kTrStride];                          // Gamma, by rows
    Op gamT[64];                                       // Gamma^T as a tile, split
    Op X[W > 1 ? W : 1][W > 1 ? 64 : 1];               // X_w as a tile, split
    v4f Y[W > 1 ? W : 1][W > 1 ? 64 : 1];              // (Gamma Y_w)^T as a tile
};

}  // namespace

template <typename T, int W, bool SPATIAL>
__global__ __launch_bounds__(64 * W, 4) void srnl_scan16_utw_kernel(const ScanParams p) {
    constexpr int D = 16;
    using XQ = XQuad<T>;
    __shared__ Shared<W> sh;
    const int wv = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const Block bl(sh.scratch[wv], static_cast<int>(threadIdx.x) & 63);
    const int lane = bl.lane, g = bl.g, c = bl.c;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};

    const int64_t lines = p.B * p.R * p.heads;
    const int64_t line = xcd_remap(blockIdx.x, lines);
    const int64_t head = line % p.heads;
    const int r = static_cast<int>((line / p.heads) % p.R);
    const int64_t b = line / (p.heads * p.R);
    const int64_t sidx = p.per_line_state ? line : r * p.heads + head;
    // rows c of the memories as tiles N(M^T); entries 4g.. of the gate vectors
    const Op MkT = split(load4f(p.Mk + (sidx * D + c) * D + 4 * g)), MvT = split(load4f(p.Mv + (sidx * D + c) * D + 4 * g));
    const v4f Mm_rows = load4f(p.Mm + (sidx * D + c) * D + 4 * g);
    const Op MmT = split(Mm_rows);
    // e and a as operand rows 4 j and 4 j + 1, so every lane's registers 0 and 1 end with e.z and a.z
    const Op gates = split((c & 3) < 2 ? load4f(((c & 1) ? p.Ma : p.Me) + sidx * D + 4 * g) : zero);

    const int C = chunk_of(p.chunk, r);
    const int64_t nc = (p.L + C - 1) / C;
    const int nblk = (C + 15) / 16;
    const int slot = 16 * wv + bl.tau;   // this lane's token of a chunk
    const bool valid = slot < C;         // every chunk but the last is whole, and the last forms no gain
    const T* xcol = static_cast<const T*>(p.x.ptr) + b * p.x.sb + r * p.x.sr + head * p.x.sh + 4 * g;
    int pa = 0, pb = 0, pc = 0, pst = 0;
    if constexpr (SPATIAL) {
        const int Wd = static_cast<int>(p.x.W), L = static_cast<int>(p.x.H * p.x.W);
        pa = r == 0 ? Wd : r == 1 ? -Wd : r == 2 ? 1 : -1;
        pb = r == 0 ? 1 : r == 1 ? -1 : r == 2 ? Wd : -Wd;
        pc = (r & 1) ? L - 1 : 0;
        pst = static_cast<int>(p.x.st);
    }
    // x of this lane's token of chunk cc as raw bits; slots past the chunk read the line's
    // first token and are zeroed when decoded
    auto load_x = [&](int64_t cc) {
        int64_t off = 0;
        if (valid) {
            if (SPATIAL && p.aligned) off = static_cast<int64_t>(pa * static_cast<int>(cc) + pb * slot + pc) * pst;
            else off = token_offset<SPATIAL>(p.x, r, cc * C + slot);
        }
        return load_xraw<T, 16>(xcol + off);
    };
    // The content memory M_m Gamma the readout of chunk cc uses (M_m itself, unrounded, for the
    // first): (M_m Gamma)^T, row c and columns 4g.. of M_m Gamma.
    auto store_content = [&](int64_t cc, v4f gam) {
        const v4f m = cc == 0 ? Mm_rows : mm(split(gam), MmT, zero);
        store_state4(p.states + (line * p.max_chunks + cc) * D * D + c * D + 4 * g,
                     make_float4(m[0], m[1], m[2], m[3]), p.split_states);
    };
    auto gamma_rows = [&]() {   // N(Gamma) from its rows in LDS
        v4f v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = sh.gam[4 * g + i][c];
        return v;
    };

    v4f gamT = bl.diagonal(1.f), gam = gamT;
    Op G = split(gamT);
    XRaw<T, 16> xr{};
    if (nc > 1 && wv < nblk) xr = load_x(0);
    for (int64_t ch = 0; ch < nc - 1; ++ch) {
        v4f K, Dl;
        if (W == 1 || wv < nblk) {
            v4s xh, xl;
            XQ::operands(xr, valid, xh, xl);
            const Op Z = split(XQ::mma(G.h, G.l, xh, xl, zero));
            if (ch + 1 < nc - 1) xr = load_x(ch + 1);   // in flight during this chunk
            K = mm(MkT, Z, zero);
            const v4f V = mm(MvT, Z, zero), pre = mm(gates, Z, zero);
            float dsq = 0.f;
            const float kn = xor16_32_sum((K[0] * K[0] + K[1] * K[1]) + (K[2] * K[2] + K[3] * K[3]));
            // ||k||^2 of the normalised key is ||k~||^2 / (||k~||^2 + 1e-6)
            const float inv = rsqrtf(kn + 1e-6f);
            K *= inv;
            Dl = K - V;
#pragma unroll
            for (int i = 0; i < 4; ++i) dsq += Dl[i] * Dl[i];
            dsq = xor16_32_sum(dsq);
            float alpha, eff;
            token_gates_fast(p.k, pre[0], pre[1], dsq, kn * inv * inv, alpha, eff);
            const Op k = split(K);
            const v4f gram = mm(k, k, zero), KT = bl.transpose(K);
            const v4f gd = mm(split(Dl), G, zero);   // (Gamma Delta)^T
            const Decays dec = bl.decays(valid ? eff : 0.f, valid ? alpha : 1.f);
            const Triangle tri = bl.triangle(dec, gram);
            if constexpr (W == 1) {
                v4f RT[1] = {mm(k, G, zero) * dec.Da_r() + gd};
                bl.solve_lower(tri, RT);
                store_content(ch, gam);
                gamT = mm(split(-(KT * dec.De_r())), split(RT[0]), gamT * dec.a());
                G = split(gamT);
                gam = bl.transpose(gamT);
            } else {
                v4f S[1] = {KT * dec.De_r()};
                bl.solve_upper(tri, S);
                const Op s = split(-S[0]);
                sh.X[wv][lane] = split(mm(split(KT * dec.Da_r()), s, bl.diagonal(dec.a())));
                sh.Y[wv][lane] = mm(s, split(gd), zero);
            }
        }
        if constexpr (W > 1) {
            __syncthreads();
            if (wv == 0) {
                // the next map is in flight while a step runs (past the last block: read, unused)
                Op X = sh.X[0][lane];
                v4f Y = sh.Y[0][lane];
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const Op x = X;
                    const v4f y = Y;
                    if (w + 1 < W) {
                        X = sh.X[w + 1][lane];
                        Y = sh.Y[w + 1][lane];
                    }
                    if (w < nblk) {
                        gamT = mm(x, G, y);
                        G = split(gamT);
                    }
                }
                sh.gamT[lane] = G;
                *reinterpret_cast<v4f*>(&sh.gam[c][4 * g]) = gamT;
            } else if (wv == W - 1) {
                store_content(ch, gam);
            }
            __syncthreads();
            if (wv != 0) G = sh.gamT[lane];
            if (wv == W - 1) gam = gamma_rows();
        }
    }
    if (wv == W - 1) store_content(nc - 1, gam);
}

// Waves per line of the few-line block-form scan: the chunk's 16-slot blocks rounded up to
// a power of two; 0 when a chunk exceeds 8 blocks (128 tokens) or the input rows are not
// aligned for vector loads.
int scan16_utw_waves(const ScanParams& sp) {
    int max_chunk = 0;
    for (int r = 0; r < sp.R; ++r) max_chunk = std::max(max_chunk, sp.chunk[r]);
    const int blocks = (max_chunk + 15) / 16;
    if (blocks > 8 || !sp.x_vec) return 0;
    int w = 1;
    while (w < blocks) w *= 2;
    return w;
}

template <typename T>
bool launch_scan16_utw(const ScanParams& sp, hipStream_t stream) {
    const int waves = scan16_utw_waves(sp);
    if (waves == 0) return false;
    const unsigned grid = static_cast<unsigned>(sp.B * sp.R * sp.heads);
    auto go = [&](auto wc, auto spc) {
        constexpr int WV = decltype(wc)::value;
        hipLaunchKernelGGL((srnl_scan16_utw_kernel<T, WV, decltype(spc)::value>), dim3(grid), dim3(64 * WV), 0, stream,
                           sp);
    };
    auto pick = [&](auto spc) {
        switch (waves) {
            case 1: go(std::integral_constant<int, 1>{}, spc); break;
            case 2: go(std::integral_constant<int, 2>{}, spc); break;
            case 4: go(std::integral_constant<int, 4>{}, spc); break;
            default: go(std::integral_constant<int, 8>{}, spc); break;
        }
    };
    if (sp.x.spatial) pick(std::true_type{});
    else pick(std::false_type{});
    return true;
}

template bool launch_scan16_utw<bf16_t>(const ScanParams&, hipStream_t);
template bool launch_scan16_utw<f16_t>(const ScanParams&, hipStream_t);
template bool launch_scan16_utw<float>(const ScanParams&, hipStream_t);

}  // namespace vh
