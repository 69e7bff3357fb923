// SRNL chunk scan for head_dim 32 (bf16, fp16 or FP32 activations): the form of
// srnl_utw.hip (one workgroup per line, one wave per 16-token block of a chunk, W waves, the
// product Gamma of the chunk gains carried) with 32-wide matrices as 2 x 2 tiles.  Reference
// recurrence: models/srnl_core/csrc/inference_recurrence.cuh:32-135, memory.cuh:219-233.
//
//   * products over the 32 features run as one 16x16x32 step of bf16 hi + lo operands (a lane's
//     quads of the two tiles as eight consecutive k), those over 16 tokens as 16x16x16; the
//     solves are FP32 with both feature tiles as right-hand sides;
//   * several blocks per chunk: the column tiles of P <- X_w^T P + (Gamma Y_w)^T do not meet, so
//     waves 0 and 1 chain one each without a barrier, while the last two waves store the
//     chunk-start content memory M_m Gamma, half of its columns each;
//   * one block per chunk (W = 1): Gamma'^T = a Gamma^T - K D_e (Gamma R)^T, no map.
//
// Bound by the dependency chain of a chunk.  Per launch on MI355X, against the form that
// carried the whole 112 x 32 state, solved (I + L) by columns on the vector unit and met at
// a barrier for every block of a chunk: 384 lines of 3,136 tokens (chunks of 56) 274 -> 204 us,
// 128 lines 215 -> 149, 1,024 lines of 784 (28) 222 -> 110, 4,096 of 196 (14) 212 -> 102, 8 of
// 196 (14) 50 -> 33; bf16 with chunks of more than 64 tokens (8 waves, one workgroup per CU; it
// was the wide scan) 1,024 lines of 6,400 (80) 1,692 -> 1,157, 384 of 16,384 (128) 1,699 -> 1,018.
// Those lines of fp16 and FP32 keep the stepped and the wide scan: their products are FP32, and
// this form's split operands were 1.1 (small gates) to 7 times (saturated ones) as far from 64
// bits (maps of 65 x 65 to 128 x 128).  A bf16 map's error is that of its split chunk states
// either way (2.5e-6, within 1%).
#include <algorithm>

#include "srnl_block_form.h"
#include "srnl_blocks.h"

namespace vh {
using namespace blocks;
using blockform::XQuad;

namespace {

// A column of two FP32 tiles (32 rows) as bf16 matrix-core operands, |v - hi - lo| <= 2^-16 |v|.
struct Col {
    v4s h[2], l[2];
};
__device__ __forceinline__ Col split(v4f t0, v4f t1) {
    Col o;
    blockform::split4(t0, o.h[0], o.l[0]);
    blockform::split4(t1, o.h[1], o.l[1]);
    return o;
}
// acc + A^T B over 32 rows
__device__ __forceinline__ v4f mm(const Col& a, const Col& b, v4f acc) { return blockform::mma3k2(a.h, a.l, b.h, b.l, acc); }
// acc + A^T B over 16 rows, tile i of a and j of b
__device__ __forceinline__ v4f mm16(const Col& a, int i, const Col& b, int j, v4f acc) {
    return blockform::mma3(a.h[i], a.l[i], b.h[j], b.l[j], acc);
}

__device__ __forceinline__ v4f load4f(const float* p) { return *reinterpret_cast<const v4f*>(p); }

// A column in LDS: hi and lo halves apart, so that a wave's 16-byte accesses meet no conflict.
struct ColStore {
    uint4 h[64], l[64];
    __device__ __forceinline__ void put(int lane, const Col& v) {
        const uint2 a = __builtin_bit_cast(uint2, v.h[0]), b = __builtin_bit_cast(uint2, v.h[1]);
        const uint2 c = __builtin_bit_cast(uint2, v.l[0]), d = __builtin_bit_cast(uint2, v.l[1]);
        h[lane] = make_uint4(a.x, a.y, b.x, b.y);
        l[lane] = make_uint4(c.x, c.y, d.x, d.y);
    }
    __device__ __forceinline__ Col get(int lane) const {
        const uint4 a = h[lane], b = l[lane];
        Col v;
        v.h[0] = __builtin_bit_cast(v4s, make_uint2(a.x, a.y));
        v.h[1] = __builtin_bit_cast(v4s, make_uint2(a.z, a.w));
        v.l[0] = __builtin_bit_cast(v4s, make_uint2(b.x, b.y));
        v.l[1] = __builtin_bit_cast(v4s, make_uint2(b.z, b.w));
        return v;
    }
};

constexpr int kGamStride = 36;   // floats per row of Gamma: 16-byte aligned, rows in different banks

template <int W>
struct Shared {
    Scratch scratch[W];
    float tr[W][16 * kTrStride];           // second transpose scratch
    float gam[W > 1 ? 32 : 1][kGamStride]; // Gamma, by rows
    ColStore G[2];                         // Gamma^T by columns of tiles
    ColStore X[W > 1 ? W : 1][2];          // X_w by columns of tiles
    v4f Y[W > 1 ? W : 1][2][2][W > 1 ? 64 : 1];   // (Gamma Y_w)^T: column tile, row tile
};

}  // namespace

template <typename T, int W, bool SPATIAL>
__global__ __launch_bounds__(64 * W, 2) void srnl_scan32_utw_kernel(const ScanParams p) {
    constexpr int D = 32;
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
    // columns i of the transposed memories: rows 16 i + c, entries 4g.. and 16 + 4g..
    auto column = [&](const float* m, int i) {
        const float* row = m + (sidx * D + 16 * i + c) * D + 4 * g;
        return split(load4f(row), load4f(row + 16));
    };
    const Col MkT[2] = {column(p.Mk, 0), column(p.Mk, 1)}, MvT[2] = {column(p.Mv, 0), column(p.Mv, 1)};
    const Col MmT[2] = {column(p.Mm, 0), column(p.Mm, 1)};
    // e and a as operand rows 4 j and 4 j + 1, so every lane's registers 0 and 1 end with e.z and a.z
    const float* gate_row = ((c & 1) ? p.Ma : p.Me) + sidx * D + 4 * g;
    const Col gates = (c & 3) < 2 ? split(load4f(gate_row), load4f(gate_row + 16)) : split(zero, zero);

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
    XRaw<T, 16> xr[2] = {};
    auto load_x = [&](int64_t cc) {
        int64_t off = 0;
        if (valid) {
            if (SPATIAL && p.aligned) off = static_cast<int64_t>(pa * static_cast<int>(cc) + pb * slot + pc) * pst;
            else off = token_offset<SPATIAL>(p.x, r, cc * C + slot);
        }
        xr[0] = XQ::load(xcol + off);
        xr[1] = XQ::load(xcol + off + 16);
    };
    // Columns 16 i + 4g.. of the content memory M_m Gamma the readout of chunk cc uses (M_m
    // itself, unrounded, for the first), from column i of Gamma's tiles.
    auto store_content = [&](int64_t cc, int i, const Col& gam) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int at = (16 * j + c) * D + 16 * i + 4 * g;
            const v4f m = cc == 0 ? load4f(p.Mm + sidx * D * D + at) : mm(gam, MmT[j], zero);
            store_state4(p.states + (line * p.max_chunks + cc) * D * D + at, make_float4(m[0], m[1], m[2], m[3]),
                         p.split_states);
        }
    };
    // W > 1: the waves that store the content, and the column of Gamma each holds for it
    constexpr int kFirstStore = W > 2 ? W - 2 : 0;
    const int part = wv - kFirstStore;
    auto gamma_column = [&]() {
        v4f t[2];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) t[k][i] = sh.gam[W > 1 ? 16 * k + 4 * g + i : 0][16 * part + c];
        return split(t[0], t[1]);
    };

    v4f gamT[2][2] = {{bl.diagonal(1.f), zero}, {zero, bl.diagonal(1.f)}};   // [column][row]
    Col G[2] = {split(gamT[0][0], gamT[0][1]), split(gamT[1][0], gamT[1][1])};
    Col gam[2] = {G[0], G[1]};   // columns of Gamma; W > 1: [0], column `part`
    if (W > 1) gam[0] = part == 1 ? G[1] : G[0];
    if (nc > 1 && wv < nblk) load_x(0);
    for (int64_t ch = 0; ch < nc - 1; ++ch) {
        if (W == 1 || wv < nblk) {
            v4s xh[2], xl[2];
            XQ::operands(xr[0], valid, xh[0], xl[0]);
            XQ::operands(xr[1], valid, xh[1], xl[1]);
            const Col Z = split(XQ::mma_k2(G[0].h, G[0].l, xh, xl, zero), XQ::mma_k2(G[1].h, G[1].l, xh, xl, zero));
            if (ch + 1 < nc - 1) load_x(ch + 1);   // in flight during this chunk
            v4f K[2] = {mm(MkT[0], Z, zero), mm(MkT[1], Z, zero)}, Dl[2];
            const v4f V[2] = {mm(MvT[0], Z, zero), mm(MvT[1], Z, zero)}, pre = mm(gates, Z, zero);
            float kn = 0.f, dsq = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) kn += K[0][i] * K[0][i] + K[1][i] * K[1][i];
            kn = xor16_32_sum(kn);
            // ||k||^2 of the normalised key is ||k~||^2 / (||k~||^2 + 1e-6)
            const float inv = rsqrtf(kn + 1e-6f);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                K[t] *= inv;
                Dl[t] = K[t] - V[t];
#pragma unroll
                for (int i = 0; i < 4; ++i) dsq += Dl[t][i] * Dl[t][i];
            }
            dsq = xor16_32_sum(dsq);
            float alpha, eff;
            token_gates_fast(p.k, pre[0], pre[1], dsq, kn * inv * inv, alpha, eff);
            const Col k = split(K[0], K[1]), dl = split(Dl[0], Dl[1]);
            const v4f gram = mm(k, k, zero);
            const v4f gd[2] = {mm(dl, G[0], zero), mm(dl, G[1], zero)};   // (Gamma Delta)^T
            // K^T by two transposes in one pass through LDS
            v4f KT[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bl.s.tr[(4 * g + i) * kTrStride + c] = K[0][i];
                sh.tr[wv][(4 * g + i) * kTrStride + c] = K[1][i];
            }
            __builtin_amdgcn_wave_barrier();
            KT[0] = load4f(&bl.s.tr[c * kTrStride + 4 * g]);
            KT[1] = load4f(&sh.tr[wv][c * kTrStride + 4 * g]);
            __builtin_amdgcn_wave_barrier();
            const Decays dec = bl.decays(valid ? eff : 0.f, valid ? alpha : 1.f);
            const Triangle tri = bl.triangle(dec, gram);
            if constexpr (W == 1) {
                v4f RT[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) RT[j] = mm(k, G[j], zero) * dec.Da_r() + gd[j];
                bl.solve_lower(tri, RT);
                store_content(ch, 0, gam[0]);
                store_content(ch, 1, gam[1]);
                const Col kd = split(-(KT[0] * dec.De_r()), -(KT[1] * dec.De_r())), rt = split(RT[0], RT[1]);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) gamT[j][i] = mm16(kd, i, rt, j, gamT[j][i] * dec.a());
                    G[j] = split(gamT[j][0], gamT[j][1]);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) gam[i] = split(bl.transpose(gamT[0][i]), bl.transpose(gamT[1][i]));
            } else {
                v4f S[2] = {KT[0] * dec.De_r(), KT[1] * dec.De_r()};
                bl.solve_upper(tri, S);
                const Col s = split(-S[0], -S[1]), ka = split(KT[0] * dec.Da_r(), KT[1] * dec.Da_r());
                const Col d = split(gd[0], gd[1]);
                const v4f aI = bl.diagonal(dec.a());
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    sh.X[wv][j].put(lane, split(mm16(ka, 0, s, j, j == 0 ? aI : zero), mm16(ka, 1, s, j, j == 1 ? aI : zero)));
#pragma unroll
                    for (int i = 0; i < 2; ++i) sh.Y[wv][j][i][lane] = mm16(s, i, d, j, zero);
                }
            }
        }
        if constexpr (W > 1) {
            if (W == 2) store_content(ch, part, gam[0]);
            __syncthreads();
            if (wv < 2) {
                Col P = G[0];
                if (wv == 1) P = G[1];
                v4f t[2];
                // the next map is in flight while a step runs (past the last block: read, unused)
                Col X[2] = {sh.X[0][0].get(lane), sh.X[0][1].get(lane)};
                v4f Y[2] = {sh.Y[0][wv][0][lane], sh.Y[0][wv][1][lane]};
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const Col x[2] = {X[0], X[1]};
                    const v4f y[2] = {Y[0], Y[1]};
                    if (w + 1 < W) {
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            X[i] = sh.X[w + 1][i].get(lane);
                            Y[i] = sh.Y[w + 1][wv][i][lane];
                        }
                    }
                    if (w < nblk) {
                        t[0] = mm(x[0], P, y[0]);
                        t[1] = mm(x[1], P, y[1]);
                        P = split(t[0], t[1]);
                    }
                }
                sh.G[wv].put(lane, P);
#pragma unroll
                for (int i = 0; i < 2; ++i) *reinterpret_cast<v4f*>(&sh.gam[W > 1 ? 16 * wv + c : 0][16 * i + 4 * g]) = t[i];
            } else if (W > 2 && part >= 0) {
                store_content(ch, part, gam[0]);
            }
            __syncthreads();
            G[0] = sh.G[0].get(lane);
            G[1] = sh.G[1].get(lane);
            if (part >= 0) gam[0] = gamma_column();
        }
    }
    if (W == 1) {
        store_content(nc - 1, 0, gam[0]);
        store_content(nc - 1, 1, gam[1]);
    } else if (part >= 0) {
        store_content(nc - 1, part, gam[0]);
    }
}

// Waves per line of the head_dim-32 block-form scan: the chunk's 16-slot blocks rounded up to
// a power of two; 0 when a chunk exceeds 8 blocks (128 tokens; 4 blocks for fp16 and FP32
// activations, whose longer chunks keep FP32 products) or the input rows are not aligned for
// vector loads.
template <typename T>
constexpr int kMaxBlocks = std::is_same<T, bf16_t>::value ? 8 : 4;

template <typename T>
int scan32_utw_waves(const ScanParams& sp) {
    int max_chunk = 0;
    for (int r = 0; r < sp.R; ++r) max_chunk = std::max(max_chunk, sp.chunk[r]);
    const int blocks = (max_chunk + 15) / 16;
    if (blocks > kMaxBlocks<T> || !sp.x_vec) return 0;
    int w = 1;
    while (w < blocks) w *= 2;
    return w;
}

template <typename T>
bool launch_scan32_utw(const ScanParams& sp, hipStream_t stream) {
    const int waves = scan32_utw_waves<T>(sp);
    if (waves == 0) return false;
    const unsigned grid = static_cast<unsigned>(sp.B * sp.R * sp.heads);
    auto go = [&](auto wc, auto spc) {
        constexpr int WV = decltype(wc)::value;
        hipLaunchKernelGGL((srnl_scan32_utw_kernel<T, WV, decltype(spc)::value>), dim3(grid), dim3(64 * WV), 0, stream,
                           sp);
    };
    auto pick = [&](auto spc) {
        switch (waves) {
            case 1: go(std::integral_constant<int, 1>{}, spc); break;
            case 2: go(std::integral_constant<int, 2>{}, spc); break;
            case 4: go(std::integral_constant<int, 4>{}, spc); break;
            default:
                if constexpr (kMaxBlocks<T> == 8) go(std::integral_constant<int, 8>{}, spc);
                break;
        }
    };
    if (sp.x.spatial) pick(std::true_type{});
    else pick(std::false_type{});
    return true;
}

template bool launch_scan32_utw<bf16_t>(const ScanParams&, hipStream_t);
template bool launch_scan32_utw<f16_t>(const ScanParams&, hipStream_t);
template bool launch_scan32_utw<float>(const ScanParams&, hipStream_t);

}  // namespace vh
