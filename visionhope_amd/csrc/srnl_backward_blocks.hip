// SRNL backward for head_dim 16 and 32: the recurrence and its adjoint in 16-token block
// form on the FP32 matrix cores.
//
// Forward of one line (srnl_backward.hip states it token by token).  With Gamma_c the
// product of the chunk gains before chunk c, the chunk-start state is S_0 Gamma_c, so only
// Gamma_c (d x d) is carried: z = Gamma_c x, k~ = M_k z, v = M_v z, gate pre-activations
// e.z and a.z, y = M_m (Gamma_c q^).  Inside a chunk, for a block of 16 token slots entered
// with gain G, with a_t the product of the block's retentions before slot t, a the product
// of all 16, and the strictly upper triangle L[s][t] = eta^_s (a_t / a_{s+1}) (k_s . k_t):
//   R (I + L) = G K D_a + Delta             (columns r_t; Delta = k - v, D_a = diag(a_t))
//   G' = a G - R D_e K^T = G X + Y          (D_e = diag(eta^_t a / a_{t+1}))
//   X = a I - K D_a S, Y = -Delta S, (I + L) S = D_e K^T.
// Adjoint, with H' = dG' the gradient of the block's exit gain (H_C = Gamma^T dGamma_{c+1}):
//   Rb (I + L^T) = -H' K D_e                (columns r_bar_t)
//   H = a H' + Rb D_a K^T = H' X^T
//   dK = -H'^T R D_e + G^T Rb D_a - K (W + W^T) + Rb + ...,  W[s][t] = eta^_s (a_t / a_{s+1}) (r_s . r_bar_t), s < t
//   d alpha_t = <H_{t+1}, G_t>,  alpha_t <H_{t+1}, G_t> = a <H', G> + sum_{u > t} a_u r_bar_u . (G k_u)
//     - sum_{s < t} eta^_s (a / a_{s+1}) r_s . (H' k_s) - sum_{s < t < u} L[s][u] (r_s . r_bar_u)
// (G_t and H_{t+1} written out: only terms that span t, so a small inner product is not the
// difference of large ones, as it was with <H_t, G_t> carried from token to token: up to 11
// times the error of a direct sum with saturated gates, now up to 4; one more product and at
// most 2.5% of the time, 4,096 lines of 448 tokens, d = 16, chunks of 56: 642 -> 659 us with
// the gains).  Then
//   dz = M_v^T dv + M_k^T dk~ + e d_pre_eta + a d_pre_alpha,  dx = Gamma^T dz,
//   dGamma_c = dGamma_{c+1} G_C^T + sum_t (dz_t x_t^T + (M_m^T dy_t) q^_t^T).
// The regrouping is exact in real arithmetic; every product is FP32
// (v_mfma_f32_16x16x4_f32), nothing is split or rounded to 16 bits.
//
// Mapping.  One workgroup per line, wave w holding block w of the current 16 W-token
// segment of a chunk (W = 1, 2, 4 or 8 waves; longer chunks take several segments).  Tiles,
// slot order and solves: srnl_blocks.h.
//
// Two kernels: the gains kernel runs the forward and leaves Gamma before every chunk (a training
// step on maps runs it as its forward, so its backward starts there; packed lines run it ahead of
// the backward), the backward kernel takes the chunks in reverse.
//
// Bound: the dependency chain of a chunk, and within it the issue of the FP32 products, which
// hold the vector pipe (34 cycles each, srnl_utw.hip); the bytes take under a tenth of the time.
// Times on MI355X against the token-by-token kernel (which head_dim 4 and 8 still run), gains +
// backward: 4,096 lines of 196 tokens, d = 16, chunks of 14: 2,480 -> 79 + 192 us; 512 lines of
// 3,136 tokens, d = 16, chunks of 56: 24,500 -> 186 + 510 us; 48 lines of 960 tokens, d = 32,
// chunks of 40 and 24: 11,800 -> 172 + 422 us; 4 lines of 196 tokens, d = 32, chunks of 64: 1,690
// -> 18 + 52 us.  With the forward repeated inside the backward kernel the first three took 249,
// 710 and 745 us after a separate forward scan of 54, 125 and 130 us; with every wave walking all
// of a chunk's maps and forming all of H, and transposes as products: 193, 540, 558 and 57 us.
// Fetching the next chunk's operands ahead changed these by under 3% either way.
#include <algorithm>
#include <cmath>

#include "srnl_backward.h"
#include "srnl_blocks.h"

namespace vh {
using namespace blocks;
namespace {

typedef v4f v4f_any __attribute__((aligned(4)));
typedef unsigned short us4_any __attribute__((ext_vector_type(4), aligned(2)));

// Four consecutive elements of an io-dtype row as FP32.  Rows start at any element (a
// contiguous tensor may be a view at an odd offset), so the loads assume no alignment.
__device__ __forceinline__ v4f load_io4(const void* p, int64_t idx, int io) {
    if (io == VH_DTYPE_F32) return *reinterpret_cast<const v4f_any*>(static_cast<const float*>(p) + idx);
    const us4_any u = *reinterpret_cast<const us4_any*>(static_cast<const uint16_t*>(p) + idx);
    v4f r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = io == VH_DTYPE_BF16 ? to_f32(bf16_t{u[i]}) : to_f32(f16_t{u[i]});
    return r;
}

__device__ __forceinline__ void store_io4(void* p, int64_t idx, int io, v4f v) {
    if (io == VH_DTYPE_F32) {
        *reinterpret_cast<v4f_any*>(static_cast<float*>(p) + idx) = v;
        return;
    }
    us4_any u;
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = io == VH_DTYPE_BF16 ? from_f32<bf16_t>(v[i]).bits : from_f32<f16_t>(v[i]).bits;
    *reinterpret_cast<us4_any*>(static_cast<uint16_t*>(p) + idx) = u;
}

// e^x within about one ulp for the normal ranges met here, in 6 instructions (hardware
// approximation and one correction) instead of the library's 10 and more.
__device__ __forceinline__ float exp1(float x) {
    constexpr float kLog2e = 1.44269504088896341f, kLog2eLow = 1.925963033500e-8f, kLn2 = 0.69314718055994531f;
    const float t = x * kLog2e, rest = fmaf(x, kLog2e, -t) + x * kLog2eLow, e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, rest * kLn2, e);
}

__device__ __forceinline__ float wave_sum(float v) { return row_group_sum<16>(xor16_32_sum(v)); }

template <int D, int W>
struct Shared {
    static constexpr int ND = D / 16, NT = ND * ND;
    // Memories as tiles [tile][lane]: N(M^T) of M_k, M_v; N(M) of M_k, M_v, M_m.
    v4f mem[5][NT][64];
    float ev[2][D];
    float E[D][D + 4];                 // dGamma of the next chunk, row major
    Scratch scratch[W];
    // Block maps X, X^T, Y^T of the segment (W > 1); also the waves' partial sums.
    v4f maps[W > 1 ? W : 1][W > 1 ? 3 : 1][NT][64];
    v4f HT[W > 1 ? NT : 1][W > 1 ? 64 : 1];   // H^T at the chunk's exit
};

// Everything the recurrence needs from the 16 tokens of one block.
template <int ND>
struct Tokens {
    v4f Z[ND], K[ND], Dl[ND];      // z, k, k - v: channel rows, slot columns
    v4f KT[ND], DlT[ND];           // the last two transposed
    Decays d;
    Triangle tri;
    float inv_k, eff, alpha;
    float dn, inv_denom, cap, deff_deta, deff_dcap, deff_dalpha, deff_dksq, s_eta, s_alpha;
};

template <int D, typename SharedT>
struct Line {
    static constexpr int ND = D / 16;
    SharedT& sh;
    const int w;
    const Block bl;
    const vh_srnl_consts& k;

    // Keys, values and gates of the block from x (channel rows; zero in slots past the
    // chunk) and Gamma^T.  Slots past the chunk act as the identity.
    template <bool DELTA_T = true>
    __device__ __forceinline__ void tokens(const v4f (&X)[ND], bool valid, const v4f (&GamT)[ND][ND],
                                           Tokens<ND>& t) const {
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            t.Z[i] = zero;
#pragma unroll
            for (int j = 0; j < ND; ++j) t.Z[i] = mm(GamT[j][i], X[j], t.Z[i]);
        }
        v4f V[ND];
        float pe = 0.f, pa = 0.f, ss = 0.f;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            t.K[i] = zero;
            V[i] = zero;
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                t.K[i] = mm(sh.mem[0][j * ND + i][bl.lane], t.Z[j], t.K[i]);
                V[i] = mm(sh.mem[1][j * ND + i][bl.lane], t.Z[j], V[i]);
            }
            const v4f e = bl.rows_of(&sh.ev[0][16 * i]), a = bl.rows_of(&sh.ev[1][16 * i]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pe += e[r] * t.Z[i][r];
                pa += a[r] * t.Z[i][r];
            }
        }
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) ss += t.K[i][r] * t.K[i][r];
        const float pe_raw = xor16_32_sum(pe), pa_raw = xor16_32_sum(pa) + k.retention_bias;
        t.inv_k = rsqrtf(xor16_32_sum(ss) + 1e-6f);
        float dd = 0.f, kk = 0.f;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                t.K[i][r] *= t.inv_k;
                t.Dl[i][r] = t.K[i][r] - V[i][r];
                dd += t.Dl[i][r] * t.Dl[i][r];
                kk += t.K[i][r] * t.K[i][r];
            }
        t.dn = __builtin_amdgcn_sqrtf(xor16_32_sum(dd) + 1e-12f);
        const float ksq = xor16_32_sum(kk);
        const float amin = k.min_retention, mu = k.injection_margin, fac = k.spectral_factor;
        const float ep = fminf(10.f, fmaxf(-10.f, pe_raw)), ap = fminf(10.f, fmaxf(-10.f, pa_raw));
        const float e_pre = exp1(ep);
        const float eta = k.step_scale * (0.69314718055994531f * __builtin_amdgcn_logf(1.f + e_pre));
        const float sg = rcp1(1.f + exp1(-ap));
        t.alpha = amin + (1.f - amin) * sg;
        t.s_eta = fabsf(pe_raw) <= 10.f ? k.step_scale * e_pre * rcp1(1.f + e_pre) : 0.f;
        t.s_alpha = fabsf(pa_raw) <= 10.f ? (1.f - amin) * sg * (1.f - sg) : 0.f;
        t.inv_denom = rcp1(t.dn + 1e-6f);
        t.cap = mu * (1.f - t.alpha) * t.inv_denom;
        // eta^ = cap (1 - e^-u) and its derivatives, u = eta / cap; Taylor series below 1/4,
        // where the differences would cancel (truncated below 2e-9)
        const float u = eta * rcp1(t.cap), e_neg = exp1(-u);
        const float near1 = u * (1.f - u * (1.f / 2 - u * (1.f / 6 - u * (1.f / 24 - u * (1.f / 120 - u * (1.f / 720 -
                            u * (1.f / 5040)))))));
        const float near2 = u * u * (1.f / 2 - u * (1.f / 3 - u * (1.f / 8 - u * (1.f / 30 - u * (1.f / 144 - u * (1.f / 840 -
                            u * (1.f / 5760)))))));
        const float one_minus = u < 0.25f ? near1 : 1.f - e_neg;
        t.eff = t.cap * one_minus;
        t.deff_deta = e_neg;
        t.deff_dcap = u < 0.25f ? near2 : one_minus - u * e_neg;
        t.deff_dalpha = 0.f;
        t.deff_dksq = 0.f;
        if (k.spectral_clamp) {
            const float inv = rcp1(fmaxf(ksq, 1e-20f)), bound = fac * t.alpha * inv;
            const float lim = __uint_as_float(__float_as_uint(bound) - 1u);   // nextafter toward 0 (bound > 0)
            const bool over = t.eff > lim;
            t.eff = over ? lim : t.eff;
            t.deff_deta = over ? 0.f : t.deff_deta;
            t.deff_dcap = over ? 0.f : t.deff_dcap;
            t.deff_dalpha = over ? fac * inv : 0.f;
            t.deff_dksq = over && ksq > 1e-20f ? -bound * inv : 0.f;
        }
        if (!valid) {
            t.eff = 0.f;
            t.alpha = 1.f;
        }
        t.d = bl.decays(t.eff, t.alpha);
        v4f gram = zero;
#pragma unroll
        for (int i = 0; i < ND; ++i) gram = mm(t.K[i], t.K[i], gram);
        t.tri = bl.triangle(t.d, gram);
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            t.KT[i] = bl.transpose(t.K[i]);
            if constexpr (DELTA_T) t.DlT[i] = bl.transpose(t.Dl[i]);
        }
    }

    // The block's maps into slot w of the segment's table: X, X^T for the adjoint, Y^T.
    __device__ __forceinline__ void store_maps(const Tokens<ND>& t) const {
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        v4f S[ND], KD[ND];
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            S[j] = t.d.De_r() * t.KT[j];
            KD[j] = -(t.d.Da_r() * t.KT[j]);
        }
        bl.solve_upper(t.tri, S);
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                const v4f x = mm(KD[i], S[j], i == j ? bl.diagonal(t.d.a()) : zero);
                sh.maps[w][0][i * ND + j][bl.lane] = x;
                sh.maps[w][1][j * ND + i][bl.lane] = bl.transpose(x);
                sh.maps[w][2][i * ND + j][bl.lane] = mm(-S[i], t.DlT[j], zero);
            }
    }
    // G^T <- X^T G^T + Y^T of block b
    __device__ __forceinline__ void apply_map(int b, v4f (&GT)[ND][ND]) const {
        v4f out[ND][ND];
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) out[i][j] = sh.maps[b][2][i * ND + j][bl.lane];
#pragma unroll
        for (int m = 0; m < ND; ++m)
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const v4f x = sh.maps[b][0][m * ND + i][bl.lane];
#pragma unroll
                for (int j = 0; j < ND; ++j) out[i][j] = mm(x, GT[m][j], out[i][j]);
            }
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) GT[i][j] = out[i][j];
    }
    // H^T <- X H^T of block b
    __device__ __forceinline__ void apply_adjoint(int b, v4f (&HT)[ND][ND]) const {
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        v4f out[ND][ND];
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) out[i][j] = zero;
#pragma unroll
        for (int m = 0; m < ND; ++m)
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const v4f x = sh.maps[b][1][m * ND + i][bl.lane];
#pragma unroll
                for (int j = 0; j < ND; ++j) out[i][j] = mm(x, HT[m][j], out[i][j]);
            }
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) HT[i][j] = out[i][j];
    }
};

// Token addresses of one line: element offsets of this lane's first channel in x (and dy, dx)
// and in q (and dq).
template <int D, bool SPATIAL>
struct LineAddress {
    static constexpr int ND = D / 16;
    using Index = std::conditional_t<SPATIAL, int, int64_t>;   // a map has fewer than 2^24 pixels
    const Index N;
    int64_t xbase, qbase, qstride;
    int r_dir;
    uint32_t height, width, channels;
    float inv_h;

    __device__ __forceinline__ LineAddress(const BwdParams& p, int64_t ln, int g) : N(static_cast<Index>(p.N)) {
        const int64_t b = ln / (p.R * p.heads), head = ln % p.heads, all = p.heads * D;
        r_dir = static_cast<int>((ln / p.heads) % p.R);
        xbase = (SPATIAL ? b * N * all + head * D : ln * N * D) + 4 * g;
        qbase = SPATIAL ? xbase : p.q_raw ? (b * p.R + r_dir) * N * all + head * D + 4 * g : xbase;
        qstride = p.q_raw ? all : D;
        height = static_cast<uint32_t>(p.H);
        width = static_cast<uint32_t>(p.W);
        channels = static_cast<uint32_t>(all);
        inv_h = p.inv_h;
    }
    // Pixel of scan index t (scan_to_pixel in 32 bits).
    __device__ __forceinline__ uint32_t pixel(int t) const {
        const uint32_t orig = static_cast<uint32_t>((r_dir & 1) ? static_cast<int>(N) - 1 - t : t);
        if (r_dir < 2) return orig;
        uint32_t col, row;
        divmod24(orig, height, inv_h, col, row);
        return row * width + col;
    }
    __device__ __forceinline__ int64_t x(Index t) const {
        if constexpr (SPATIAL) return xbase + static_cast<int64_t>(pixel(t)) * channels;
        else return xbase + t * D;
    }
    __device__ __forceinline__ int64_t q(Index t, int64_t x_offset) const {
        if constexpr (SPATIAL) return x_offset;
        else return qbase + t * qstride;
    }
    // x of token slot tl of the chunk starting at token `start`, zero past the chunk.
    __device__ __forceinline__ bool load_tokens(const BwdParams& p, Index start, int tl, int C, v4f (&X)[ND]) const {
        const Index t = start + tl;
        const bool valid = tl < C && t < N;
        const int64_t at = x(valid ? t : 0);
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            X[i] = v4f{0.f, 0.f, 0.f, 0.f};
            if (valid) X[i] = load_io4(p.x, at + 16 * i, p.io_dtype);
        }
        return valid;
    }
};

template <int D, int W>
struct GainShared {
    static constexpr int ND = D / 16, NT = ND * ND;
    v4f mem[3][NT][64];                // N(M^T) of M_k, M_v, M_m
    float ev[2][D];
    float gam[D][D + 4];               // Gamma, by rows
    Scratch scratch[W];
    v4f maps[W > 1 ? W : 1][W > 1 ? 2 : 1][NT][64];   // X and (Gamma Y)^T of the segment's blocks
};

// The forward of the training path: Gamma before every chunk (for the backward) and the
// chunk-start content memories M_m Gamma (for the readout), in FP32 products throughout.
// Waves hold the blocks of a chunk; the first D / 16 waves chain the maps, one column tile of
// Gamma^T each: P <- X^T P + (Gamma Y)^T from P = Gamma^T (srnl_utw.hip).
template <int D, int W, bool SPATIAL>
__global__ __launch_bounds__(64 * W, (D == 16 ? 4 : 1)) void srnl_backward_gains_kernel(const BwdParams p) {
    constexpr int ND = D / 16, NT = ND * ND, DD = D * D;
    __shared__ GainShared<D, W> sh;
    const int w = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const Line<D, GainShared<D, W>> L{sh, w, Block(sh.scratch[w], static_cast<int>(threadIdx.x) & 63), p.k};
    const Block& bl = L.bl;
    const int lane = bl.lane, g = bl.g, c = bl.c, tau = bl.tau;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};

    const int64_t ln = xcd_remap(blockIdx.x, gridDim.x);
    const int64_t RH = p.R * p.heads, s = p.per_line ? ln : ln % RH;
    const LineAddress<D, SPATIAL> at(p, ln, g);
    using Index = typename LineAddress<D, SPATIAL>::Index;
    const int C = chunk_of(p.chunk, at.r_dir);
    const Index nc = (at.N + C - 1) / C;
    const int nb = (C + 15) / 16, nseg = (nb + W - 1) / W;
    float* const my_gam = p.states + ln * p.nc * DD;
    float* const my_content = p.content ? p.content + ln * p.nc * DD : nullptr;

    for (int t = w; t < 3 * NT; t += W) {
        const int m = t / NT, i = (t % NT) / ND, j = t % ND;
        sh.mem[m][t % NT][lane] =
            *reinterpret_cast<const v4f_any*>(p.m0[2 - m] + s * DD + (16 * j + c) * D + 16 * i + 4 * g);
    }
    if (threadIdx.x < 2 * D)
        sh.ev[threadIdx.x / D][threadIdx.x % D] = p.m0[3 + threadIdx.x / D][s * D + threadIdx.x % D];
    __syncthreads();

    v4f GamT[ND][ND];
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
        for (int j = 0; j < ND; ++j) GamT[i][j] = i == j ? bl.diagonal(1.f) : zero;
    // Tiles of (M_m Gamma)^T, spread over the waves from the last: row 16 j + c, columns
    // 16 i + 4 g.. of M_m Gamma (M_m itself for the first chunk).
    auto store_content = [&](Index ch) {
        if (my_content == nullptr) return;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j)
                if (W - 1 - (i * ND + j) % W == w) {
                    v4f m = zero;
                    if (ch == 0) m = sh.mem[2][i * ND + j][lane];
                    else
#pragma unroll
                        for (int k = 0; k < ND; ++k) {
                            v4f gam;
                            if constexpr (W == 1) gam = bl.transpose(GamT[i][k]);
                            else
#pragma unroll
                                for (int r = 0; r < 4; ++r) gam[r] = sh.gam[16 * k + 4 * g + r][16 * i + c];
                            m = mm(gam, sh.mem[2][k * ND + j][lane], m);
                        }
                    store_state4(my_content + static_cast<int64_t>(ch) * DD + (16 * j + c) * D + 16 * i + 4 * g,
                                 make_float4(m[0], m[1], m[2], m[3]), p.content_split != 0);
                }
    };
    for (Index ch = 0; ch < nc - 1; ++ch) {
        store_content(ch);
        float* const out = my_gam + static_cast<int64_t>(ch + 1) * DD;
        if constexpr (W == 1) {
            v4f X[ND], RT[ND], next[ND][ND];
            Tokens<ND> t;
            const bool valid = at.load_tokens(p, ch * C, tau, C, X);
            L.tokens(X, valid, GamT, t);
#pragma unroll
            for (int j = 0; j < ND; ++j) RT[j] = t.d.Da_r() * t.KT[j] + t.DlT[j];
            bl.solve_lower(t.tri, RT);
            // Gamma^T <- G^T Gamma^T, G = a I - R D_e K^T
            v4f G[ND][ND];
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j)
                    G[i][j] = mm(-RT[i], t.d.De_r() * t.KT[j], i == j ? bl.diagonal(t.d.a()) : zero);
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    next[i][j] = zero;
#pragma unroll
                    for (int m = 0; m < ND; ++m) next[i][j] = mm(G[m][i], GamT[m][j], next[i][j]);
                }
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    GamT[i][j] = next[i][j];
                    *reinterpret_cast<v4f_any*>(out + (16 * j + c) * D + 16 * i + 4 * g) = next[i][j];
                }
        } else {
            v4f P[ND];   // waves below ND: column tile w of the chained Gamma^T
#pragma unroll
            for (int j = 0; j < ND; ++j)
                if (w == j)
#pragma unroll
                    for (int i = 0; i < ND; ++i) P[i] = GamT[i][j];
            for (int seg = 0; seg < nseg; ++seg) {
                const int nbs = min(W, nb - seg * W);
                if (seg > 0) __syncthreads();   // the previous segment's maps are read
                if (w < nbs) {
                    v4f X[ND], S[ND], KD[ND], gd[ND];
                    Tokens<ND> t;
                    const bool valid = at.load_tokens(p, ch * C, 16 * (seg * W + w) + tau, C, X);
                    L.template tokens<false>(X, valid, GamT, t);
#pragma unroll
                    for (int j = 0; j < ND; ++j) {
                        S[j] = t.d.De_r() * t.KT[j];
                        KD[j] = -(t.d.Da_r() * t.KT[j]);
                        gd[j] = zero;   // (Gamma Delta)^T
#pragma unroll
                        for (int i = 0; i < ND; ++i) gd[j] = mm(t.Dl[i], GamT[i][j], gd[j]);
                    }
                    bl.solve_upper(t.tri, S);
#pragma unroll
                    for (int i = 0; i < ND; ++i)
#pragma unroll
                        for (int j = 0; j < ND; ++j) {
                            sh.maps[w][0][i * ND + j][lane] = mm(KD[i], S[j], i == j ? bl.diagonal(t.d.a()) : zero);
                            sh.maps[w][1][i * ND + j][lane] = mm(-S[i], gd[j], zero);
                        }
                }
                __syncthreads();
#pragma unroll
                for (int j = 0; j < ND; ++j)
                    if (w == j)
                        for (int blk = 0; blk < nbs; ++blk) {
                            v4f next[ND];
#pragma unroll
                            for (int i = 0; i < ND; ++i) {
                                next[i] = sh.maps[blk][1][i * ND + j][lane];
#pragma unroll
                                for (int m = 0; m < ND; ++m) next[i] = mm(sh.maps[blk][0][m * ND + i][lane], P[m], next[i]);
                            }
#pragma unroll
                            for (int i = 0; i < ND; ++i) P[i] = next[i];
                        }
            }
#pragma unroll
            for (int j = 0; j < ND; ++j)
                if (w == j)
#pragma unroll
                    for (int i = 0; i < ND; ++i) {
                        *reinterpret_cast<v4f*>(&sh.gam[16 * j + c][16 * i + 4 * g]) = P[i];
                        *reinterpret_cast<v4f_any*>(out + (16 * j + c) * D + 16 * i + 4 * g) = P[i];
                    }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j)
                    GamT[i][j] = *reinterpret_cast<const v4f*>(&sh.gam[16 * j + c][16 * i + 4 * g]);
        }
    }
    store_content(nc - 1);
}

template <int ND>
__device__ __forceinline__ void copy_tiles(const v4f (&from)[ND][ND], v4f (&to)[ND][ND]) {
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
        for (int j = 0; j < ND; ++j) to[i][j] = from[i][j];
}

// Readouts' gradients a wave without a block takes at most.  256 lines, backward of 8 chunks,
// d = 16, against every wave taking those of its own block: 2 of 4 waves spare, 1 readout each,
// 67 -> 60 us; 3 of 8, 2 each, 97 -> 89; 2 of 8, 3 each, 100 -> 97; 1 of 8, 7 readouts, 103 ->
// 124.  d = 32 (12 chunks): 2 of 4, 1 each, 206 -> 178; 1 of 4, 3 readouts, 218 -> 225.
template <int D>
constexpr int kSpareReadouts = D == 16 ? 3 : 2;

// Waves per SIMD the register budget is cut for.
template <int D, int W>
constexpr int kMinWaves = D == 16 ? (W == 1 ? 3 : 2) : 1;

template <int D, int W, bool SPATIAL>
__global__ __launch_bounds__(64 * W, (kMinWaves<D, W>)) void srnl_backward_blocks_kernel(const BwdParams p) {
    constexpr int ND = D / 16, NT = ND * ND, SD = 3 * D * D + 2 * D, DD = D * D;
    using Tok = Tokens<ND>;
    __shared__ Shared<D, W> sh;
    const int w = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const Line<D, Shared<D, W>> L{sh, w, Block(sh.scratch[w], static_cast<int>(threadIdx.x) & 63), p.k};
    const Block& bl = L.bl;
    const int lane = bl.lane, g = bl.g, c = bl.c, tau = bl.tau;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};

    const int64_t ln = blockIdx.x;
    const int64_t RH = p.R * p.heads, s = p.per_line ? ln : ln % RH;
    const int r_dir = static_cast<int>((ln / p.heads) % p.R);
    const int64_t head = ln % p.heads;
    const int C = chunk_of(p.chunk, r_dir);
    const LineAddress<D, SPATIAL> at_(p, ln, g);
    using Index = typename LineAddress<D, SPATIAL>::Index;
    const Index N = at_.N, nc = (N + C - 1) / C;
    const int nb = (C + 15) / 16, nseg = (nb + W - 1) / W;
    const bool q_raw = SPATIAL || p.q_raw;
    const int64_t C_all = p.heads * D;
    auto x_at = [&](Index t) { return at_.x(t); };
    auto q_at = [&](Index t, int64_t x_off) { return at_.q(t, x_off); };
    const int64_t plane = SPATIAL ? r_dir * p.B * N * C_all : 0;
    const float* const my_gam = p.states + ln * p.nc * DD;
    float* const my_seg = p.gtraj + (ln * W + w) * static_cast<int64_t>(p.segs) * DD;

    // ---- memories into LDS -------------------------------------------------------------
    for (int t = w; t < 5 * NT; t += W) {
        const int m = t / NT, i = (t % NT) / ND, j = t % ND;
        const float* src = p.m0[m == 0 || m == 2 ? 2 : m == 4 ? 0 : 1] + s * DD;
        v4f v;
#pragma unroll
        for (int r = 0; r < 4; ++r)   // N(M^T): column 16 j + c of the tile is row 16 j + c of M
            v[r] = m < 2 ? src[(16 * j + c) * D + 16 * i + 4 * g + r] : src[(16 * i + 4 * g + r) * D + 16 * j + c];
        // the gradient of y_r is the direction weight times dy: folded into the rows of M_m
        if (SPATIAL && m == 4)
            v *= *reinterpret_cast<const v4f_any*>(p.scale + r_dir * C_all + head * D + 16 * i + 4 * g);
        sh.mem[m][t % NT][lane] = v;
    }
    if (threadIdx.x < 2 * D)
        sh.ev[threadIdx.x / D][threadIdx.x % D] = p.m0[3 + threadIdx.x / D][s * D + threadIdx.x % D];
    __syncthreads();

    auto load_x = [&](Index ch, int blk, bool& valid, v4f (&X)[ND]) {
        valid = at_.load_tokens(p, ch * C, 16 * blk + tau, C, X);
    };
    auto store_dx = [&](int64_t at, v4f v) {
        if constexpr (SPATIAL) store_io4(p.dx_planes, plane + at, p.io_dtype, v);
        else *reinterpret_cast<v4f_any*>(p.dx + at) = v;
    };
    auto identity = [&](v4f (&M)[ND][ND]) {
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) M[i][j] = i == j ? bl.diagonal(1.f) : zero;
    };
    // R^T from K^T G^T of the block's entry gain (R (I + L) = G K D_a + Delta).
    auto solve_r = [&](const Tok& t, const v4f (&KG)[ND], v4f (&RT)[ND]) {
#pragma unroll
        for (int j = 0; j < ND; ++j) RT[j] = t.d.Da_r() * KG[j] + t.DlT[j];
        bl.solve_lower(t.tri, RT);
    };

    v4f GamT[ND][ND];

    // ---- chunks in reverse -------------------------------------------------------------
    v4f dMm[ND][ND], dMv[ND][ND], dMk[ND][ND], dEv[ND], dAv[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        dEv[i] = dAv[i] = zero;
#pragma unroll
        for (int j = 0; j < ND; ++j) dMm[i][j] = dMv[i][j] = dMk[i][j] = zero;
    }
    for (Index ch = nc - 1; ch >= 0; --ch) {
        v4f Gam[ND][ND];
        if (ch == 0) {
            identity(GamT);
            identity(Gam);
        } else {
            const float* src = my_gam + static_cast<int64_t>(ch) * DD;
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    GamT[i][j] = *reinterpret_cast<const v4f_any*>(src + (16 * j + c) * D + 16 * i + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) Gam[i][j][r] = src[(16 * i + 4 * g + r) * D + 16 * j + c];
                }
        }
        v4f Ep[ND][ND];   // this wave's part of dGamma_c; dGamma_{c+1} G_C^T is in the last wave's
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j) Ep[i][j] = zero;

        // Gradients of this wave's block (chunk block blk) from the adjoint H of its exit
        // gain; GTb: the transposed gain at its start (the identity when W is 1).
        auto block_gradients = [&](int blk, const Tok& t, const v4f (&X)[ND], bool valid, const v4f (&RT)[ND],
                                   const v4f (&KG)[ND], const v4f (&GTb)[ND][ND], const v4f (&HT)[ND][ND],
                                   const v4f (&H)[ND][ND]) {
            v4f RbT[ND], R[ND], Rb[ND];
            float hg = 0.f, rr = 0.f;
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                v4f kh = zero;
#pragma unroll
                for (int i = 0; i < ND; ++i) {
                    kh = mm(t.K[i], HT[i][j], kh);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if constexpr (W > 1) hg += HT[i][j][r] * GTb[i][j][r];
                        else if (i == j) hg += 4 * g + r == c ? HT[i][j][r] : 0.f;
                    }
                }
                RbT[j] = -(t.d.De_r() * kh);
            }
            hg = wave_sum(hg);
            bl.solve_upper(t.tri, RbT);
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                R[i] = bl.transpose(RT[i]);
                Rb[i] = bl.transpose(RbT[i]);
#pragma unroll
                for (int r = 0; r < 4; ++r) rr += Rb[i][r] * R[i][r];
            }
            rr = xor16_32_sum(rr);
            const float d_eff = t.eff > 0.f ? rr * rcp1(t.eff) : 0.f;
            const float d_cap = d_eff * t.deff_dcap;
            const float d_epre = d_eff * t.deff_deta * t.s_eta;
            const float cdn = -d_cap * t.cap * t.inv_denom * rcp1(t.dn), cks = 2.f * d_eff * t.deff_dksq;
            v4f P = zero, Ws, Q, first;
#pragma unroll
            for (int i = 0; i < ND; ++i) P = mm(R[i], Rb[i], P);
            const v4f PT = bl.transpose(P);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool earlier = bl.row_time(r) < tau;
                Ws[r] = earlier ? P[r] : PT[r];
                Q[r] = earlier ? t.tri.nC[r] * P[r] : 0.f;
                first[r] = earlier ? 1.f : 0.f;
            }
            Ws = bl.decayed(t.d, Ws);
            // row u, column t: the terms of pairs (s, u) with s < t
            const v4f pairs = mm(Q, first, zero);
            float kg = 0.f, kh = 0.f;
            v4f dk[ND], dv[ND], ZT[ND];
            float kdot = 0.f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                v4f hr = zero, gr = zero;
#pragma unroll
                for (int m = 0; m < ND; ++m) {
                    hr = mm(H[m][i], R[m], hr);
                    if constexpr (W > 1) gr = mm(bl.transpose(GTb[i][m]), Rb[m], gr);
                }
                if constexpr (W == 1) gr = Rb[i];
                const v4f kw = mm(t.KT[i], Ws, zero);
                dk[i] = gr * t.d.Da() - hr * t.d.De() - kw + Rb[i] + t.Dl[i] * cdn + t.K[i] * cks;
                dv[i] = -Rb[i] - t.Dl[i] * cdn;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    kdot += dk[i][r] * t.K[i][r];
                    kg += t.K[i][r] * gr[r];
                    kh += t.K[i][r] * hr[r];
                }
            }
            kdot = xor16_32_sum(kdot);
            // alpha_t <H_{t+1}, G_t>
            v4f later, before;
            bl.rows(xor16_32_sum(kg) * t.d.Da(), xor16_32_sum(kh) * t.d.De(), later, before);
            float hg_t = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                hg_t += bl.row_time(r) > tau ? pairs[r] + later[r] : bl.row_time(r) < tau ? -before[r] : 0.f;
            hg_t = xor16_32_sum(hg_t) + t.d.a() * hg;
            const float d_alpha = hg_t * rcp1(t.alpha) - d_cap * p.k.injection_margin * t.inv_denom + d_eff * t.deff_dalpha;
            const float d_apre = valid ? d_alpha * t.s_alpha : 0.f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                dk[i] = (dk[i] - t.K[i] * kdot) * t.inv_k;
                dEv[i] += t.Z[i] * d_epre;
                dAv[i] += t.Z[i] * d_apre;
                ZT[i] = bl.transpose(t.Z[i]);
            }
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const v4f dvT = bl.transpose(dv[i]), dkT = bl.transpose(dk[i]);
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    dMv[i][j] = mm(dvT, ZT[j], dMv[i][j]);
                    dMk[i][j] = mm(dkT, ZT[j], dMk[i][j]);
                }
            }
            v4f dz[ND], XT[ND];
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                dz[j] = bl.rows_of(&sh.ev[0][16 * j]) * d_epre + bl.rows_of(&sh.ev[1][16 * j]) * d_apre;
#pragma unroll
                for (int i = 0; i < ND; ++i) {
                    dz[j] = mm(sh.mem[3][i * ND + j][lane], dv[i], dz[j]);
                    dz[j] = mm(sh.mem[2][i * ND + j][lane], dk[i], dz[j]);
                }
                XT[j] = bl.transpose(X[j]);
            }
            const int64_t at = x_at(valid ? ch * C + 16 * blk + tau : 0);
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                v4f dx = zero;
#pragma unroll
                for (int i = 0; i < ND; ++i) dx = mm(Gam[i][j], dz[i], dx);
                if (valid) store_dx(at + 16 * j, dx);
                const v4f dzT = bl.transpose(dz[j]);
#pragma unroll
                for (int i = 0; i < ND; ++i) Ep[j][i] = mm(dzT, XT[i], Ep[j][i]);
            }
        };

        if (ch < nc - 1) {
            auto e_rows = [&](int m, int i) {   // tile (m, i) of dGamma_{c+1}
                v4f e;
#pragma unroll
                for (int r = 0; r < 4; ++r) e[r] = sh.E[16 * m + 4 * g + r][16 * i + c];
                return e;
            };
            Tok t;
            v4f X[ND], RT[ND], GT[ND][ND], HT[ND][ND], H[ND][ND];
            v4f GTb[ND][ND];   // G^T at the start of this wave's block of the segment
            bool valid = false;
            if constexpr (W == 1) {
                load_x(ch, 0, valid, X);
                L.tokens(X, valid, GamT, t);
                solve_r(t, t.KT, RT);
#pragma unroll
                for (int i = 0; i < ND; ++i)
#pragma unroll
                    for (int j = 0; j < ND; ++j)
                        GT[i][j] = mm(t.d.De_r() * t.KT[i], -RT[j], i == j ? bl.diagonal(t.d.a()) : zero);
            } else {
                // H^T at the chunk's exit, Gamma^T dGamma_{c+1}: a tile per wave, shared
#pragma unroll
                for (int i = 0; i < ND; ++i)
#pragma unroll
                    for (int j = 0; j < ND; ++j)
                        if (W - 1 - (i * ND + j) % W == w) {
                            v4f h = zero;
#pragma unroll
                            for (int m = 0; m < ND; ++m) h = mm(e_rows(m, i), Gam[m][j], h);
                            sh.HT[i * ND + j][lane] = h;
                        }
                identity(GT);
                for (int seg = 0; seg < nseg; ++seg) {
                    const int nbs = min(W, nb - seg * W);
                    if (nseg > 1)
#pragma unroll
                        for (int i = 0; i < NT; ++i)
                            *reinterpret_cast<v4f_any*>(my_seg + seg * DD + i * 256 + 4 * lane) = GT[i / ND][i % ND];
                    if (seg > 0) __syncthreads();   // every wave has read the previous segment's maps
                    if (w < nbs) {
                        load_x(ch, seg * W + w, valid, X);
                        L.tokens(X, valid, GamT, t);
                        L.store_maps(t);
                    }
                    __syncthreads();
                    // Up to this wave's block; the whole product for a following segment and, on
                    // the last wave, for dGamma_{c+1} G_C^T.  (The adjoint below is the other way
                    // round, so no wave walks the chunk twice.)
                    const int upto = w == W - 1 || seg + 1 < nseg ? nbs : w < nbs ? w : 0;
                    for (int blk = 0; blk < upto; ++blk) {
                        if (blk == w) copy_tiles(GT, GTb);
                        L.apply_map(blk, GT);
                    }
                    if (upto == w) copy_tiles(GT, GTb);
                }
            }
            // dGamma_{c+1} G_C^T and the adjoint of the chunk gain, dG_C = Gamma^T dGamma_{c+1}
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    if constexpr (W == 1) {
                        HT[i][j] = zero;
#pragma unroll
                        for (int m = 0; m < ND; ++m) HT[i][j] = mm(e_rows(m, i), Gam[m][j], HT[i][j]);
                        H[j][i] = bl.transpose(HT[i][j]);
                    } else {
                        HT[i][j] = sh.HT[i * ND + j][lane];
                    }
                    if (W == 1 || w == W - 1)
#pragma unroll
                        for (int m = 0; m < ND; ++m)
                            Ep[i][j] = mm(*reinterpret_cast<const v4f*>(&sh.E[16 * i + c][16 * m + 4 * g]), GT[m][j], Ep[i][j]);
                }
            if constexpr (W == 1) {
                block_gradients(0, t, X, valid, RT, t.KT, GT, HT, H);
            } else {
                for (int seg = nseg - 1; seg >= 0; --seg) {
                    const int nbs = min(W, nb - seg * W);
                    if (seg != nseg - 1) {
#pragma unroll
                        for (int i = 0; i < NT; ++i)
                            GTb[i / ND][i % ND] = *reinterpret_cast<const v4f_any*>(my_seg + seg * DD + i * 256 + 4 * lane);
                        __syncthreads();   // every wave has read the later segment's maps
                        if (w < nbs) {
                            load_x(ch, seg * W + w, valid, X);
                            L.tokens(X, valid, GamT, t);
                            L.store_maps(t);
                        }
                        __syncthreads();
                        for (int blk = 0; blk < w; ++blk) L.apply_map(blk, GTb);   // a segment with a successor is full
                    }
                    // H^T from the segment's exit to this block's exit (and on to the segment's
                    // start when an earlier segment continues from there)
                    v4f HTb[ND][ND];
                    for (int blk = nbs - 1; blk >= 0; --blk) {
                        if (blk == w) copy_tiles(HT, HTb);
                        if (seg == 0 && blk <= w) break;
                        L.apply_adjoint(blk, HT);
                    }
                    if (w < nbs) {
#pragma unroll
                        for (int i = 0; i < ND; ++i)
#pragma unroll
                            for (int j = 0; j < ND; ++j) H[i][j] = bl.transpose(HTb[j][i]);
                        v4f KG[ND];
#pragma unroll
                        for (int j = 0; j < ND; ++j) {
                            KG[j] = zero;
#pragma unroll
                            for (int i = 0; i < ND; ++i) KG[j] = mm(t.K[i], GTb[i][j], KG[j]);
                        }
                        solve_r(t, KG, RT);
                        block_gradients(seg * W + w, t, X, valid, RT, KG, GTb, HTb, H);
                    }
                }
            }
        }

        // Readout: y = M_m Gamma q^ of every token of the chunk.
        // Waves without a block of the chunk take it while the others are in their gradients, where
        // that leaves a wave few enough of them (kSpareReadouts).
        const int spare = ch < nc - 1 ? W - nb : 0;
        const int idle = spare > 0 && nb <= kSpareReadouts<D> * spare ? spare : 0;
        const int first = idle == 0 ? w : w >= nb ? w - nb : nb;
        for (int blk = first; blk < nb; blk += idle > 0 ? idle : W) {
            const int tl = 16 * blk + tau;
            const Index tok = ch * C + tl;
            const bool valid = tl < C && tok < N;
            const int64_t at = x_at(valid ? tok : 0), qat = q_at(valid ? tok : 0, at);
            v4f q[ND], dy[ND];
            float qq = 0.f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                q[i] = dy[i] = zero;
                if (valid) {
                    q[i] = load_io4(p.q, qat + 16 * i, q_raw ? p.io_dtype : VH_DTYPE_F32);
                    dy[i] = *reinterpret_cast<const v4f_any*>(p.dy + at + 16 * i);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) qq += q[i][r] * q[i][r];
            }
            float qinv = 1.f;
            if (q_raw) qinv = 1.f / fmaxf(sqrtf(xor16_32_sum(qq)), 1e-12f);
            v4f dp[ND], qT[ND], dpT[ND];
#pragma unroll
            for (int i = 0; i < ND; ++i) q[i] *= qinv;
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                dp[j] = zero;
#pragma unroll
                for (int i = 0; i < ND; ++i) dp[j] = mm(sh.mem[4][i * ND + j][lane], dy[i], dp[j]);
                qT[j] = bl.transpose(q[j]);
                dpT[j] = bl.transpose(dp[j]);
            }
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                v4f pT = zero;
#pragma unroll
                for (int i = 0; i < ND; ++i) pT = mm(q[i], GamT[i][j], pT);
#pragma unroll
                for (int i = 0; i < ND; ++i) {
                    dMm[i][j] = mm(bl.transpose(dy[i]), pT, dMm[i][j]);
                    Ep[i][j] = mm(dpT[i], qT[j], Ep[i][j]);
                }
            }
            v4f dq[ND];
            float qdot = 0.f;
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                dq[j] = zero;
#pragma unroll
                for (int i = 0; i < ND; ++i) dq[j] = mm(Gam[i][j], dp[i], dq[j]);
#pragma unroll
                for (int r = 0; r < 4; ++r) qdot += dq[j][r] * q[j][r];
            }
            qdot = xor16_32_sum(qdot);
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                if (q_raw) dq[j] = (qinv > 9.999e11f ? dq[j] : dq[j] - q[j] * qdot) * qinv;
                if (valid) {
                    if constexpr (SPATIAL) store_io4(p.dq_planes, plane + qat + 16 * j, p.io_dtype, dq[j]);
                    else *reinterpret_cast<v4f_any*>(p.dq + qat + 16 * j) = dq[j];
                    if (ch == nc - 1) store_dx(at + 16 * j, zero);   // the last chunk's x reaches no output
                }
            }
        }

        // dGamma_c: the waves' parts, in wave order.
        if constexpr (W > 1) {
            __syncthreads();   // every wave has read the maps and dGamma_{c+1}
#pragma unroll
            for (int i = 0; i < NT; ++i) sh.maps[w][0][i][lane] = Ep[i / ND][i % ND];
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j)
                if ((i * ND + j) % W == w) {
                    v4f e = zero;
                    if constexpr (W == 1) e = Ep[i][j];
                    else
                        for (int v = 0; v < W; ++v) e += sh.maps[v][0][i * ND + j][lane];
#pragma unroll
                    for (int r = 0; r < 4; ++r) sh.E[16 * i + 4 * g + r][16 * j + c] = e[r];
                }
        __syncthreads();
    }

    // ---- the line's gradient of its initial memories -------------------------------------
    float* const dst = p.dline + ln * SD;
    auto store_matrix = [&](int m, const v4f (&M)[ND][ND]) {
        if constexpr (W > 1) {
#pragma unroll
            for (int i = 0; i < NT; ++i) sh.maps[w][0][i][lane] = M[i / ND][i % ND];
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < NT; ++i)
            if (i % W == w) {
                v4f e = M[i / ND][i % ND];
                if constexpr (W > 1) {
                    e = zero;
                    for (int v = 0; v < W; ++v) e += sh.maps[v][0][i][lane];
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[m * DD + (16 * (i / ND) + 4 * g + r) * D + 16 * (i % ND) + c] = e[r];
            }
        if constexpr (W > 1) __syncthreads();
    };
    store_matrix(0, dMm);
    store_matrix(1, dMv);
    store_matrix(2, dMk);
    // gate vectors: the 16 slot columns, then the waves (through the transpose scratch)
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float e = row_group_sum<16>(dEv[i][r]), a = row_group_sum<16>(dAv[i][r]);
            sh.scratch[w].tr[16 * i + 4 * g + r] = e;
            sh.scratch[w].tr[D + 16 * i + 4 * g + r] = a;
        }
    __syncthreads();
    if (threadIdx.x < 2 * D) {
        float v = 0.f;
        for (int u = 0; u < W; ++u) v += sh.scratch[u].tr[threadIdx.x];
        dst[3 * DD + threadIdx.x] = v;
    }
}

}  // namespace

// Waves per line: one 16-token block each, up to 8 (4 at d = 32, where a wave's registers
// and the map table are four times as large); longer chunks run in segments.  With a compute
// unit for every line (256), twice that: the spare waves take the readout's gradients.  256
// lines, forward + backward: d = 16, 28 x 28 maps 272 -> 223 us, 64 x 64 628 -> 565; d = 32,
// 28 x 28 577 -> 470.  With more lines the spare waves would keep a second line off the unit.
int bwd_block_waves(int head_dim, int64_t max_chunk, int64_t lines) {
    const int most = head_dim == 16 ? 8 : 4;
    int w = 1;
    while (w < most && 16 * w < max_chunk) w *= 2;
    if (w > 1 && w < most && lines <= 256) w *= 2;
    return w;
}

namespace {

template <typename F>
void by_shape(int head_dim, int waves, F&& go) {
    auto by_waves = [&](auto d) {
        switch (waves) {
            case 1: go(d, std::integral_constant<int, 1>{}); break;
            case 2: go(d, std::integral_constant<int, 2>{}); break;
            case 4: go(d, std::integral_constant<int, 4>{}); break;
            default:
                if constexpr (decltype(d)::value == 16) go(d, std::integral_constant<int, 8>{});
                break;
        }
    };
    if (head_dim == 16) by_waves(std::integral_constant<int, 16>{});
    else by_waves(std::integral_constant<int, 32>{});
}

}  // namespace

int launch_backward_gains(const BwdParams& p, bool spatial, int head_dim, int waves, int64_t lines, hipStream_t stream) {
    by_shape(head_dim, waves, [&](auto d, auto w) {
        constexpr int D = decltype(d)::value, W = decltype(w)::value;
        const dim3 grid(static_cast<unsigned>(lines)), block(64 * W);
        if (spatial) hipLaunchKernelGGL((srnl_backward_gains_kernel<D, W, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((srnl_backward_gains_kernel<D, W, false>), grid, block, 0, stream, p);
    });
    return check_launch("srnl_backward_gains_kernel");
}

int launch_backward_blocks(const BwdParams& p, int head_dim, int waves, int64_t lines, hipStream_t stream) {
    by_shape(head_dim, waves, [&](auto d, auto w) {
        constexpr int D = decltype(d)::value, W = decltype(w)::value;
        const dim3 grid(static_cast<unsigned>(lines)), block(64 * W);
        if (p.scale) hipLaunchKernelGGL((srnl_backward_blocks_kernel<D, W, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((srnl_backward_blocks_kernel<D, W, false>), grid, block, 0, stream, p);
    });
    return check_launch("srnl_backward_blocks_kernel");
}

}  // namespace vh
