// Training-side kernels of a bf16 linear layer out = x W^T + b whose operands are the rows of
// channels-last maps: the operands autocast casts on every call, and the gradients of W and b.
// The products with x and dy on the left (the forward and dx = dy W) are 1x1 convolutions
// (pointwise.hip).
#include <algorithm>

#include "srnl_device.h"

namespace vh {
namespace {

typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));
typedef unsigned short us8_any __attribute__((ext_vector_type(8), aligned(2)));

// W [N, K] and b [N] (any io dtype) as the matrix-core operands: W and W^T in bf16, b rounded to
// bf16 and kept in FP32.  One launch instead of four casts and a transpose copy.
template <typename T>
__global__ __launch_bounds__(256) void linear_operands_kernel(const T* w, const T* b, int64_t N, int64_t K, bf16_t* w16,
                                                              bf16_t* wt16, float* b32) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx < N * K) {
        const bf16_t v = from_f32<bf16_t>(to_f32(w[idx]));
        w16[idx] = v;
        wt16[(idx % K) * N + idx / K] = v;
    }
    if (idx < N) b32[idx] = to_f32(from_f32<bf16_t>(to_f32(b[idx])));
}

constexpr int kTok = 64;            // tokens per step
constexpr int kSide = 128;          // channels of dy and of x per workgroup, at most
constexpr int kRow = kTok * 2 + 8;  // bytes per LDS row (one channel's tokens): 8-byte aligned

struct WeightGradParams {
    const bf16_t *dy, *x;   // [M, N], [M, K]
    float* part;            // [gridDim.x, N * K + N]
    int64_t M, N, K, tokens;   // tokens: per workgroup
};

// Partial dW = dy^T x and db = sum dy over a range of tokens, for a block of up to 128 x 128
// (blockIdx.y, z).  The sum runs over tokens, so both operands are wanted token-minor while the
// maps are channel-minor: each step of 64 tokens goes through LDS transposed (two tokens of a
// channel per 4-byte write), the next step's loads in flight meanwhile.  Wave w takes dy
// channels 32 w.. of the block; db is a product with ones.  Bound by HBM at these widths (2 N K
// flops against 2 (N + K) bytes per token).  B 128, 14 x 14 x 128 channels: 12.8 MB, 98
// workgroups, 17 us and 4 us for the sum (a library product, whose few output tiles each ran
// through all 25,088 tokens, and a sum for db: 105 + 17 us); B 64, 56 x 56 x 32: 25.7 MB, 15 +
// 7 us (148 + 16 us).
__global__ __launch_bounds__(256) void linear_weight_grad_kernel(const WeightGradParams p) {
    __shared__ __align__(16) unsigned char lds[2][kSide * kRow];
    const int tid = static_cast<int>(threadIdx.x), wv = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int64_t n0 = static_cast<int64_t>(blockIdx.y) * kSide, k0 = static_cast<int64_t>(blockIdx.z) * kSide;
    const int nn = static_cast<int>(min<int64_t>(kSide, p.N - n0)), nk = static_cast<int>(min<int64_t>(kSide, p.K - k0));
    const int64_t first = static_cast<int64_t>(blockIdx.x) * p.tokens, last = min(p.M, first + p.tokens);
    v4f acc[2][8], ones_acc[2];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ones_acc[i] = zero;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = zero;
    }
    v8bf_t ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = static_cast<__bf16>(1.f);

    // item (pair of tokens, group of 8 channels) of operand o: two 16-byte loads, 8 LDS writes
    struct Item {
        us8_any a, b;
    };
    Item items[2][2];
    auto load = [&](int64_t t0) {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int groups = (o ? nk : nn) / 8;
            const int64_t stride = o ? p.K : p.N;
            const uint16_t* src = reinterpret_cast<const uint16_t*>(o ? p.x + k0 : p.dy + n0);
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const int idx = tid + 256 * it, pair = idx / groups, cg = idx % groups;
                us8_any zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
                items[o][it] = {zero8, zero8};
                if (pair < kTok / 2) {
                    const int64_t t = t0 + 2 * pair;
                    if (t < last) items[o][it].a = *reinterpret_cast<const us8_any*>(src + t * stride + 8 * cg);
                    if (t + 1 < last) items[o][it].b = *reinterpret_cast<const us8_any*>(src + (t + 1) * stride + 8 * cg);
                }
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int groups = (o ? nk : nn) / 8;
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const int idx = tid + 256 * it, pair = idx / groups, cg = idx % groups;
                if (pair < kTok / 2)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        *reinterpret_cast<uint32_t*>(&lds[o][(8 * cg + j) * kRow + 4 * pair]) =
                            static_cast<uint32_t>(items[o][it].a[j]) | (static_cast<uint32_t>(items[o][it].b[j]) << 16);
            }
        }
    };
    // eight consecutive tokens (32 step + 8 g ..) of channel row of operand o
    auto operand = [&](int o, int row, int step) {
        const uint2* q = reinterpret_cast<const uint2*>(&lds[o][row * kRow + 64 * step + 16 * g]);
        const uint2 a = q[0], b = q[1];
        return __builtin_bit_cast(v8bf_t, make_uint4(a.x, a.y, b.x, b.y));
    };

    if (first < last) load(first);
    for (int64_t t0 = first; t0 < last; t0 += kTok) {
        store();
        __syncthreads();
        if (t0 + kTok < last) load(t0 + kTok);
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            v8bf_t a[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (32 * wv + 16 * i < nn) {
                    a[i] = operand(0, 32 * wv + 16 * i + r, step);
                    if (k0 == 0) ones_acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], ones, ones_acc[i], 0, 0, 0);
                }
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (16 * j < nk) {
                    const v8bf_t b = operand(1, 16 * j + r, step);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        if (32 * wv + 16 * i < nn)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[i][j], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    float* const out = p.part + static_cast<int64_t>(blockIdx.x) * (p.N * p.K + p.N);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (32 * wv + 16 * i >= nn) continue;
        const int64_t row = n0 + 32 * wv + 16 * i + 4 * g;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (16 * j < nk) out[(row + q) * p.K + k0 + 16 * j + r] = acc[i][j][q];
            if (k0 == 0 && r == 0) out[p.N * p.K + row + q] = ones_acc[i][q];
        }
    }
}

// Sums of the partial rows: 32 values and 8 interleaved parts per workgroup, added in order.
__global__ __launch_bounds__(256) void linear_grad_reduce_kernel(const float* part, int64_t parts, int64_t width,
                                                                 int64_t weights, float* dw, float* db) {
    __shared__ float sums[8][32];
    const int lane = static_cast<int>(threadIdx.x) & 31, row = static_cast<int>(threadIdx.x) >> 5;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 32 + lane;
    float acc = 0.f;
    if (idx < width) {
#pragma unroll 4
        for (int64_t i = row; i < parts; i += 8) acc += part[i * width + idx];
    }
    sums[row][lane] = acc;
    __syncthreads();
    if (row != 0 || idx >= width) return;
#pragma unroll
    for (int i = 1; i < 8; ++i) acc += sums[i][lane];
    if (idx < weights) dw[idx] = acc;
    else db[idx - weights] = acc;
}

// Workgroups over the tokens: about 256 tokens each (whole steps of 64; M = 257 gives 192 and
// 65), at most 512 of them, and partial sums of at most 8 MB unless a single part is larger,
// written and read once more (at 256 tokens and 128 + 128 channels a workgroup reads 128 KB and
// writes 64).
int64_t weight_grad_parts(int64_t M, int64_t N, int64_t K) {
    const int64_t width = N * K + N;
    return std::max<int64_t>(1, std::min({(M + 255) / 256, static_cast<int64_t>(512), (int64_t(2) << 20) / width}));
}

}  // namespace
}  // namespace vh

using namespace vh;

extern "C" {

int vh_linear_operands(const void* weight, const void* bias, int32_t dtype, int64_t N, int64_t K, void* w16, void* wt16,
                       float* b32, void* stream) {
    VH_REQUIRE(weight && bias && w16 && wt16 && b32, VH_ERR_ARG, "linear operand pointers must not be null");
    VH_REQUIRE(N > 0 && K > 0 && N * K < (int64_t(1) << 31), VH_ERR_SHAPE, "linear operands expect a nonempty weight");
    VH_REQUIRE(valid_dtype(dtype), VH_ERR_DTYPE, "unsupported dtype code %d", dtype);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>((std::max(N * K, N) + 255) / 256));
    auto go = [&](auto tv) {
        using T = decltype(tv);
        hipLaunchKernelGGL(linear_operands_kernel<T>, grid, dim3(256), 0, s, static_cast<const T*>(weight),
                           static_cast<const T*>(bias), N, K, static_cast<bf16_t*>(w16), static_cast<bf16_t*>(wt16), b32);
    };
    if (dtype == VH_DTYPE_F32) go(float{});
    else if (dtype == VH_DTYPE_BF16) go(bf16_t{});
    else go(f16_t{});
    return check_launch("linear_operands_kernel");
}

size_t vh_linear_weight_grad_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || N % 16 != 0 || K % 16 != 0) return 0;
    return static_cast<size_t>(weight_grad_parts(M, N, K) * (N * K + N)) * sizeof(float);
}

int vh_linear_weight_grad(const void* dy, const void* x, int64_t M, int64_t N, int64_t K, float* dw, float* db,
                          void* workspace, size_t workspace_bytes, void* stream) {
    VH_REQUIRE(dy && x && dw && db, VH_ERR_ARG, "linear weight gradient pointers must not be null");
    VH_REQUIRE(M > 0 && N > 0 && K > 0 && N % 16 == 0 && K % 16 == 0, VH_ERR_SHAPE,
               "linear weight gradient expects widths that are multiples of 16, got %lld and %lld", (long long)N,
               (long long)K);
    VH_REQUIRE(N * K < (int64_t(1) << 31) && M * std::max(N, K) < (int64_t(1) << 40), VH_ERR_SHAPE,
               "linear weight gradient operands too large");
    const size_t need = vh_linear_weight_grad_workspace_bytes(M, N, K);
    VH_REQUIRE(workspace && workspace_bytes >= need, VH_ERR_WORKSPACE, "linear weight gradient needs %zu bytes, got %zu",
               need, workspace ? workspace_bytes : (size_t)0);
    WeightGradParams p{};
    p.dy = static_cast<const bf16_t*>(dy);
    p.x = static_cast<const bf16_t*>(x);
    p.part = static_cast<float*>(workspace);
    p.M = M; p.N = N; p.K = K;
    const int64_t parts = weight_grad_parts(M, N, K);
    p.tokens = ((M + parts - 1) / parts + kTok - 1) / kTok * kTok;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(parts), static_cast<unsigned>((N + kSide - 1) / kSide),
                    static_cast<unsigned>((K + kSide - 1) / kSide));
    hipLaunchKernelGGL(linear_weight_grad_kernel, grid, dim3(256), 0, s, p);
    const int rc = check_launch("linear_weight_grad_kernel");
    if (rc) return rc;
    const int64_t width = N * K + N;
    hipLaunchKernelGGL(linear_grad_reduce_kernel, dim3(static_cast<unsigned>((width + 31) / 32)), dim3(256), 0, s, p.part,
                       parts, width, N * K, dw, db);
    return check_launch("linear_grad_reduce_kernel");
}

}  // extern "C"
