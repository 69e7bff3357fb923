// The 16-token block form on the FP32 matrix cores: tile products, token order, decays and
// triangular solves shared by the scans with one workgroup per line (srnl_utw.hip,
// srnl_utw32.hip) and the backward (srnl_backward_blocks.hip).
//
// A tile is 4 registers: lane (g = l / 16, c = l % 16) holds rows 4g..4g+3 of column c, which
// is what the matrix core returns, the B operand of that matrix and the A operand of its
// transpose; so mm(A, B) = A^T B needs no data movement, and where a transpose is needed it
// goes through wave-private LDS.  Token slots are permuted: slot index n stands for time
// 4 (n % 4) + n / 4 of the block, which puts four consecutive times into one register index,
// so one rank-4 matrix instruction eliminates them: a 16 x 16 triangular solve is 7
// instructions, with the 4 x 4 diagonal inverses formed on the VALU (solving by columns on
// the VALU took about 1,500 cycles against 350).
#pragma once

#include "srnl_device.h"

namespace vh {
namespace blocks {

constexpr int kTrStride = 20;   // floats per row of the transpose scratch (16-byte aligned rows)

// acc + A^T B
__device__ __forceinline__ v4f mm(v4f a, v4f b, v4f acc) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mfma4(a[j], b[j], acc);
    return acc;
}

template <int CTRL>
__device__ __forceinline__ float dpp0(float v) {   // 0 where the source lane is outside the row
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

template <int CTRL>
__device__ __forceinline__ float dpp1(float v) {   // 1 where the source lane is outside the row
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(1.f), __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// 1 / x within about one ulp: hardware approximation and one correction.
__device__ __forceinline__ float rcp1(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, r, 1.f), r, r);
}

// Wave-private LDS of a block.
struct Scratch {
    float tr[16 * kTrStride];   // transposes
    float sc[2][16];            // per-slot scalars, read four rows at a time
    float diag[64];             // the 4 x 4 diagonal blocks of L, negated
};

// Decays of a block, from eta^ and the retentions of its slots (0 and 1 past the chunk).  With
// a_t the product of the retentions before slot t, head = a_8 that of the first 8 times and
// tail that of the last 8,
//   rho_s = eta^_s head / a_{s+1},  kappa_t = a_t / head,
// so eta^_s a_t / a_{s+1} = rho_s kappa_t, D_e = diag(eta^_t a / a_{t+1}) = tail rho and D_a =
// diag(a_t) = head kappa.  Taken about the middle every factor stays inside 2^+-117 for the
// smallest retention the gate clamps allow.  By column, and for the lane's four rows.
//
// The products are formed by multiplication, at most five roundings each.  As 2^ of prefix
// sums of log2 they took the same time (4,096 lines of 196 tokens, d = 16, chunks of 14: scan
// 44 us, backward 139 against 140 us now), but saturated gates sum to 231 and the difference
// of two such sums lost 8 bits: with gate vectors of N(0, 2^2) gradients were 1.1 to 1.6 times
// (geometric means over seeds; up to 17 times) as far from 64 bits as token-by-token products,
// now 0.8 to 1.2 times.
struct Decays {
    v4f rho_r, kappa_r;
    float rho, kappa, head, tail;
    __device__ __forceinline__ float De() const { return rho * tail; }
    __device__ __forceinline__ float Da() const { return kappa * head; }
    __device__ __forceinline__ v4f De_r() const { return rho_r * scalar(tail); }
    __device__ __forceinline__ v4f Da_r() const { return kappa_r * scalar(head); }
    __device__ __forceinline__ float a() const { return head * tail; }

private:
    // The asm keeps the compiler from widening the load to a vector, which left the struct in
    // scratch memory.
    static __device__ __forceinline__ float scalar(float v) {
        asm("" : "+v"(v));
        return v;
    }
};
// L[s][t] = rho_s kappa_t (k_s . k_t) above the diagonal: the symmetric tile -L - L^T, and this
// lane's entry of the inverses of the 4 x 4 diagonal blocks for the lower and the upper solve.
struct Triangle {
    v4f nC;
    float dl, du;
};

struct Block {
    Scratch& s;
    const int lane, g, c, tau;   // tau: time of slot c within the block

    __device__ __forceinline__ Block(Scratch& scratch, int l)
        : s(scratch), lane(l), g(l >> 4), c(l & 15), tau(4 * (l & 3) + ((l & 15) >> 2)) {}

    __device__ __forceinline__ v4f transpose(v4f v) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) s.tr[(4 * g + i) * kTrStride + c] = v[i];
        __builtin_amdgcn_wave_barrier();
        const v4f r = *reinterpret_cast<const v4f*>(&s.tr[c * kTrStride + 4 * g]);
        __builtin_amdgcn_wave_barrier();
        return r;
    }
    __device__ __forceinline__ v4f rows_of(const float* p) const { return *reinterpret_cast<const v4f*>(p + 4 * g); }
    // Two values per slot column (the same in every row of lanes) as those of the lane's rows.
    __device__ __forceinline__ void rows(float u, float v, v4f& u_r, v4f& v_r) const {
        s.sc[0][c] = u;
        s.sc[1][c] = v;
        __builtin_amdgcn_wave_barrier();
        u_r = rows_of(s.sc[0]);
        v_r = rows_of(s.sc[1]);
        __builtin_amdgcn_wave_barrier();
    }
    __device__ __forceinline__ int row_time(int i) const { return 4 * i + g; }
    __device__ __forceinline__ v4f diagonal(float v) const {   // v I as a tile
        v4f r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = 4 * g + i == c ? v : 0.f;
        return r;
    }

    __device__ __forceinline__ Decays decays(float eff, float alpha) const {
        Decays d;
        float incl = alpha * dpp1<0x114>(alpha);   // within the slot's group of four times
        incl *= dpp1<0x118>(incl);
        const float excl = dpp1<0x114>(incl);
        float t = alpha * dpp0<0x128>(alpha);      // the group's product
        t *= dpp0<0x124>(t);
        const float t0 = dpp0<0x00>(t), t1 = dpp0<0x55>(t), t2 = dpp0<0xAA>(t), t3 = dpp0<0xFF>(t);   // of each quad lane
        d.head = t0 * t1;
        d.tail = t2 * t3;
        // a at the group's start = head num / den
        const int j = c & 3;
        const float num = j == 3 ? t2 : 1.f, den = j == 0 ? d.head : j == 1 ? t1 : 1.f;
        d.kappa = num * excl * rcp1(den);
        d.rho = eff * den * rcp1(num * incl);
        rows(d.rho, d.kappa, d.rho_r, d.kappa_r);
        return d;
    }
    // v scaled by eta^_s a_t / a_{s+1} of the earlier slot s and the later slot t of (row,
    // column); zero on the diagonal
    __device__ __forceinline__ v4f decayed(Decays d, v4f v) const {
        v4f r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool row_first = row_time(i) < tau;
            const float rho_r = d.rho_r[i], kappa_r = d.kappa_r[i], rho = d.rho, kappa = d.kappa;
            const float first = row_first ? rho_r : rho, second = row_first ? kappa : kappa_r;
            r[i] = row_time(i) == tau ? 0.f : v[i] * first * second;
        }
        return r;
    }

    __device__ __forceinline__ Triangle triangle(Decays d, v4f gram) const {
        Triangle t;
        t.nC = decayed(d, -gram);
        // Inverse of the 4 x 4 unit triangle of this slot's group of four times: this lane's
        // entry is that of times min(g, f), max(g, f) of group c % 4, f = c / 4.
        const int grp = c & 3, f = c >> 2;
        s.diag[grp * 16 + 4 * g + f] = grp == 0 ? t.nC[0] : grp == 1 ? t.nC[1] : grp == 2 ? t.nC[2] : t.nC[3];
        __builtin_amdgcn_wave_barrier();
        const v4f r0 = *reinterpret_cast<const v4f*>(s.diag + grp * 16);
        const v4f r1 = *reinterpret_cast<const v4f*>(s.diag + grp * 16 + 4);
        const v4f r2 = *reinterpret_cast<const v4f*>(s.diag + grp * 16 + 8);
        __builtin_amdgcn_wave_barrier();
        // r holds N = -L: (I - N)^-1 = I + N + N^2 + N^3
        const float t02 = r0[2] + r0[1] * r1[2], t13 = r1[3] + r1[2] * r2[3];
        const float t03 = r0[3] + r0[1] * t13 + r0[2] * r2[3];
        const int lo = min(g, f), hi = max(g, f);
        const float from0 = hi == 1 ? r0[1] : hi == 2 ? t02 : t03, from1 = hi == 2 ? r1[2] : t13;
        const float inv = lo == 0 ? from0 : lo == 1 ? from1 : r2[3];
        t.dl = g < f ? inv : 0.f;
        t.du = f < g ? inv : 0.f;
        return t;
    }

    // B <- (I + L^T)^-1 B and B <- (I + L)^-1 B for token-row tiles.
    template <int ND>
    __device__ __forceinline__ void solve_lower(const Triangle& t, v4f (&b)[ND]) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float a1 = (c & 3) == k ? t.dl : 0.f, a2 = (c & 3) > k ? t.nC[k] : 0.f;
#pragma unroll
            for (int j = 0; j < ND; ++j) b[j] = mfma4(a1, b[j][k], b[j]);
            if (k < 3)
#pragma unroll
                for (int j = 0; j < ND; ++j) b[j] = mfma4(a2, b[j][k], b[j]);
        }
    }
    template <int ND>
    __device__ __forceinline__ void solve_upper(const Triangle& t, v4f (&b)[ND]) const {
#pragma unroll
        for (int k = 3; k >= 0; --k) {
            const float a1 = (c & 3) == k ? t.du : 0.f, a2 = (c & 3) < k ? t.nC[k] : 0.f;
#pragma unroll
            for (int j = 0; j < ND; ++j) b[j] = mfma4(a1, b[j][k], b[j]);
            if (k > 0)
#pragma unroll
                for (int j = 0; j < ND; ++j) b[j] = mfma4(a2, b[j][k], b[j]);
        }
    }
};

}  // namespace blocks
}  // namespace vh
