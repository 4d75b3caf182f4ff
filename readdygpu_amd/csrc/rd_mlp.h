// rd_mlp.h -- BF16 MLP 3 -> 64 -> 64 -> 64 -> 3 (SiLU) on gfx950 MFMA.
//
// A wave evaluates tiles of 16 samples with v_mfma_f32_16x16x32_bf16 (FP32
// accumulation).  Lane l = 16 g + j holds, for sample j of the tile and every
// feature tile ti, the four features 16 ti + 4 g + r, r = 0..3:
// exactly the accumulator layout of the 16x16 MFMA (column j, rows 4g + r).
// The same registers serve as the B operand of the next layer when the
// weights' K order is permuted to match: logical k = 8 g + t of K-block kb is
// feature F(kb, g, t) = (2 kb + t/4) 16 + 4 g + t%4.  Activations therefore
// never leave registers in the forward pass.  Layer 1 (K = 3) runs on the
// VALU in FP32 (positions need more than BF16's 8 bits); layer 4 runs on MFMA
// with its 3 output rows padded to 16.
//
// Weight vector (FP32 master, 8771 values):
//   W1[64][3] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[3][64] b4[3]
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define RD_MLP_NPARAM 8771
#define RD_MLP_W1 0
#define RD_MLP_B1 192
#define RD_MLP_W2 256
#define RD_MLP_B2 4352
#define RD_MLP_W3 4416
#define RD_MLP_B3 8512
#define RD_MLP_W4 8576
#define RD_MLP_B4 8768
#define RD_MLP_ROW 8776          // partial-gradient row: 8771 grads + loss, padded

typedef __bf16 rd_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rd_f32x4 __attribute__((ext_vector_type(4)));

// BF16 weights in MFMA A-operand order (16 B per lane per fragment)
struct RdMlpPack {
    rd_bf16x8 w2[4][2][64];      // A = W2, K permuted           [out tile][kb][lane]
    rd_bf16x8 w3[4][2][64];
    rd_bf16x8 w4[2][64];         // A = W4, rows 3..15 zero
    rd_bf16x8 w2t[4][2][64];     // A = W2^T, K permuted (backward)
    rd_bf16x8 w3t[4][2][64];
    rd_bf16x8 w4t[4][64];        // A = W4^T, K = 3 real of 32
    float w1[64 * 3];            // BF16-rounded W1 as FP32
    float b1[64], b2[64], b3[64], b4[4];
    // inference copies: layer 1 and the biases times -log2(e), W4 times
    // -ln 2 (the forward pass then works on -log2(e) z throughout)
    float w1s[64 * 3];
    float b1s[64], b2s[64], b3s[64];
    rd_bf16x8 w4s[2][64];
};

#define RD_MLP_NLOG2E -1.44269504f   // -log2(e)
#define RD_MLP_NLN2 -0.693147181f    // -ln(2) = 1 / -log2(e)

// position normalisation and output scale of a trained surrogate
struct RdMlpNorm {
    float lo[3];
    float sc[3];                 // 2 / (hi - lo)
    float gscale;                // output * gscale = dU/dx
    float pad;
};

// K permutation: feature held by (K-block kb, lane group g, element t)
__host__ __device__ inline int rd_mlp_feat(int kb, int g, int t) { return (2 * kb + t / 4) * 16 + 4 * g + (t & 3); }

// SiLU with the hardware exp2 and reciprocal (v_exp_f32, v_rcp_f32: one
// transcendental each, ~1 ulp), not the IEEE division sequence
__device__ __forceinline__ float rd_sigmoid(float z)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504f));
}
// derivative of SiLU from z and its sigmoid s
__device__ __forceinline__ float rd_dsilu(float z, float s) { return s * (1.0f + z * (1.0f - s)); }

// B operand of K-block kb from the lane's activations of one sample tile
__device__ __forceinline__ rd_bf16x8 rd_mlp_bop(const float (&a)[4][4], int kb)
{
    rd_bf16x8 v;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = (__bf16)a[2 * kb + t / 4][t & 3];
    return v;
}

#define RD_MFMA(A, B, C) __builtin_amdgcn_mfma_f32_16x16x32_bf16((A), (B), (C), 0, 0, 0)

// z = W h + b of a 64x64 layer for one sample tile; w: the lane's weight
// fragments, b: the lane's biases (features 16 to + 4 g + r), or 0
__device__ __forceinline__ void rd_mlp_layer64(const rd_bf16x8 (&w)[4][2], const rd_f32x4 (&b)[4],
                                               const float (&h)[4][4], float (&z)[4][4])
{
    const rd_bf16x8 h0 = rd_mlp_bop(h, 0), h1 = rd_mlp_bop(h, 1);
#pragma unroll
    for (int to = 0; to < 4; ++to) {
        rd_f32x4 acc = b[to];
        acc = RD_MFMA(w[to][0], h0, acc);
        acc = RD_MFMA(w[to][1], h1, acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) z[to][r] = acc[r];
    }
}

// h = SiLU(z), s = sigmoid(z)
__device__ __forceinline__ void rd_mlp_silu_all(const float (&z)[4][4], float (&s)[4][4], float (&h)[4][4])
{
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[b][r] = rd_sigmoid(z[b][r]);
            h[b][r] = z[b][r] * s[b][r];
        }
}

// sum over the 16 lanes of a lane group (lanes with equal lane>>4), in every
// lane; the order of an xor butterfly over 1, 2, 4, 8, whose last two steps
// are mirrors here (after two steps the lanes of a quad hold the same sum)
__device__ __forceinline__ float rd_sum16(float v)
{
    auto dpp = [](float x, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v += dpp(v, std::integral_constant<int, 0xB1>());      // quad_perm [1,0,3,2]
    v += dpp(v, std::integral_constant<int, 0x4E>());      // quad_perm [2,3,0,1]
    v += dpp(v, std::integral_constant<int, 0x141>());     // row_half_mirror
    v += dpp(v, std::integral_constant<int, 0x140>());     // row_mirror
    return v;
}
