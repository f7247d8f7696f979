// Device pieces of the learned proposal network shared by the MFMA kernels
// (ud2_mlp.hip) and the fused learned MC kernel (ud2_learned.hip).
//
// Network: y = w3 . relu(W2^T a1 + b2) + b3, a1 = bf16(relu(W1^T xn + b1)),
// xn = bf16((x - mu) * inv_sigma); 80 inputs, two hidden layers of 256.
//
// Tiling: one wave scores a group of 16 candidates. Every layer is computed
// transposed, out^T[hidden][cand] = W^T[hidden][k] . in^T[k][cand]. Scoring
// uses CDNA4's v_mfma_f32_16x16x32_bf16: the weights are the A operand (lane l
// holds row l % 16 and 8 k values of block 32 kb + 8 (l / 16) .. +7, a 16-byte
// load), the activations the B operand (lane l holds candidate l % 16, the same
// k). The accumulator of a 16 x 16 output tile puts rows 4 (l / 16) .. +3 of
// candidate l % 16 on lane l; the two tiles 2 kb and 2 kb + 1 together give lane
// l the 8 hidden units 32 kb + 4 (l / 16) + {0..3, 16..19}, which is the B
// operand of the next layer's K block kb when that layer's weights take the
// same order of k (w2s, packed so), so hidden activations never leave the
// registers. Layer 1 has K = 80: three 32-wide blocks, the last one zero past
// k = 80 (lanes 32-63 hold zeros): a chain of accumulating MFMAs keeps one
// opcode (an accumulator written by one MFMA opcode and read by another as
// SrcC needs wait states that a chain of one opcode does not).
// The training kernels (backward pass) use the 16x16x16 form throughout, with
// the weights in natural order. Weights stream from L2 (166 KB in bf16).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ud2_internal.h"

namespace ud2 {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ float bf2f_s(short b) { return bf2f(uint16_t(b)); }

// Round to nearest even; NaN stays NaN (quietened), overflow rounds to inf: v_cvt_pk_bf16_f32, whose result is that
// of the integer rounding for every float. A conversion in integer operations with a branch for infinities and NaN cut
// the training kernel into a hundred basic blocks, each waiting for its own loads.
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }

// Loads of what no kernel that uses them writes (weights, and in the weight-gradient GEMMs the operands), through the
// constant address space, so that they may be issued ahead of barriers and stores.
template <class T>
__device__ __forceinline__ T cload(const void* p) {
    return *(const __attribute__((address_space(4))) T*)(p);
}
__device__ __forceinline__ bf16x4 ld4(const uint16_t* p) { return cload<bf16x4>(p); }

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ bf16x8 ldw8(const uint16_t* p) { return cload<bf16x8>(p); }

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
}

// Place of hidden unit h in the K = 32 order of layer 2 (w2s and the staged hidden rows): h = 32 kb +
// 16 t + 4 q + i goes to 32 kb + 8 q + 4 t + i.
__host__ __device__ constexpr int k32_slot(int h) {
    return (h & ~31) + 8 * ((h >> 2) & 3) + 4 * ((h >> 4) & 1) + (h & 3);
}

// Sum and minimum over the 16 lanes of a lane row (lanes 16 q .. 16 q + 15), by DPP row exchanges.
template <int CTRL>
__device__ __forceinline__ float row16_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row16_sum(float v) {
    v += row16_dpp<0xB1>(v);
    v += row16_dpp<0x4E>(v);
    v += row16_dpp<0x141>(v);
    v += row16_dpp<0x140>(v);
    return v;
}
__device__ __forceinline__ float row16_min(float v) {
    v = fminf(v, row16_dpp<0xB1>(v));
    v = fminf(v, row16_dpp<0x4E>(v));
    v = fminf(v, row16_dpp<0x141>(v));
    v = fminf(v, row16_dpp<0x140>(v));
    return v;
}

// Normalised inputs of candidate `row` as B operands of the 5 K blocks of layer 1.
__device__ __forceinline__ void load_inputs(const MlpDev& W, const uint16_t* xr, int q, bf16x4 xb[5]) {
#pragma unroll
    for (int ks = 0; ks < 5; ks++) {
        const bf16x4 raw = ld4(xr + 16 * ks + 4 * q);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int f = 16 * ks + 4 * q + i;
            xb[ks][i] = short(f2bf((bf2f_s(raw[i]) - W.mu[f]) * W.inv_sigma[f]));
        }
    }
}

// Layer-1 tile mt: hidden units 16 mt + 4 q + i of candidate `row`, after bias and ReLU, in bf16.
__device__ __forceinline__ bf16x4 layer1_tile(const MlpDev& W, const bf16x4 xb[5], int mt, int row, int q) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* wf = W.w1 + (mt * 5 * kWave + 16 * q + row) * 4;
#pragma unroll
    for (int ks = 0; ks < 5; ks++) acc = mfma16(ld4(wf + ks * kWave * 4), xb[ks], acc);
    bf16x4 h;
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = short(f2bf(fmaxf(acc[i] + W.b1[16 * mt + 4 * q + i], 0.0f)));
    return h;
}

// z2 tile ot (outputs 16 ot + 4 q + i of candidate `row`), before bias.
__device__ __forceinline__ f32x4 layer2_tile(const MlpDev& W, const bf16x4 a1[16], int ot, int row, int q) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* wf = W.w2t + (ot * 16 * kWave + 16 * q + row) * 4;
#pragma unroll
    for (int kt = 0; kt < 16; kt++) acc = mfma16(ld4(wf + kt * kWave * 4), a1[kt], acc);
    return acc;
}

// Normalised inputs of candidate `row` as B operands of layer 1 in the scoring form: K block kb holds
// features 32 kb + 8 q .. +7, zero past feature 79 (block 2, q >= 2). Every load stays in the row.
__device__ __forceinline__ void load_inputs32(const MlpDev& W, const uint16_t* xr, int q, bf16x8 xb[3]) {
#pragma unroll
    for (int kb = 0; kb < 3; kb++) {
        const int f0 = kb < 2 ? 32 * kb + 8 * q : 64 + 8 * (q & 1);
        const bf16x8 raw = ld8(xr + f0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const short v = short(f2bf((bf2f_s(raw[i]) - W.mu[f0 + i]) * W.inv_sigma[f0 + i]));
            xb[kb][i] = (kb < 2 || q < 2) ? v : short(0);
        }
    }
}

// Layer-1 tile mt in the scoring form: hidden units 16 mt + 4 q + i of candidate `row`, after bias and
// ReLU, in bf16.
__device__ __forceinline__ bf16x4 layer1_tile32(const MlpDev& W, const bf16x8 xb[3], int mt, int row, int q) {
    const uint16_t* wf = W.w1s + (mt * 3 * kWave + 16 * q + row) * 8;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 3; kb++) acc = mfma32(ldw8(wf + kb * kWave * 8), xb[kb], acc);
    bf16x4 h;
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = short(f2bf(fmaxf(acc[i] + W.b1[16 * mt + 4 * q + i], 0.0f)));
    return h;
}

// The w3-weighted, ReLU'd layer-2 outputs of tile ot summed on this lane.
__device__ __forceinline__ float layer3_part(const MlpDev& W, f32x4 acc, int ot, int q) {
    float yp = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int o = 16 * ot + 4 * q + i;
        yp += W.w3[o] * fmaxf(acc[i] + W.b2[o], 0.0f);
    }
    return yp;
}

// Scores of the 16 candidates whose bf16 inputs are rows [16][80] at x (global
// or LDS memory, 16-byte aligned): lanes 16 q + r all return the score of candidate r.
__device__ __forceinline__ float mlp_group_scores(const MlpDev& W, const uint16_t* x) {
    const int l = threadIdx.x % kWave, row = l & 15, q = l >> 4;
    bf16x8 xb[3];
    load_inputs32(W, x + row * kFeat, q, xb);
    bf16x8 a1[8];  // K block kb of layer 2: tiles 2 kb and 2 kb + 1 of layer 1
#pragma unroll
    for (int kb = 0; kb < 8; kb++) {
        const bf16x4 lo = layer1_tile32(W, xb, 2 * kb, row, q), hi = layer1_tile32(W, xb, 2 * kb + 1, row, q);
        a1[kb] = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    float yp = 0.0f;
#pragma unroll 2
    for (int ot = 0; ot < 16; ot++) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        const uint16_t* wf = W.w2s + (ot * 8 * kWave + l) * 8;
#pragma unroll
        for (int kb = 0; kb < 8; kb++) acc = mfma32(ldw8(wf + kb * kWave * 8), a1[kb], acc);
        yp += layer3_part(W, acc, ot, q);
    }
    yp += __shfl_xor(yp, 16);
    yp += __shfl_xor(yp, 32);
    return yp + W.b3[0];
}

// The same scores with the hidden activations staged through LDS instead of
// registers (for kernels whose other phases need the registers): x holds the
// 16 bf16 input rows, the hidden layer is [rows][kA1Stride] bf16 with rows below
// `split` at a1 and the others at a1b (all LDS, 16-byte aligned, private to the
// wave). The rows at a1 may overlay x: x is read into registers first.
// Only candidates below `rows` (8 or 16) are scored: an output column of the
// MFMA depends on its own input column alone, so the lanes of the other
// candidates stage nothing and read candidate 0's hidden row, and their scores
// (to be ignored) are candidate 0's.
__device__ __forceinline__ float mlp_group_scores_lds(const MlpDev& W, const uint16_t* x, uint16_t* a1,
                                                      uint16_t* a1b, int split, int rows) {
    const int l = threadIdx.x % kWave, row = l & 15, q = l >> 4;
    bf16x8 xb[3];
    load_inputs32(W, x + row * kFeat, q, xb);
    // the hidden row of candidate `row` in the K = 32 order of layer 2 (k32_slot): tile mt's four units
    // of this lane at 32 (mt / 2) + 8 q + 4 (mt % 2)
    const bool live = row < rows;
    const int r = live ? row : 0;
    uint16_t* a1row = r < split ? a1 + r * kA1Stride : a1b + (r - split) * kA1Stride;
    for (int mt = 0; mt < 16; mt++) {
        const bf16x4 h = layer1_tile32(W, xb, mt, row, q);
        if (live) *reinterpret_cast<bf16x4*>(a1row + 32 * (mt >> 1) + 8 * q + 4 * (mt & 1)) = h;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float yp = 0.0f;
    const uint16_t* ar = a1row + 8 * q;
    for (int ot = 0; ot < 16; ot++) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        const uint16_t* wf = W.w2s + (ot * 8 * kWave + l) * 8;
#pragma unroll 4
        for (int kb = 0; kb < 8; kb++) acc = mfma32(ldw8(wf + kb * kWave * 8), ld8(ar + 32 * kb), acc);
        yp += layer3_part(W, acc, ot, q);
    }
    yp += __shfl_xor(yp, 16);
    yp += __shfl_xor(yp, 32);
    return yp + W.b3[0];
}

}  // namespace ud2
