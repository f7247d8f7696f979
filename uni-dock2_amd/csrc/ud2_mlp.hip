// BF16 MFMA kernels of the learned MC proposal network (no reference
// counterpart): inference, backward pass, weight-gradient GEMM, loss, Adam.
// The tiling and the network are described in ud2_mlp.h.
#include "ud2_mlp.h"

namespace ud2 {

// Inference: y[16 gi + r] for the 16 rows of group groups[gi] (or gi).
__global__ __launch_bounds__(256) void mlp_fwd_kernel(MlpDev W, const uint16_t* __restrict__ x,
                                                      const int32_t* __restrict__ groups, int64_t n_groups,
                                                      float* __restrict__ y) {
    const int64_t gi = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (gi >= n_groups) return;
    const int64_t g = groups ? (int64_t)groups[gi] : gi;
    const int l = threadIdx.x % kWave, row = l & 15, q = l >> 4;
    const float yv = mlp_group_scores(W, x + g * kGroup * kFeat);
    if (q == 0) y[gi * kGroup + row] = yv;
}

// One group of the minibatch per block, the tiles of each layer dealt to the four waves and the hidden rows
// shared through LDS. LOSS: the group's scores (the forward pass), d loss / d y_hat of the group-centred loss with
// labels clipped at (group minimum + 6), and the backward pass; else the backward pass of the
// d loss / d y_hat in T.dy. The backward pass recomputes the hidden layers and writes the
// operands of the weight-gradient GEMMs (xn, a1, dz1, dz2 in bf16, as MFMA fragments) and the group's partial sums of
// dw3, db2, db1, db3 and the loss. A group's loss needs its own scores only, so one launch does what a forward, a
// loss and a backward kernel did. The tile loops stay loops: unrolled, a block runs once through 40 KB of cold
// code. The weights lie as fragments in the order of the lanes: from rows of 512 bytes, 16 lines a load, this
// kernel took 101 us for 1,024 groups, with the fragments 51 us (the three kernels 158 us).
template <bool LOSS>
__global__ __launch_bounds__(256) void mlp_train_kernel(MlpDev W, MlpTrain T) {
    constexpr int kTiles = 16, kMine = kTiles / kWavesPerBlock;  // 16-unit tiles of a hidden layer, and of a wave
    __shared__ bf16x8 s_k32[kTiles / 2][kWave];  // hidden rows in the scoring form
    __shared__ float s_y[kTiles][kWave];
    __shared__ bf16x4 s_a1[kTiles][kWave], s_dz2[kTiles][kWave];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int gi = blockIdx.x;
    const int64_t g = T.groups ? (int64_t)T.groups[gi] : gi;
    const int l = threadIdx.x % kWave, row = l & 15, q = l >> 4;
    const size_t col = (size_t)gi * kGroup + row;
    // where unit 4 q + i of a tile of 16 goes for this lane's row, with this group's fragments of tile 0
    const size_t at = ((size_t)gi * kWave + 16 * (row >> 2) + 4 * q) * 4 + (row & 3), tile = (size_t)T.n_groups * kWave * 4;
    const uint16_t* x = T.x + (g * kGroup + row) * kFeat;
    float* part = T.part + (size_t)gi * kPartStride;
    bf16x4 xb[5];
    load_inputs(W, x, q, xb);
    float dy;
    if (LOSS) {
        // mlp_group_scores, with its sums in the same order
        bf16x8 xk[3];
        load_inputs32(W, x, q, xk);
#pragma unroll 1
        for (int k = 0; k < kMine / 2; k++) {
            const int kb = kMine / 2 * w + k;
            const bf16x4 lo = layer1_tile32(W, xk, 2 * kb, row, q), hi = layer1_tile32(W, xk, 2 * kb + 1, row, q);
            s_k32[kb][l] = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
        __syncthreads();
        bf16x8 a[kTiles / 2];
#pragma unroll
        for (int kb = 0; kb < kTiles / 2; kb++) a[kb] = s_k32[kb][l];
#pragma unroll 1
        for (int k = 0; k < kMine; k++) {
            const int ot = kMine * w + k;
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            const uint16_t* wf = W.w2s + (ot * 8 * kWave + l) * 8;
#pragma unroll
            for (int kb = 0; kb < 8; kb++) acc = mfma32(ldw8(wf + kb * kWave * 8), a[kb], acc);
            s_y[ot][l] = layer3_part(W, acc, ot, q);
        }
        __syncthreads();
        float yp = 0.0f;
#pragma unroll
        for (int ot = 0; ot < kTiles; ot++) yp += s_y[ot][l];
        yp += __shfl_xor(yp, 16);
        yp += __shfl_xor(yp, 32);
        const float yhat = yp + W.b3[0];
        const float lab = T.label[g * kGroup + row];
        const float yc = isfinite(lab) ? lab : INFINITY;
        const float ymin = row16_min(yc);
        const float r = yhat - fminf(yc, ymin + 6.0f);
        float rbar = 0.0f;
#pragma unroll
        for (int i = 0; i < kGroup; i++) rbar += __shfl(r, i, kGroup);  // in candidate order
        rbar *= 1.0f / kGroup;
        const float c = isfinite(ymin) ? r - rbar : 0.0f;
        dy = 2.0f * c / (float(T.n_groups) * kGroup);
        float ls = 0.0f;
#pragma unroll
        for (int i = 0; i < kGroup; i++) ls += __shfl(c, i, kGroup) * __shfl(c, i, kGroup);
        if (threadIdx.x == 0) part[3 * kHidden + 1] = ls;
    } else {
        dy = T.dy[col];
    }
#pragma unroll
    for (int ks = 0; ks < 5; ks++)
        if (ks % kWavesPerBlock == w) {
#pragma unroll
            for (int i = 0; i < 4; i++) T.xn[tile * ks + at + 4 * i] = uint16_t(xb[ks][i]);
        }
#pragma unroll 1
    for (int k = 0; k < kMine; k++) {
        const int mt = kMine * w + k;
        const bf16x4 h = layer1_tile(W, xb, mt, row, q);
        s_a1[mt][l] = h;
#pragma unroll
        for (int i = 0; i < 4; i++) T.a1[tile * mt + at + 4 * i] = uint16_t(h[i]);
    }
    __syncthreads();
    bf16x4 a1[kTiles];
#pragma unroll
    for (int mt = 0; mt < kTiles; mt++) a1[mt] = s_a1[mt][l];
#pragma unroll 1
    for (int k = 0; k < kMine; k++) {
        const int ot = kMine * w + k;
        const f32x4 acc = layer2_tile(W, a1, ot, row, q);
        bf16x4 dz;
        f32x4 sw3, sb2;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int o = 16 * ot + 4 * q + i;
            const float z = acc[i] + W.b2[o];
            const float a2 = fmaxf(z, 0.0f);
            const float d = z > 0.0f ? dy * W.w3[o] : 0.0f;
            const uint16_t db = f2bf(d);
            dz[i] = short(db);
            T.dz2[tile * ot + at + 4 * i] = db;
            sw3[i] = row16_sum(dy * a2);
            sb2[i] = row16_sum(d);
        }
        s_dz2[ot][l] = dz;
        if (row == 0) {
            *reinterpret_cast<f32x4*>(part + 16 * ot + 4 * q) = sw3;
            *reinterpret_cast<f32x4*>(part + kHidden + 16 * ot + 4 * q) = sb2;
        }
    }
    __syncthreads();
    bf16x4 dz2[kTiles];
#pragma unroll
    for (int ot = 0; ot < kTiles; ot++) dz2[ot] = s_dz2[ot][l];
    // dA1^T[h][cand] = W2[h][:] . dz2^T[:][cand]; dz1 = dA1 where a1 > 0
#pragma unroll 1
    for (int k = 0; k < kMine; k++) {
        const int ht = kMine * w + k;
        const bf16x4 mine = s_a1[ht][l];
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, sb1;
        const uint16_t* wf = W.w2 + (ht * 16 * kWave + l) * 4;
#pragma unroll
        for (int kt = 0; kt < kTiles; kt++) acc = mfma16(ld4(wf + kt * kWave * 4), dz2[kt], acc);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float d = bf2f_s(mine[i]) > 0.0f ? acc[i] : 0.0f;
            T.dz1[tile * ht + at + 4 * i] = f2bf(d);
            sb1[i] = row16_sum(d);
        }
        if (row == 0) *reinterpret_cast<f32x4*>(part + 2 * kHidden + 16 * ht + 4 * q) = sb1;
    }
    const float sdy = row16_sum(dy);
    if (threadIdx.x == 0) part[3 * kHidden] = sdy;
}

// Weight-gradient GEMMs, C[M][N] = A[M][K] . B[N][K]^T with K the minibatch's rows, nb blocks of 16 (the groups), over K
// split into `splits` equal ranges: a wave forms a tile of 16 TM x 16 TN over one range and writes it to
// part[range][M][N]. A and B are stored fragment by fragment (tile, block, lane), so a wave's load is 512
// consecutive bytes; a wave loads TM + TN fragments for TM * TN MFMAs. Bound by the latency of those loads.
// 16 x 16 tiles over feature-major rows, 16 lines a load, took 90 us for dW1 and dW2 of 16,384 rows; every
// 16 x 16 tile still sums in the same order.
template <int TM, int TN>
__device__ __forceinline__ void gemm_tile(const uint16_t* A, const uint16_t* B, int N, int nb, int tile, int range,
                                          int splits, float* part) {
    const int l = threadIdx.x % kWave, row = l & 15, q = l >> 4;
    const int ntn = N / (16 * TN), m0 = tile / ntn * TM, n0 = tile % ntn * TN;
    const int kc = nb / splits;
    const uint16_t* ar = A + (((int64_t)m0 * nb + (int64_t)range * kc) * kWave + l) * 4;
    const uint16_t* br = B + (((int64_t)n0 * nb + (int64_t)range * kc) * kWave + l) * 4;
    const int64_t next = (int64_t)nb * kWave * 4;  // the next tile's fragments
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int k = 0; k < kc; k++) {
        bf16x4 va[TM], vb[TN];
#pragma unroll
        for (int i = 0; i < TM; i++) va[i] = ld4(ar + next * i + k * kWave * 4);
#pragma unroll
        for (int j = 0; j < TN; j++) vb[j] = ld4(br + next * j + k * kWave * 4);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = mfma16(va[i], vb[j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                part[(size_t)(16 * (m0 + i) + 4 * q + e) * N + 16 * (n0 + j) + row] = acc[i][j][e];
}

// Both weight gradients: of the 40 tiles of a range of rows, the first 8 are dW1's (80 x 32), the others dW2's
// (64 x 32); a block is one wave, and where the ranges divide evenly over the XCDs all waves of a
// range run on the same one, whose L2 cache then holds it (16,384 rows: 1.7 MB a range).
// Range s of a weight's partial sums is at gpart[s][kGradW].
constexpr int kTiles1 = kHidden / 32, kTiles2 = kHidden / 64 * (kHidden / 32);
__global__ __launch_bounds__(kWave) void mlp_wgrad_kernel(MlpTrain T, int splits, float* __restrict__ gpart) {
    const int b = blockIdx.x;
    const bool even = splits % kXcds == 0;
    const int j = even ? b / kXcds : b;
    const int s = even ? b % kXcds + kXcds * (j / (kTiles1 + kTiles2)) : j / (kTiles1 + kTiles2);
    const int t = j % (kTiles1 + kTiles2);
    float* part = gpart + (size_t)s * kGradW;
    if (t < kTiles1)
        gemm_tile<5, 2>(T.xn, T.dz1, kHidden, T.n_groups, t, s, splits, part);
    else
        gemm_tile<4, 2>(T.a1, T.dz2, kHidden, T.n_groups, t - kTiles1, s, splits, part + kFeat * kHidden);
}

// bf16 device copies of parameter i of value p.
__device__ __forceinline__ void pack_param(int i, float p, const MlpPack& D) {
    if (i < kOffB1) {
        const int f = i / kHidden, h = i % kHidden;
        D.w1[frag16(h, f, 5)] = D.w1s[frag32(h, f, 3)] = f2bf(p);
    } else if (i >= kOffW2 && i < kOffB2) {
        const int h = (i - kOffW2) / kHidden, o = (i - kOffW2) % kHidden;
        const uint16_t b = f2bf(p);
        D.w2[frag16(h, o, 16)] = b;
        D.w2t[frag16(o, h, 16)] = b;
        D.w2s[frag32(o, k32_slot(h), 8)] = b;
    } else if (i >= kOffW3 && i < kOffB3) {
        D.w3r[i - kOffW3] = bf2f(f2bf(p));
    }
}

// The gradient of every parameter from its partial sums, stored (grad) or applied: Adam (Kingma & Ba, ICLR'15) with
// bias corrections c1 = 1 - beta1^t, c2 = 1 - beta2^t, and the parameter's bf16 copies. The first
// blocks take a weight per thread over the GEMMs' ranges, the others 16 sums per block (dw3, db2, db1, db3)
// over the groups, in their order: the block loads kUpdateRows groups at a time into LDS, and a
// thread per sum adds them up. The last block sums the loss. (A thread per sum reading global memory group
// by group took 238 us for 1,024 groups, most of the step; all of this kernel takes 12 us.)
constexpr int kUpdateWBlocks = kGradW / 256, kUpdateSBlocks = (3 * kHidden + 1 + 15) / 16, kUpdateRows = 512;
static_assert(kGradW % 256 == 0, "whole blocks of weights");
__global__ __launch_bounds__(256) void mlp_update_kernel(const float* __restrict__ gpart, int splits,
                                                         const float* __restrict__ part, int n_groups, float* grad,
                                                         MlpAdam O, MlpPack D) {
    int i;
    float g = 0.0f;
    if (blockIdx.x < kUpdateWBlocks) {
        const int k = blockIdx.x * 256 + threadIdx.x;
        for (int s = 0; s < splits; s++) g += gpart[(size_t)s * kGradW + k];
        i = k < kFeat * kHidden ? kOffW1 + k : kOffW2 + (k - kFeat * kHidden);
    } else if (blockIdx.x < kUpdateWBlocks + kUpdateSBlocks) {
        __shared__ float sh[kUpdateRows][17];
        const int t = threadIdx.x / 16, k = threadIdx.x % 16;
        const int c = (blockIdx.x - kUpdateWBlocks) * 16 + k;
        for (int b0 = 0; b0 < n_groups; b0 += kUpdateRows) {
            const int n = min(kUpdateRows, n_groups - b0);
#pragma unroll
            for (int r = 0; r < kUpdateRows; r += 16)  // no branch: the loads are in flight together
                sh[r + t][k] = part[(size_t)(b0 + min(r + t, n - 1)) * kPartStride + c];
            __syncthreads();
            if (t == 0) {
#pragma unroll 16
                for (int r = 0; r < n; r++) g += sh[r][k];
            }
            __syncthreads();
        }
        if (t != 0 || c > 3 * kHidden) return;
        i = c < kHidden ? kOffW3 + c : c < 2 * kHidden ? kOffB2 + c - kHidden
          : c < 3 * kHidden ? kOffB1 + c - 2 * kHidden : kOffB3;
    } else {
        if (!O.loss) return;
        __shared__ float sl[256];
        for (int b = threadIdx.x; b < n_groups; b += 256) g += part[(size_t)b * kPartStride + 3 * kHidden + 1];
        sl[threadIdx.x] = g;
        __syncthreads();
        for (int h = 128; h > 0; h >>= 1) {
            if (int(threadIdx.x) < h) sl[threadIdx.x] += sl[threadIdx.x + h];
            __syncthreads();
        }
        if (threadIdx.x == 0) O.loss[0] = sl[0] * O.loss_scale;
        return;
    }
    if (grad) {
        grad[i] = g;
        return;
    }
    const float m = O.beta1 * O.m[i] + (1.0f - O.beta1) * g;
    const float v = O.beta2 * O.v[i] + (1.0f - O.beta2) * g * g;
    O.m[i] = m;
    O.v[i] = v;
    const float p = O.p[i] - O.lr * (m / O.c1) / (sqrtf(v / O.c2) + O.eps);
    O.p[i] = p;
    pack_param(i, p, D);
}

// bf16 device copies of the weights from the canonical FP32 parameters.
__global__ void mlp_pack_kernel(const float* __restrict__ P, MlpPack D) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kMlpNParam) pack_param(i, P[i], D);
}

// ------------------------------------------------------------- launchers
hipError_t launch_mlp_forward(const MlpDev& W, const uint16_t* x, const int32_t* groups, int64_t n_groups, float* y,
                              hipStream_t s) {
    if (n_groups <= 0) return hipSuccess;
    hipLaunchKernelGGL(mlp_fwd_kernel, dim3((unsigned)((n_groups + 3) / 4)), dim3(256), 0, s, W, x, groups, n_groups,
                       y);
    return hipGetLastError();
}

hipError_t launch_mlp_train(const MlpDev& W, const MlpTrain& T, int splits, float* gpart, hipStream_t s) {
    if (T.n_groups <= 0 || splits <= 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)T.n_groups), block(256);
    if (T.dy) hipLaunchKernelGGL(mlp_train_kernel<false>, grid, block, 0, s, W, T);
    else hipLaunchKernelGGL(mlp_train_kernel<true>, grid, block, 0, s, W, T);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(mlp_wgrad_kernel, dim3((unsigned)((kTiles1 + kTiles2) * splits)), dim3(kWave), 0, s, T, splits,
                       gpart);
    return hipGetLastError();
}

hipError_t launch_mlp_update(const float* gpart, int splits, const float* part, int n_groups, float* grad,
                             const MlpAdam& O, const MlpPack& D, hipStream_t s) {
    hipLaunchKernelGGL(mlp_update_kernel, dim3(kUpdateWBlocks + kUpdateSBlocks + 1), dim3(256), 0, s, gpart, splits,
                       part, n_groups, grad, O, D);
    return hipGetLastError();
}

hipError_t launch_mlp_pack(const float* params, const MlpPack& D, hipStream_t s) {
    hipLaunchKernelGGL(mlp_pack_kernel, dim3((kMlpNParam + 255) / 256), dim3(256), 0, s, params, D);
    return hipGetLastError();
}

}  // namespace ud2
