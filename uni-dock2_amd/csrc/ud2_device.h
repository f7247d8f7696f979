// Device-side building blocks of the docking hot path for gfx950 (CDNA4, wave64),
// shared by the kernel translation units (ud2_kernels.hip, ud2_learned.hip).
//
// Execution model: one docking chain (or one scored pose) per wavefront. Atom
// a lives on lane a % 64, register slot a / 64 (APL = atoms per lane, a
// template parameter), so coordinates and per-atom gradients stay in VGPRs;
// the dihedral vector and every BFGS vector (gradient, direction, y, -Hy) are
// one VGPR each with component k on lane k; the inverse Hessian is a per-wave
// LDS tile whose row i only lane i reads and writes. Energies, torques and
// dot products are wave reductions. Intra-molecular pairs of ligands of up to 64 atoms are scored in
// packed steps, a pair per lane, whose shares the atoms collect through a per-wave LDS tile; past 64
// atoms along folded diagonals (atom a with atom (a + d) mod natom), each atom keeping its own pair
// forces in registers and passing the partner's share on through the tile. No atomics anywhere. MFMA is
// not used: the physics is gather and VALU work on chains of dependent operations, bound by VALU issue,
// the LDS pipe and latency together.
//
// The algorithm follows the reference's device code (E/ =
// unidock/unidock_engine/): cal_e_f_tile / cal_grad_tile (E/src/cuda/bfgs.cuh:
// 69-394), the torsion and rigid pose updates (bfgs.cuh:443-618), line search
// and BFGS (bfgs.cuh:623-829), mutation / randomisation / MC (E/src/cuda/mc.cu:
// 18-398), RMSD clustering (E/src/cuda/cluster.cu:16-135) and final scoring
// (E/src/score/score.cpp:12-108).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ud2_internal.h"

namespace ud2 {

// ------------------------------------------------------------- constants
// vdW radii (E/src/constants/constants.h:21-43) and per-type flags:
// bit0 hydrophobic, bit1 acceptor, bit2 donor (E/src/score/vina.h:49-65).
static __constant__ float c_vdw[kNumTypes] = {1.1f, 1.92f, 1.9f, 1.9f, 1.8f, 1.8f, 1.8f, 1.8f, 1.7f, 1.7f, 1.7f,
                                       1.7f, 1.5f, 2.2f, 2.1f, 2.0f, 1.8f, 2.0f, 2.2f, 2.3f, 1.2f};
static __constant__ int c_tflags[kNumTypes] = {0, 0, 1, 0, 0, 4, 2, 6, 0, 4, 2, 6, 1, 0, 0, 0, 1, 1, 1, 0, 4};

constexpr float kPi = 3.1415927f;               // E/src/myutils/common.h:45
constexpr float kEps = 1.1920928955078125e-7f;  // FLT_EPSILON (common.h:13)
constexpr float kR2Cut = 64.0f;                 // E/src/score/vina.h:130
constexpr float kR2Reach = 64.2f;               // squared reach of a cull: the cutoff and some roundings
constexpr float kVCap = 10.0f, kVCapAuth = 1000.0f, kSlope = 1e6f;  // constants.h:16-19
constexpr int kTypeH = 0;

// ------------------------------------------------------------ wave utils
__device__ __forceinline__ int lane() { return __lane_id(); }

__device__ __forceinline__ float rdl(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ int rdl_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// Sum over each 16-lane row with DPP row exchanges (quad_perm [1,0,3,2], quad_perm [2,3,0,1],
// row_half_mirror, row_mirror): every lane of a row ends with the row sum, in the same bits, whichever
// row it is.
__device__ __forceinline__ float row_sum(float v) {
    v += dpp_f<0xB1>(v);
    v += dpp_f<0x4E>(v);
    v += dpp_f<0x141>(v);
    v += dpp_f<0x140>(v);
    return v;
}

// Sum over the 64 lanes: the four row sums read from lanes 0, 16, 32, 48 and added in a fixed order.
// The result is uniform (scalar register). Called in wave-uniform control flow only (all lanes active).
__device__ __forceinline__ float wave_sum(float v) {
    v = row_sum(v);
    return ((rdl(v, 0) + rdl(v, 16)) + rdl(v, 32)) + rdl(v, 48);
}

// Squared distance with explicit fused multiply-adds, so that every kernel that inlines it rounds it
// the same way: the 8 A cutoff test on it must not depend on which kernel evaluates a pose (a pair
// entering or leaving the cutoff moves the energy by up to about 0.004).
__device__ __forceinline__ float sq_dist(float rx, float ry, float rz) {
    return __builtin_fmaf(rz, rz, __builtin_fmaf(ry, ry, rx * rx));
}

// Sums of products with the fused multiply-adds written out: the compiler's choice of which product
// of a * b + c * d to fuse depends on the surrounding code (how often a product is reused, whether an
// operand sits in a scalar register), so the same expression could round differently in two kernels
// that inline it. Every expression of two or more products on the pose path goes through these.
__device__ __forceinline__ float fmaf_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// a b + c d, c d rounded first
__device__ __forceinline__ float madd2(float a, float b, float c, float d) { return __builtin_fmaf(a, b, c * d); }
// a b - c d, c d rounded first
__device__ __forceinline__ float msub2(float a, float b, float c, float d) { return __builtin_fmaf(a, b, -(c * d)); }
// a b + c d + e f, evaluated as ((a b) + c d) + e f
__device__ __forceinline__ float madd3(float a, float b, float c, float d, float e, float f) {
    return __builtin_fmaf(e, f, __builtin_fmaf(c, d, a * b));
}

// Hardware reciprocal / square root / reciprocal square root (about 1 ulp).
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }

// A value all lanes agree on, moved to a scalar register.
__device__ __forceinline__ float uni(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// ------------------------------------------------------------ tile utils
// A tile is the group of TW lanes that runs one chain: the whole wave (TW = 64), or one half of it
// (TW = 32, two chains of the same ligand per wave, lanes 0-31 and 32-63). Each function below acts
// within the calling lane's tile; with TW = 64 they are the wave operations above. Control flow that
// depends on a chain's state (line-search trials, acceptance, the kind of mutation) is uniform per
// tile, not per wave, so with TW = 32 the two halves may run different branches under the execution
// mask; the tile operations are called where every lane of the running tiles is active.

// Lane index within the tile, and the tile's first lane in the wave.
template <int TW>
__device__ __forceinline__ int tlane() {
    int l = __lane_id();
    asm volatile("" : "+v"(l));
    return TW == kWave ? l : (l & (TW - 1));
}
template <int TW>
__device__ __forceinline__ int tbase() { return TW == kWave ? 0 : (__lane_id() & ~(TW - 1)); }

// A value that the compiler knows nothing of: it is rounded here and nothing is fused across.
__device__ __forceinline__ float opaque(float v) {
    asm("" : "+v"(v));
    return v;
}

// A value every lane of the tile agrees on: moved to a scalar register for a whole-wave tile, kept in
// its vector register (one value per tile) otherwise. Either way the value is rounded and opaque at
// this point: the compiler cannot fuse the operation that produced it into the ones that use it (a
// multiply into a later add, as one fused multiply-add), so both tile widths round alike.
template <int TW>
__device__ __forceinline__ float tuni(float v) {
    if constexpr (TW == kWave) {
        return uni(v);
    } else {
        return opaque(v);
    }
}

// Sum over the tile's lanes. For TW = 32 the tile's two row sums, the same bits a whole-wave sum
// adds first when lanes 32-63 hold zeros.
template <int TW>
__device__ __forceinline__ float tsum(float v) {
    static_assert(TW == kWave || TW == 32, "tiles are 64 or 32 lanes");
    if constexpr (TW == kWave) {
        return wave_sum(v);
    } else {
        v = row_sum(v);
        const float lo = rdl(v, 0) + rdl(v, 16), hi = rdl(v, 32) + rdl(v, 48);
        return (__lane_id() & 32) ? hi : lo;
    }
}

// Sums of four values over the tile's lanes: lane l (ln: tlane) gets that of v[l % 4], in the bits of tsum. The first two
// exchanges of row_sum halve the values in flight instead of repeating themselves for each (a lane adds up the
// values of its own place in the quad), the row sums are exchanged by two lane swaps instead of four lane reads per
// value: 21 VALU instructions for what takes four tsum 48.
template <int TW>
__device__ __forceinline__ float tsum4(int ln, float v0, float v1, float v2, float v3) {
    const bool odd = ln & 1, up = ln & 2;
    const float a = (odd ? v1 : v0) + dpp_f<0xB1>(odd ? v0 : v1);
    const float b = (odd ? v3 : v2) + dpp_f<0xB1>(odd ? v2 : v3);
    float c = (up ? b : a) + dpp_f<0x4E>(up ? a : b);
    c += dpp_f<0x1B>(dpp_f<0x141>(c));  // lane ^ 4: the half row mirrored, then each quad
    c += dpp_f<0x128>(c);               // lane ^ 8: the row rotated by 8
    const auto swap16 = [](float v, float& r0, float& r1) {  // the rows of each half: its first everywhere, its second
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        r0 = __uint_as_float(r[0]);
        r1 = __uint_as_float(r[1]);
    };
    if constexpr (TW == kWave) {
        const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false, false);
        float r0, r1, r2, r3;
        swap16(__uint_as_float(h[0]), r0, r1);
        swap16(__uint_as_float(h[1]), r2, r3);
        return ((r0 + r1) + r2) + r3;
    } else {
        float r0, r1;
        swap16(c, r0, r1);
        return r0 + r1;
    }
}

// Lane l of the tile, l the same for every lane of the wave (a constant or a wave-uniform index).
template <int TW>
__device__ __forceinline__ float trdl(float v, int l) {
    if constexpr (TW == kWave) return rdl(v, l);
    else return (__lane_id() & 32) ? rdl(v, 32 + l) : rdl(v, l);
}

// Lane l of the tile, l per lane (mod TW).
template <int TW>
__device__ __forceinline__ float tshfl(float v, int l) { return __shfl(v, l & (TW - 1), TW); }
template <int TW>
__device__ __forceinline__ int tshfl_i(int v, int l) { return __shfl(v, l & (TW - 1), TW); }

// Lane l of the tile, l the same for every lane of the tile (but, with TW = 32, not necessarily for
// both tiles of the wave: a chain's random draw, say).
template <int TW>
__device__ __forceinline__ float tread(float v, int l) {
    if constexpr (TW == kWave) return rdl(v, l);
    else return tshfl<TW>(v, l);
}

// The tile's lanes where pred holds, bit l = tile lane l.
template <int TW>
__device__ __forceinline__ unsigned long long tballot(bool pred) {
    const unsigned long long b = __ballot(pred);
    if constexpr (TW == kWave) return b;
    else return (b >> tbase<TW>()) & 0xffffffffull;
}

// A mask over tile lanes (bit l = tile lane l) as a mask over the wave's lanes, every tile the same.
template <int TW>
__device__ __forceinline__ unsigned long long tmask(unsigned long long m) {
    if constexpr (TW == kWave) return m;
    else return (m & 0xffffffffull) | (m << 32);
}

// A kernel's arguments, read where they are used. Taken by value, the compiler loads them all at the kernel's
// entry, and with the addresses and constants that it also forms there, they overflow the 102 SGPRs
// into lanes of vector registers and those into scratch memory (the six-wave learned search kernel: 246 SGPRs and
// 90 VGPRs spilled, 2 TB/s of HBM traffic mostly for them). reread() makes the compiler forget a value's
// origin, so that nothing read through it is hoisted out of the function (tlane does the same for LDS
// addresses): 20 and 36 spilled, the 1,024-ligand learned search 371 -> 331 ms, the MC kernel's SGPR spills
// 157 -> 0 and its registers without spills 123 -> 95.
template <class T>
using Karg = const __attribute__((address_space(4))) T;
using KHead = Karg<ArgHead>;
using KLig = Karg<DevLig>;
using LigArg = Karg<LigSetDev>;
using SceneArg = Karg<SceneDev>;

template <class T>
__device__ __forceinline__ T reread(T v) {
    asm volatile("" : "+s"(v));
    return v;
}
template <class T>
__device__ __forceinline__ Karg<T>* kernel_args() {
    return (Karg<T>*)__builtin_amdgcn_kernarg_segment_ptr();
}

// Dynamic LDS of a launch; every wave owns a slice of it.
extern __shared__ float s_lds[];

// Orders this wave's LDS traffic (one wave owns its LDS slice; no block barrier).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// --------------------------------------------------------------- scoring
// Vina::eval_ef (E/src/score/vina.h:216-245) for a heavy-atom pair at surface distance d.
// Written for CDNA4's issue rates: an FP32 add, multiply or FMA (its clamp to [0, 1] free) takes 2 cycles of a
// SIMD, any compare, select, minimum or integer operation 4, a transcendental 8. So the ramps take their flags
// from kh and kb instead of selects, the repulsion's min(d, 0) is -8 clamp(-d / 8) (d > -8; exact, as the
// scaling by a power of two is), and a ramp r in (0, 1), where its derivative is not zero, is told by
// r - r r > 0, which holds for exactly the d of the two compares with its ends.
__device__ __forceinline__ float eval_ramps(float d, float kh, float kb, float* dedd) {
    // gauss1 (offset 0, width 0.5): exp(-4 d^2) = 2^(-4 log2(e) d^2), derivative -8 d exp(-4 d^2);
    // gauss2 (offset 3, width 2): exp(-(u / 2)^2) = 2^(-log2(e) / 4 u^2), u = d - 3, derivative -(u / 2) exp(..)
    const float e1 = __builtin_amdgcn_exp2f(-5.7707801635558535f * (d * d));
    const float u = d - 3.0f;
    const float e2 = __builtin_amdgcn_exp2f(-0.36067376022224085f * (u * u));
    float e = msub2(-0.035579f, e1, 0.005156f, e2);
    float f = madd2((0.035579f * 8.0f) * d, e1, (0.005156f * 0.5f) * u, e2);
    // repulsion, d < 0
    const float m = fminf(fmaxf(d * -0.125f, 0.0f), 1.0f);
    e = fmaf_((0.840245f * 64.0f) * m, m, e);
    f = fmaf_(0.840245f * -16.0f, m, f);
    // hydrophobic, slope_interp(0.5, 1.5)
    const float h = fminf(fmaxf(kh - d, 0.0f), 1.0f);
    e = fmaf_(-0.035069f, h, e);
    f += fmaf_(-h, h, h) > 0.0f ? 0.035069f : 0.0f;
    // hydrogen bond, slope_interp(-0.7, 0)
    const float b = fminf(fmaxf(d * kb, 0.0f), 1.0f);
    e = fmaf_(-0.587439f, b, e);
    f += fmaf_(-b, b, b) > 0.0f ? 0.587439f * (1.0f / 0.7f) : 0.0f;
    *dedd = f;
    return e;
}

// The same with the pair flags: bit0 both hydrophobic, bit1 hydrogen-bond capable.
__device__ __forceinline__ float eval_ef(float d, int flags, float* dedd) {
    return eval_ramps(d, ramp_hyd(flags), ramp_hb(flags), dedd);
}

__device__ __forceinline__ int pair_flags(int ti, int tj) {
    int a = c_tflags[ti], b = c_tflags[tj];
    int hyd = (a & b & 1);
    int hb = (((a >> 1) & (b >> 2)) | ((a >> 2) & (b >> 1))) & 1;
    return hyd | (hb << 1);
}

// Pair flags of an atom with type flags a against each possible partner flag set b = 0..7, two bits
// per b at bit 2 b: the intra-pair loops look up a pair's flags with one shift of this table.
__device__ __forceinline__ uint32_t pair_lut(int a) {
    uint32_t t = 0;
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const int hyd = a & b & 1;
        const int hb = (((a >> 1) & (b >> 2)) | ((a >> 2) & (b >> 1))) & 1;
        t |= uint32_t(hyd | (hb << 1)) << (2 * b);
    }
    return t;
}

// The energy of eval_ef in two parts with the same roundings: what depends on the surface distance d alone
// (the return value, and the unweighted hydrophobic and hydrogen-bond terms h and b), and the flag terms.
__device__ __forceinline__ float eval_radial(float d, float& h, float& b) {
    const float e1 = __builtin_amdgcn_exp2f(-5.7707801635558535f * (d * d));
    const float u = d - 3.0f;
    const float e2 = __builtin_amdgcn_exp2f(-0.36067376022224085f * (u * u));
    const float dn = fminf(d, 0.0f);
    h = fminf(fmaxf(1.5f - d, 0.0f), 1.0f);
    b = fminf(fmaxf(-d * (1.0f / 0.7f), 0.0f), 1.0f);
    return fmaf_(0.840245f * dn, dn, msub2(-0.035579f, e1, 0.005156f, e2));
}
__device__ __forceinline__ float add_flag_terms(float e0, float h, float b, int flags) {
    const float e = fmaf_((flags & 1) ? -0.035069f : 0.0f, h, e0);
    return fmaf_((flags & 2) ? -0.587439f : 0.0f, b, e);
}

// A receptor atom's vdW radius and type flags in one word (ud2_internal.h, atom_word).
__device__ __forceinline__ float word_radius(uint32_t w) { return __uint_as_float((w & 0xFFFFFFu) + 0x3F800000u); }
__device__ __forceinline__ uint32_t word_flags2(uint32_t w) { return w >> 24; }

// The receptor atoms that can be within the cutoff of a point, in receptor order: a reach list, or for a point
// that no cell holds the whole receptor, or nothing.
struct Reach {
    int begin, end;
    bool whole;
};

__device__ __forceinline__ Reach reach_of(SceneArg& S, float px, float py, float pz) {
    const float gx = (px - S.rorigin[0]) * S.rinv, gy = (py - S.rorigin[1]) * S.rinv, gz = (pz - S.rorigin[2]) * S.rinv;
    Reach r{0, 0, false};
    if (gx >= 0.0f && gx < float(S.rn[0]) && gy >= 0.0f && gy < float(S.rn[1]) && gz >= 0.0f && gz < float(S.rn[2])) {
        const int c = (int(gz) * S.rn[1] + int(gy)) * S.rn[0] + int(gx);
        const int2 at = S.reach_off[c];
        r.begin = at.x;
        r.end = at.y;
    } else {
        r.whole = px >= S.rec_lo[0] && px <= S.rec_hi[0] && py >= S.rec_lo[1] && py <= S.rec_hi[1] &&
                  pz >= S.rec_lo[2] && pz <= S.rec_hi[2];
    }
    return r;
}

// A load of read-only data at an address every lane agrees on, through the constant address space:
// a scalar load into SGPRs (the data is written before the kernel starts and never during it).
template <class T>
__device__ __forceinline__ T uload(const T* p) {
    return *(const __attribute__((address_space(4))) T*)(p);
}

// f(x, y, z, atom_word) for each of them, in receptor order. A list is read four entries ahead of their use
// (each lane its own list, so a load touches a line per lane, which bounds it together with the pair terms'
// VALU work); the whole receptor by scalar loads one entry ahead, by all lanes once one of them needs it: its loop costs the wave the same
// for one lane as for 64. The atoms out of reach added nothing to the sum, so it has the same bits. Against the loop over
// 2,000 atoms for every ligand atom: 20,011 direct evaluations of a 57-atom ligand 1,266 -> 238 us, the re-score and
// decomposition of 10,210 poses 982 -> 152 us, a direct-mode search of 8 ligands 745 -> 43 ms; those evaluations 30 A
// off the box, over the whole receptor, 843 us.
template <class F>
__device__ __forceinline__ void for_reach(SceneArg& S, const Reach& r, F f) {
    if (__ballot(r.whole) != 0ull) {
        typedef float f32x4_t __attribute__((ext_vector_type(4)));
        const f32x4_t* rec = reinterpret_cast<const f32x4_t*>(S.rec);
        const int nrec = S.nrec;
        f32x4_t q = uload(rec);  // there is an entry past the last
#pragma unroll 1
        for (int j = 0; j < nrec; j++) {
            const f32x4_t next = uload(rec + j + 1);
            f(q.x, q.y, q.z, __float_as_uint(q.w));
            q = next;
        }
        return;
    }
    for (int j = r.begin; j < r.end; j += kReachPad) {
        float4 q[kReachPad];
#pragma unroll
        for (int i = 0; i < kReachPad; i++) q[i] = S.reach[j + i];
#pragma unroll
        for (int i = 0; i < kReachPad; i++) f(q[i].x, q[i].y, q[i].z, __float_as_uint(q[i].w));
    }
}

// normalize_angle (E/src/myutils/mymath.h:38-47).
__device__ __forceinline__ float normalize_angle(float x) {
    x = x - 2.0f * kPi * truncf(x * (1.0f / (2.0f * kPi)));  // fmod(x, 2 pi)
    if (x < -kPi) x += 2.0f * kPi;
    if (x > kPi) x -= 2.0f * kPi;
    return x;
}

struct Mat3 {
    float m[9];
};

// Rotation matrix of a unit quaternion (w, x, y, z) = (q.x, q.y, q.z, q.w).
__device__ __forceinline__ Mat3 quat_to_mat(float4 q) {
    const float w = q.x, x = q.y, y = q.z, z = q.w;
    Mat3 R;
    const float ww = w * w, xx = x * x, yy = y * y, zz = z * z;
    R.m[0] = ((ww + xx) - yy) - zz;          R.m[1] = 2.0f * msub2(x, y, w, z);     R.m[2] = 2.0f * madd2(x, z, w, y);
    R.m[3] = 2.0f * madd2(x, y, w, z);       R.m[4] = ((ww - xx) + yy) - zz;       R.m[5] = 2.0f * msub2(y, z, w, x);
    R.m[6] = 2.0f * msub2(x, z, w, y);       R.m[7] = 2.0f * madd2(y, z, w, x);     R.m[8] = ((ww - xx) - yy) + zz;
    return R;
}

// rotvec_to_quaternion (E/src/geometry/quaternion.h:90-107); returns (w, x, y, z) in (.x, .y, .z, .w).
__device__ __forceinline__ float4 rotvec_to_quat(float v0, float v1, float v2) {
    const float th = fsqrt(sq_dist(v0, v1, v2));
    float s, c;
    __sincosf(th * 0.5f, &s, &c);  // th is a step-sized angle: the hardware sin/cos is accurate here
    // renormalised: c^2 + s^2 = 1 to an ulp, so R(q) does not scale the ligand (|q|^2 would, per update)
    const float rn = frsq(madd2(c, c, s, s));
    s *= rn;
    c *= rn;
    const float k = th > kEps ? s * frcp(th) : 0.0f;
    return th > kEps ? make_float4(c, v0 * k, v1 * k, v2 * k) : make_float4(1.0f, 0.0f, 0.0f, 0.0f);
}

// acos on [-1, 1] by Abramowitz & Stegun 4.4.46: acos(x) = sqrt(1 - x) P7(x) for
// x in [0, 1] (|error| <= 2e-8), acos(-x) = pi - acos(x).
__device__ __forceinline__ float acos_as(float x) {
    const float ax = fabsf(x);
    float p = -0.0012624911f;
    p = p * ax + 0.0066700901f;
    p = p * ax - 0.0170881256f;
    p = p * ax + 0.0308918810f;
    p = p * ax - 0.0501743046f;
    p = p * ax + 0.0889789874f;
    p = p * ax - 0.2145988016f;
    p = p * ax + 1.5707963050f;
    const float r = fsqrt(1.0f - ax) * p;
    return x < 0.0f ? 3.14159265358979f - r : r;
}

// quaternion_to_rotvec (quaternion.h:115-130) of a unit quaternion: theta =
// 2 acos(w), s = sin(theta / 2) = sqrt(1 - w^2).
__device__ __forceinline__ float3 quat_to_rotvec(float4 q) {
    const float w = fminf(fmaxf(q.x, -1.0f), 1.0f);
    const float th = 2.0f * acos_as(w);
    const float s = fsqrt(fmaxf(fmaf_(-w, w, 1.0f), 0.0f));
    const float k = s > kEps ? th * frcp(s) : 0.0f;
    return make_float3(q.y * k, q.z * k, q.w * k);
}

// Orientation gradient of cal_grad_tile (E/src/cuda/bfgs.cuh:122-190): g_k =
// <dR/dv_k, sum f (x) R^T w> with dR/dv of cal_grad_of_rot_over_vec
// (E/src/geometry/rotation.h:80-144) evaluated at v', the rotation vector of the
// same rotation with its angle in [0, pi] (rotvec_to_axis_angle(norm = true),
// rotation.h:19-46). Since dR/dv'_k R^T = [J(v') e_k]x with J the left Jacobian of
// SO(3), g = J(v')^T tau, tau = sum_a (x_a - c) x f_a:
//   g = tau - a v' x tau + b v' x (v' x tau), a = (1 - cos t)/t^2, b = (t - sin t)/t^3.
__device__ __forceinline__ float3 orient_grad(float v0, float v1, float v2, float t0, float t1, float t2) {
    const float ang = fsqrt(sq_dist(v0, v1, v2));
    float th = 0.0f, w0 = 0.0f, w1 = 0.0f, w2 = 0.0f;
    if (ang > kEps) {
        th = ang - 2.0f * kPi * floorf(ang * (1.0f / (2.0f * kPi)));  // normalize_angle_2pi
        float sg = 1.0f;
        if (th > kPi) { th = 2.0f * kPi - th; sg = -1.0f; }
        const float k = sg * th * frcp(ang);
        w0 = v0 * k; w1 = v1 * k; w2 = v2 * k;
    }
    const float q = th * th;
    float a, b;
    if (th < 0.5f) {  // Taylor series; truncation error below 1e-9 at th = 0.5
        a = 0.5f - q * (1.0f / 24.0f - q * (1.0f / 720.0f - q * (1.0f / 40320.0f)));
        b = (1.0f / 6.0f) - q * (1.0f / 120.0f - q * (1.0f / 5040.0f - q * (1.0f / 362880.0f)));
    } else {
        float s, c;
        __sincosf(th, &s, &c);  // th in [0.5, pi]
        const float iq = frcp(q);
        a = (1.0f - c) * iq;
        b = (th - s) * iq * frcp(th);
    }
    const float c0 = msub2(w1, t2, w2, t1), c1 = msub2(w2, t0, w0, t2), c2 = msub2(w0, t1, w1, t0);  // v' x tau
    const float d0 = msub2(w1, c2, w2, c1), d1 = msub2(w2, c0, w0, c2), d2 = msub2(w0, c1, w1, c0);  // v' x (v' x tau)
    return make_float3(fmaf_(b, d0, fmaf_(-a, c0, t0)), fmaf_(b, d1, fmaf_(-a, c1, t1)), fmaf_(b, d2, fmaf_(-a, c2, t2)));
}

// Trilinear value and gradient of map `slot` at p; clamped axes have zero derivative.
__device__ __forceinline__ float grid_eval(SceneArg& S, int slot, float px, float py, float pz, float& gx,
                                          float& gy, float& gz) {
    float g[3] = {(px - S.gorigin[0]) * S.ginv, (py - S.gorigin[1]) * S.ginv, (pz - S.gorigin[2]) * S.ginv};
    int i0[3];
    float fr[3];
    bool cl[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        float top = float(S.gn[d] - 1);
        cl[d] = !(g[d] >= 0.0f && g[d] <= top);
        float v = fminf(fmaxf(g[d], 0.0f), top);
        int i = int(floorf(v));
        i = i > S.gn[d] - 2 ? S.gn[d] - 2 : i;
        i0[d] = i;
        fr[d] = v - float(i);
    }
    // the cell's 8 corners: one 32-byte sector of the cell-major copy
    const int cx = S.gn[0] - 1, cxy = cx * (S.gn[1] - 1);
    const float4* m = S.cells + 2 * ((size_t)slot * (size_t)cxy * (S.gn[2] - 1) + (size_t)i0[2] * cxy + i0[1] * cx + i0[0]);
    const float4 lo = m[0], hi = m[1];
    const float c000 = lo.x, c100 = lo.y, c010 = lo.z, c110 = lo.w;
    const float c001 = hi.x, c101 = hi.y, c011 = hi.z, c111 = hi.w;
    float fx = fr[0], fy = fr[1], fz = fr[2], hx = 1.0f - fx, hy = 1.0f - fy, hz = 1.0f - fz;
    float v00 = madd2(c000, hx, c100, fx), v10 = madd2(c010, hx, c110, fx);
    float v01 = madd2(c001, hx, c101, fx), v11 = madd2(c011, hx, c111, fx);
    float v0 = madd2(v00, hy, v10, fy), v1 = madd2(v01, hy, v11, fy);
    float dx = madd2(madd2(c100 - c000, hy, c110 - c010, fy), hz, madd2(c101 - c001, hy, c111 - c011, fy), fz);
    float dy = madd2(v10 - v00, hz, v11 - v01, fz);
    float dz = v1 - v0;
    gx = cl[0] ? 0.0f : dx * S.ginv;
    gy = cl[1] ? 0.0f : dy * S.ginv;
    gz = cl[2] ? 0.0f : dz * S.ginv;
    return madd2(v0, hz, v1, fz);
}

// ----------------------------------------------------------------- state
template <int APL>
struct WPose {
    float x[APL], y[APL], z[APL];
    float c0, c1, c2;   // centre (uniform)
    float r0, r1, r2;   // rot_vec of the last rotation increment (uniform)
    float dihe;         // lane t: dihedral t
    float e;            // energy (uniform)
};

// Per-tile constants of the ligand being processed: its descriptor and the kernel's arguments are read
// where they are used (see reread), the lane's own values are kept. The tile's LDS slice
// (offsets in floats into s_lds) holds: lx float4 coordinates [TW*APL], lf
// pair-force tile [3][TW*APL], lo a saved pose, lt the ligand's torsion table,
// lh the inverse Hessian (row i at lh + i * ld).
template <int APL, int TW = kWave, bool LAZY = true>
struct Ctx {
    KHead* K;
    KLig* lig;
    int base, ld;
    int type[APL];      // XS type; -1 for lanes beyond natom
    int slot[APL];      // grid map of the atom's type
    float rad[APL];     // vdW radius of the atom's type (0 beyond natom)
    uint32_t lut[APL];  // pair flags with a partner of doubled type flags f: (lut >> f) & 3 (see pair_lut)
    int mode;
    mutable int evals;  // energy evaluations of the current work item
    bool stage;         // pose updates may stage torsion steps in the coordinate / pair-force area

    // LAZY: read where used; else left to the compiler to load once and keep, which a kernel that has
    // registers to spare and no other waves to hide a scalar load behind runs faster with.
    template <class T>
    static __device__ __forceinline__ T lazy(T v) {
        if constexpr (LAZY) return reread(v);
        else return v;
    }
    __device__ __forceinline__ LigArg& L() const { return lazy(K)->L; }
    __device__ __forceinline__ SceneArg& S() const { return lazy(K)->S; }
    __device__ __forceinline__ KLig& d() const { return *lazy(lig); }
    __device__ __forceinline__ bool biased() const {
        LigArg& l = L();
        return l.bias_type != 0 && l.bias_start;
    }
    __device__ __forceinline__ int natom() const { return d().natom; }
    __device__ __forceinline__ int ntors() const { return d().ntors; }
    __device__ __forceinline__ int npair() const { return d().npair; }
    __device__ __forceinline__ int nheavy() const { return d().nheavy; }
    __device__ __forceinline__ int dim() const { return 6 + d().ntors; }
    __device__ __forceinline__ int lx() const {
        if constexpr (TW == kWave) return lazy(base);
        else return base;
    }
    __device__ __forceinline__ int lf() const { return lx() + 4 * TW * APL; }
    __device__ __forceinline__ int lo() const { return lx() + 7 * TW * APL; }
    __device__ __forceinline__ int lfl() const { return lx() + lds_flags_offset(APL, TW); }
    __device__ __forceinline__ int lt() const { return lx() + lds_fixed_floats(APL, TW); }
    __device__ __forceinline__ int lh() const { return lx() + lds_head_floats(APL, ld, TW); }
};

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void load_ctx(Ctx<APL, TW, LAZY>& C, KHead* K, int lig, int mode, int base, int ld) {
    static_assert(TW == kWave || APL == 1, "a tile narrower than the wave holds one atom per lane");
    const int tl = tlane<TW>();
    // the same for every lane of the wave (base: of the tile)
    C.K = K;
    C.lig = (KLig*)(K->L.ligs + __builtin_amdgcn_readfirstlane(lig));
    C.base = TW == kWave ? __builtin_amdgcn_readfirstlane(base) : base;
    C.ld = ld;
    C.mode = mode;
    C.evals = 0;
    C.stage = true;
    LigArg& L = C.L();
    SceneArg& S = C.S();
    KLig& d = C.d();
    const int lfl = C.lfl(), lt = C.lt();
#pragma unroll
    for (int k = 0; k < APL; k++) {
        int a = tl + TW * k;
        C.type[k] = a < d.natom ? __float_as_int(L.atom_x0[d.atom_off + a].w) : -1;
        C.slot[k] = (mode == kGrid && C.type[k] > 0) ? S.slot_tab[C.type[k]] : 0;
        const int fa = C.type[k] >= 0 ? c_tflags[C.type[k]] : 0;
        C.rad[k] = C.type[k] >= 0 ? c_vdw[C.type[k]] : 0.0f;
        C.lut[k] = pair_lut(fa);
        // the atom's doubled type flags, read by its pair partners; this part of the slice is not
        // overlaid by anything else, so it is written once per work item
        reinterpret_cast<int*>(s_lds + lfl)[a] = 2 * fa;
    }
    // torsion table: lane t copies torsion t once, so the kinematics and the gradient read
    // the torsion tree from LDS instead of global memory on every step
    if (tl < d.ntors) {
        const int tg = d.tors_off + tl;
        const int2 ax = L.tors_axis[tg];
        const int2 rr = L.tors_range[tg];
        const float2 r0 = L.ranges[rr.x];
        float* e = s_lds + lt + tl * tors_entry_floats(APL);
        // from | to << 8 | order << 16 | rank << 24 (atoms < 256, torsions < 64)
        const int word = (ax.x & 0xff) | ((ax.y & 0xff) << 8) | (((ax.y >> 16) & 0xff) << 16) | (((ax.x >> 16) & 0xff) << 24);
        *reinterpret_cast<float4*>(e) = make_float4(__int_as_float(word), __int_as_float(rr.y), r0.x, r0.y);
#pragma unroll
        for (int k = 0; k < APL; k++) {
            const unsigned long long m = L.tors_mask[(size_t)tg * kMaxApl + k];
            e[4 + 2 * k] = __uint_as_float(uint32_t(m));
            e[5 + 2 * k] = __uint_as_float(uint32_t(m >> 32));
        }
    }
    wave_lds_fence();
}

// Entry t of the torsion table: axis atoms, number of allowed ranges and the first range, ord, the
// torsion applied t-th in leaf-first order, and rank, the place of torsion t in that order.
struct TorsEnt {
    int from, to, ord, rank, nrange;
    float lo, hi;
};

template <int APL>
__device__ __forceinline__ TorsEnt tors_ent_at(int lt, int t) {
    const float4 h = *reinterpret_cast<const float4*>(s_lds + lt + t * tors_entry_floats(APL));
    const int ax = __float_as_int(h.x);
    TorsEnt e;
    e.from = ax & 0xff;
    e.to = (ax >> 8) & 0xff;
    e.ord = (ax >> 16) & 0xff;
    e.rank = (ax >> 24) & 0xff;
    e.nrange = __float_as_int(h.y);
    e.lo = h.z;
    e.hi = h.w;
    return e;
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ TorsEnt tors_ent(const Ctx<APL, TW, LAZY>& C, int t) { return tors_ent_at<APL>(C.lt(), t); }

// Rotated-atom mask of torsion t over atom slot k (bit l = atom l + 64 k).
template <int APL>
__device__ __forceinline__ unsigned long long tors_mask_at(int lt, int t, int k) {
    const float2 m = *reinterpret_cast<const float2*>(s_lds + lt + t * tors_entry_floats(APL) + 4 + 2 * k);
    return (unsigned long long)__float_as_uint(m.x) | ((unsigned long long)__float_as_uint(m.y) << 32);
}
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ unsigned long long tors_mask(const Ctx<APL, TW, LAZY>& C, int t, int k) {
    return tors_mask_at<APL>(C.lt(), t, k);
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ bool heavy(const Ctx<APL, TW, LAZY>& C, int k) { return C.type[k] > kTypeH; }
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ bool valid(const Ctx<APL, TW, LAZY>& C, int k) { return C.type[k] >= 0; }

// Position of atom a (tile lane a % TW, slot a / TW), a the same for every lane of the tile.
template <int TW, int APL>
__device__ __forceinline__ float3 atom_pos(const WPose<APL>& P, int a) {
    const int k = a / TW, l = a % TW;
    float3 r = make_float3(0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int kk = 0; kk < APL; kk++)
        if (kk == k) r = make_float3(tread<TW>(P.x[kk], l), tread<TW>(P.y[kk], l), tread<TW>(P.z[kk], l));
    return r;
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void centroid(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P) {
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++)
        if (valid(C, k)) { sx += P.x[k]; sy += P.y[k]; sz += P.z[k]; }
    const float inv = 1.0f / float(C.natom());
    const float c = tsum4<TW>(tlane<TW>(), sx, sy, sz, 0.0f) * inv;
    P.c0 = trdl<TW>(c, 0);
    P.c1 = trdl<TW>(c, 1);
    P.c2 = trdl<TW>(c, 2);
}

// Pose slots in the wave's LDS slice: slot 0 parks the BFGS start pose, slot 1
// the accepted MC pose. A slot holds x, y, z per atom and the dihedrals per lane,
// then c, rot_vec and the energy.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ int pose_slot(const Ctx<APL, TW, LAZY>& C, int slot) {
    return C.lo() + slot * (TW * (3 * APL + 1) + 8);
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void save_pose(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, int slot = 0) {
    const int ln = tlane<TW>();
    const int lo = pose_slot(C, slot);
#pragma unroll
    for (int k = 0; k < APL; k++) {
        s_lds[lo + (3 * k) * TW + ln] = P.x[k];
        s_lds[lo + (3 * k + 1) * TW + ln] = P.y[k];
        s_lds[lo + (3 * k + 2) * TW + ln] = P.z[k];
    }
    s_lds[lo + 3 * APL * TW + ln] = P.dihe;
    const int u = lo + (3 * APL + 1) * TW;
    if (ln == 0) {
        s_lds[u] = P.c0; s_lds[u + 1] = P.c1; s_lds[u + 2] = P.c2;
        s_lds[u + 3] = P.r0; s_lds[u + 4] = P.r1; s_lds[u + 5] = P.r2;
        s_lds[u + 6] = P.e;
    }
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void restore_pose(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, int slot = 0) {
    wave_lds_fence();
    const int ln = tlane<TW>();
    const int lo = pose_slot(C, slot);
#pragma unroll
    for (int k = 0; k < APL; k++) {
        P.x[k] = s_lds[lo + (3 * k) * TW + ln];
        P.y[k] = s_lds[lo + (3 * k + 1) * TW + ln];
        P.z[k] = s_lds[lo + (3 * k + 2) * TW + ln];
    }
    P.dihe = s_lds[lo + 3 * APL * TW + ln];
    const int u = lo + (3 * APL + 1) * TW;
    P.c0 = tuni<TW>(s_lds[u]); P.c1 = tuni<TW>(s_lds[u + 1]); P.c2 = tuni<TW>(s_lds[u + 2]);
    P.r0 = tuni<TW>(s_lds[u + 3]); P.r1 = tuni<TW>(s_lds[u + 4]); P.r2 = tuni<TW>(s_lds[u + 5]);
    P.e = tuni<TW>(s_lds[u + 6]);
}

// clamp_by_ranges (E/src/myutils/mymath.h:133-158) over the torsion's ranges.
__device__ __forceinline__ float clamp_ranges(LigArg& L, int tg, float ang) {
    const int2 rr = L.tors_range[tg];
    for (int i = 0; i < rr.y; i++) {
        const float2 r = L.ranges[rr.x + i];
        if (ang >= r.x && ang <= r.y) return ang;
    }
    float best = ang, md = 100.0f;
    for (int i = 0; i < rr.y; i++) {
        const float2 r = L.ranges[rr.x + i];
        const float dl = fabsf(ang - r.x), dh = fabsf(ang - r.y);
        if (dl < md) { md = dl; best = r.x; }
        if (dh < md) { md = dh; best = r.y; }
    }
    return best;
}

// clamp_ranges of torsion t from its table entry: one allowed range inline, more from global memory.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float clamp_tors(const Ctx<APL, TW, LAZY>& C, const TorsEnt& e, int tg, float ang) {
    if (e.nrange != 1) return clamp_ranges(C.L(), tg, ang);
    if (ang >= e.lo && ang <= e.hi) return ang;
    const float dl = fabsf(ang - e.lo), dh = fabsf(ang - e.hi);
    float best = ang, md = 100.0f;
    if (dl < md) { md = dl; best = e.lo; }
    if (dh < md) best = e.hi;
    return best;
}

// One torsion step, apply_grad_update_dihe_tile (E/src/cuda/bfgs.cuh:443-527);
// the centroid is refreshed by the caller after the last torsion (only the
// final centroid is ever read, bfgs.cuh:531-548, 576-578).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void apply_torsion(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, int t, float inc_raw) {
    const int tg = C.d().tors_off + t;
    const TorsEnt te = tors_ent(C, t);
    const float dt = tread<TW>(P.dihe, t);
    float inc = normalize_angle(inc_raw);
    const float nw = tuni<TW>(clamp_tors(C, te, tg, normalize_angle(dt + inc)));
    inc = nw - dt;
    if (tlane<TW>() == t) P.dihe = nw;
    const float3 xt = atom_pos<TW>(P, te.to), xf = atom_pos<TW>(P, te.from);
    float ux = xt.x - xf.x, uy = xt.y - xf.y, uz = xt.z - xf.z;
    const float l = fsqrt(sq_dist(ux, uy, uz));
    if (l <= kEps) { ux = 1.0f; uy = 0.0f; uz = 0.0f; }
    else { const float il = frcp(l); ux *= il; uy *= il; uz *= il; }
    float s, c;
    __sincosf(inc, &s, &c);
    const float rn = frsq(madd2(c, c, s, s));  // unit (c, s): no growth of the rotated fragment per step
    ux = tuni<TW>(ux); uy = tuni<TW>(uy); uz = tuni<TW>(uz); s = tuni<TW>(s * rn); c = tuni<TW>(c * rn);
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const unsigned long long mk = tors_mask(C, t, k);
        if ((mk >> tlane<TW>()) & 1ull) {
            const float vx = P.x[k] - xt.x, vy = P.y[k] - xt.y, vz = P.z[k] - xt.z;
            const float m = (1.0f - c) * madd3(ux, vx, uy, vy, uz, vz);
            const float cxv = msub2(uy, vz, uz, vy), cyv = msub2(uz, vx, ux, vz), czv = msub2(ux, vy, uy, vx);
            P.x[k] = madd3(c, vx, m, ux, s, cxv) + xt.x;
            P.y[k] = madd3(c, vy, m, uy, s, cyv) + xt.y;
            P.z[k] = madd3(c, vz, m, uz, s, czv) + xt.z;
        }
    }
}

// Rigid rotation about o by q, then translation so that o maps to n.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void rigid_move(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, float4 q, float ox, float oy, float oz,
                                           float nx, float ny, float nz) {
    Mat3 R = quat_to_mat(q);
#pragma unroll
    for (int i = 0; i < 9; i++) R.m[i] = tuni<TW>(R.m[i]);
#pragma unroll
    for (int k = 0; k < APL; k++) {
        if (!valid(C, k)) continue;
        const float wx = P.x[k] - ox, wy = P.y[k] - oy, wz = P.z[k] - oz;
        P.x[k] = madd3(R.m[0], wx, R.m[1], wy, R.m[2], wz) + nx;
        P.y[k] = madd3(R.m[3], wx, R.m[4], wy, R.m[5], wz) + ny;
        P.z[k] = madd3(R.m[6], wx, R.m[7], wy, R.m[8], wz) + nz;
    }
}

// Position of atom a (tile lane a % TW, slot a / TW) for every lane, each with its own a.
template <int TW, int APL>
__device__ __forceinline__ float3 lane_gather(const WPose<APL>& P, int a) {
    float3 r = make_float3(0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const float x = tshfl<TW>(P.x[k], a), y = tshfl<TW>(P.y[k], a), z = tshfl<TW>(P.z[k], a);
        if (a / TW == k) r = make_float3(x, y, z);
    }
    return r;
}

// Staged torsion steps of one pose update: a rotation matrix R (9 floats), the pivot (3) and the
// rotated-atom mask words (2 per atom slot) per torsion, padded to 16-byte rows, in the slice's
// coordinate / pair-force area (idle between an energy's gradient and the next evaluation).
template <int APL>
__host__ __device__ constexpr int tstage_floats() { return (12 + 2 * APL + 3) & ~3; }
template <int APL, int TW = kWave>
__host__ __device__ constexpr int tstage_cap() { return 7 * TW * APL / tstage_floats<APL>(); }
static_assert(tstage_cap<1, kTileNarrow>() == kTileNarrowTors, "narrow tiles take the ligands whose torsion steps they stage");

// All torsion steps of one pose update, leaf first. A torsion's pivot and axis atoms are
// moved only by its ancestors, which come later, so lane t first computes torsion t's step
// from the coordinates before the update: the angle normalised and clamped into the allowed
// ranges (as apply_torsion), the pivot, the unit axis and (cos, sin), as a rotation matrix. The
// steps are staged in LDS in application order and the rotations then read them with broadcast LDS
// loads (no VALU work per value), each masked atom moved as R (x - p) + p. Ligands with more
// torsions than the stage holds read the steps from the torsion lanes instead.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void apply_torsions_leaf_first(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, float dir, float alpha) {
    const int ln = tlane<TW>(), nt = C.ntors();
    const float inc_raw = tshfl<TW>(dir, ln + 6) * alpha;  // torsion components sit on lanes 6 + t
    // every lane reads an entry (lanes past ntors read entry 0) and gathers its axis atoms
    const TorsEnt te = tors_ent(C, ln < nt ? ln : 0);
    const float3 xt = lane_gather<TW>(P, te.to), xf = lane_gather<TW>(P, te.from);
    float px = 0.0f, py = 0.0f, pz = 0.0f, ux = 1.0f, uy = 0.0f, uz = 0.0f, c = 1.0f, s = 0.0f;
    int ord = 0;
    uint32_t mlo[APL], mhi[APL];
#pragma unroll
    for (int k = 0; k < APL; k++) mlo[k] = mhi[k] = 0u;
    if (ln < nt) {
        ord = te.ord;
        float inc = normalize_angle(inc_raw);
        const float nw = clamp_tors(C, te, C.d().tors_off + ln, normalize_angle(P.dihe + inc));
        inc = nw - P.dihe;
        P.dihe = nw;
        px = xt.x; py = xt.y; pz = xt.z;
        const float ax = xt.x - xf.x, ay = xt.y - xf.y, az = xt.z - xf.z;
        const float l = fsqrt(sq_dist(ax, ay, az));
        if (l > kEps) { const float il = frcp(l); ux = ax * il; uy = ay * il; uz = az * il; }
        __sincosf(inc, &s, &c);
        const float rn = frsq(madd2(c, c, s, s));
        s *= rn;
        c *= rn;
#pragma unroll
        for (int k = 0; k < APL; k++) {
            const unsigned long long m = tors_mask(C, ln, k);
            mlo[k] = uint32_t(m);
            mhi[k] = uint32_t(m >> 32);
        }
    }
    if (C.stage && nt <= tstage_cap<APL, TW>()) {
        constexpr int SE = tstage_floats<APL>();
        const int lx = C.lx();
        if (ln < nt) {
            // Rodrigues: R = c I + s [u]x + (1 - c) u u^T
            const float oc = 1.0f - c;
            float* st = s_lds + lx + te.rank * SE;
            const float ox = oc * ux, oy = oc * uy, oz = oc * uz;
            reinterpret_cast<float4*>(st)[0] =
                make_float4(fmaf_(ox, ux, c), msub2(ox, uy, s, uz), madd2(ox, uz, s, uy), madd2(oy, ux, s, uz));
            reinterpret_cast<float4*>(st)[1] =
                make_float4(fmaf_(oy, uy, c), msub2(oy, uz, s, ux), msub2(oz, ux, s, uy), madd2(oz, uy, s, ux));
            reinterpret_cast<float4*>(st)[2] = make_float4(fmaf_(oz, uz, c), px, py, pz);
#pragma unroll
            for (int k = 0; k < APL; k++) {
                st[12 + 2 * k] = __uint_as_float(mlo[k]);
                st[13 + 2 * k] = __uint_as_float(mhi[k]);
            }
        }
        wave_lds_fence();
#pragma unroll 1
        for (int q = 0; q < nt; q++) {
            const float* st = s_lds + lx + q * SE;
            const float4 r0 = reinterpret_cast<const float4*>(st)[0], r1 = reinterpret_cast<const float4*>(st)[1],
                         r2 = reinterpret_cast<const float4*>(st)[2];
#pragma unroll
            for (int k = 0; k < APL; k++) {
                // the masks are the ligand's (every tile of the wave stages the same words)
                const uint32_t lo = __builtin_amdgcn_readfirstlane(__float_as_uint(st[12 + 2 * k]));
                const uint32_t hi = __builtin_amdgcn_readfirstlane(__float_as_uint(st[13 + 2 * k]));
                if (__builtin_amdgcn_inverse_ballot_w64(tmask<TW>((unsigned long long)lo | ((unsigned long long)hi << 32)))) {
                    const float vx = P.x[k] - r2.y, vy = P.y[k] - r2.z, vz = P.z[k] - r2.w;
                    P.x[k] = madd3(r0.x, vx, r0.y, vy, r0.z, vz) + r2.y;
                    P.y[k] = madd3(r0.w, vx, r1.x, vy, r1.y, vz) + r2.z;
                    P.z[k] = madd3(r1.z, vx, r1.w, vy, r2.x, vz) + r2.w;
                }
            }
        }
        wave_lds_fence();
        return;
    }
#pragma unroll 1
    for (int q = 0; q < nt; q++) {
        if constexpr (TW == kWave) {
            const int t = rdl_i(ord, q);
            const float tx = rdl(px, t), ty = rdl(py, t), tz = rdl(pz, t);
            const float vx0 = rdl(ux, t), vy0 = rdl(uy, t), vz0 = rdl(uz, t), ct = rdl(c, t), st = rdl(s, t);
#pragma unroll
            for (int k = 0; k < APL; k++) {
                const uint32_t wlo = uint32_t(rdl_i(int(mlo[k]), t)), whi = uint32_t(rdl_i(int(mhi[k]), t));
                const uint32_t w = ln < 32 ? wlo : whi;
                if ((w >> (ln & 31)) & 1u) {
                    const float vx = P.x[k] - tx, vy = P.y[k] - ty, vz = P.z[k] - tz;
                    const float m = (1.0f - ct) * madd3(vx0, vx, vy0, vy, vz0, vz);
                    const float cxv = msub2(vy0, vz, vz0, vy), cyv = msub2(vz0, vx, vx0, vz), czv = msub2(vx0, vy, vy0, vx);
                    P.x[k] = madd3(ct, vx, m, vx0, st, cxv) + tx;
                    P.y[k] = madd3(ct, vy, m, vy0, st, cyv) + ty;
                    P.z[k] = madd3(ct, vz, m, vz0, st, czv) + tz;
                }
            }
        } else {
            // a narrow tile holds at most 32 atoms: the low mask word of torsion t covers them
            const int t = tshfl_i<TW>(ord, q);
            const float tx = tshfl<TW>(px, t), ty = tshfl<TW>(py, t), tz = tshfl<TW>(pz, t);
            const float vx0 = tshfl<TW>(ux, t), vy0 = tshfl<TW>(uy, t), vz0 = tshfl<TW>(uz, t);
            const float ct = tshfl<TW>(c, t), st = tshfl<TW>(s, t);
            const uint32_t w = uint32_t(tshfl_i<TW>(int(mlo[0]), t));
            if ((w >> ln) & 1u) {
                const float vx = P.x[0] - tx, vy = P.y[0] - ty, vz = P.z[0] - tz;
                const float m = (1.0f - ct) * madd3(vx0, vx, vy0, vy, vz0, vz);
                const float cxv = msub2(vy0, vz, vz0, vy), cyv = msub2(vz0, vx, vx0, vz), czv = msub2(vx0, vy, vy0, vx);
                P.x[0] = madd3(ct, vx, m, vx0, st, cxv) + tx;
                P.y[0] = madd3(ct, vy, m, vy0, st, cyv) + ty;
                P.z[0] = madd3(ct, vz, m, vz0, st, czv) + tz;
            }
        }
    }
}

// apply_grad_update_pose_tile (bfgs.cuh:560-618): torsions (leaf first when the
// ligand's torsion tree allows it, else in index order), then centre += alpha *
// dir[0..2] and a rotation by q(alpha * dir[3..5]) about the old centre;
// rot_vec := alpha * dir[3..5]. dir is lane-distributed.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void apply_update(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, float dir, float alpha) {
    const int nt = C.ntors();
    if (C.d().leaf_first) {
        if (nt > 0) apply_torsions_leaf_first(C, P, dir, alpha);
    } else {
#pragma unroll 1
        for (int t = 0; t < nt; t++) apply_torsion(C, P, t, trdl<TW>(dir, 6 + t) * alpha);
    }
    if (nt > 0) centroid(C, P);
    if (C.L().constraint) return;  // constraint docking: no rigid step (bfgs.cuh:571)
    const float o0 = P.c0, o1 = P.c1, o2 = P.c2;
    P.c0 = tuni<TW>(o0 + alpha * trdl<TW>(dir, 0));
    P.c1 = tuni<TW>(o1 + alpha * trdl<TW>(dir, 1));
    P.c2 = tuni<TW>(o2 + alpha * trdl<TW>(dir, 2));
    const float v0 = tuni<TW>(trdl<TW>(dir, 3) * alpha), v1 = tuni<TW>(trdl<TW>(dir, 4) * alpha),
                v2 = tuni<TW>(trdl<TW>(dir, 5) * alpha);
    const float4 q = rotvec_to_quat(v0, v1, v2);
    P.r0 = v0; P.r1 = v1; P.r2 = v2;
    rigid_move(C, P, q, o0, o1, o2, P.c0, P.c1, P.c2);
}

// Per-atom energy gradient (-force) of one evaluation, atom a on lane a % 64.
template <int APL>
struct Forces {
    float fx[APL], fy[APL], fz[APL];
};

// Energy of bias site b (x, y, z, V) at atom position p, and s with dE/dp = s * r,
// r = site - p. pos: Gaussian well V k exp(-|r|^2 / r2) (Vina::eval_ef_pos,
// E/src/score/vina.h:277-289). align: a k k_a / (1 + exp(3 (1 - |r|))), k_a = 0.1 for
// hydrogen, else 30 (Vina::eval_ef_zalign, vina.h:306-324; |r| = 0 divides by zero
// as there).
__device__ __forceinline__ float bias_site_energy(int bias_type, float bias_k, float4 b, float r2, int type,
                                                  float rx, float ry, float rz, float& s) {
    const float v = b.w * bias_k;
    const float rr = sq_dist(rx, ry, rz);
    if (bias_type == 1) {
        const float e = v * __expf(-rr / r2);
        s = e * 2.0f / r2;
        return e;
    }
    const float d = sqrtf(rr);
    const float ka = type == kTypeH ? 0.1f : 30.0f;
    const float ei = __expf(3.0f * (1.0f - d));
    const float e = v * ka / (1.0f + ei);
    s = -e * ei / (1.0f + ei) * 3.0f / d;
    return e;
}

// Bias sites of every atom (hydrogens included), uncurled (the bias block of
// cal_e_f_tile, bfgs.cuh:355-388): returns this lane's energy and adds dE/dx to F.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float bias_forces(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, Forces<APL>& F) {
    LigArg& L = C.L();
    float e = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        if (!valid(C, k)) continue;
        const int a = C.d().atom_off + tlane<TW>() + TW * k;
        const int j1 = L.bias_start[a + 1];
        for (int j = L.bias_start[a]; j < j1; j++) {
            const float4 b = L.bias_site[j];
            const float rx = b.x - P.x[k], ry = b.y - P.y[k], rz = b.z - P.z[k];
            float s;
            e += bias_site_energy(L.bias_type, L.bias_k, b, L.bias_r2[j], C.type[k], rx, ry, rz, s);
            F.fx[k] += s * rx; F.fy[k] += s * ry; F.fz[k] += s * rz;
        }
    }
    return e;
}

// Byte address of lane l for ds_bpermute.
__device__ __forceinline__ int lane_addr(int l) { return l << 2; }
__device__ __forceinline__ float bperm(int addr, float v) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}

// Exchange of a vector per lane through the wave's pair-force tile (x, y and z, 64 floats each at f): every lane
// puts its own, then reads those of any lanes by their byte offsets 4 * lane.
__device__ __forceinline__ void share_put(int f, int ln, float x, float y, float z) {
    wave_lds_fence();
    s_lds[f + ln] = x;
    s_lds[f + kWave + ln] = y;
    s_lds[f + 2 * kWave + ln] = z;
    wave_lds_fence();
}
__device__ __forceinline__ float3 share_get(int f, uint32_t off) {
    const float* p = reinterpret_cast<const float*>(reinterpret_cast<const char*>(s_lds + f) + off);
    return make_float3(p[0], p[kWave], p[2 * kWave]);
}

// One intra pair (bfgs.cuh:305-353) within the cutoff, at separation (rx, ry, rz) = x_i - x_j, its square rr,
// radius sum rs and flag constants kh, kb: the curled pair energy and the energy gradient on i; the
// partner's is the negative. The per-pair curl has cap v_cap.
__device__ __forceinline__ float pair_core(float rx, float ry, float rz, float rr, float rs, float kh, float kb,
                                           float v_cap, float& px, float& py, float& pz) {
    // r and 1 / r from one reciprocal square root; eps^2 keeps coincident atoms finite (it is below
    // half an ulp of any squared distance that is not tiny)
    const float inv = frsq(rr + kEps * kEps);
    float dd;
    const float ep = eval_ramps(fmaf_(rr, inv, -rs), kh, kb, &dd);
    const float cs = ep > 0.0f ? v_cap * frcp(v_cap + ep) : 1.0f;
    const float sc = dd * inv * (cs * cs);
    px = sc * rx; py = sc * ry; pz = sc * rz;
    return opaque(ep * cs);  // a rounded product, not fused into the sum it is added to
}

// The pair of an atom at (xi, yi, zi) (radius ri, pair-flag table lut) with the LDS slot (x, y, z, radius) xj of
// doubled type flags fj2; zero beyond the 8 A cutoff. SKIP: by a branch, which pays where a wave's pairs are often all
// beyond it; three and four slots per lane are computed side by side without (8 ligands of 200 atoms searched 53.6 -> 46.7 ms,
// 100,000 evaluations of one 8.17 -> 7.59).
template <bool SKIP = true>
__device__ __forceinline__ float pair_grad(float xi, float yi, float zi, float ri, uint32_t lut, float4 xj, int fj2,
                                           float v_cap, float& px, float& py, float& pz) {
    const float rx = xi - xj.x, ry = yi - xj.y, rz = zi - xj.z;
    const float rr = sq_dist(rx, ry, rz);
    const bool in = rr < kR2Cut;
    if (SKIP && !in) return 0.0f;
    const int fl = int(lut >> fj2) & 3;
    const float e = pair_core(rx, ry, rz, rr, ri + xj.w, ramp_hyd(fl), ramp_hb(fl), v_cap, px, py, pz);
    if constexpr (!SKIP) {
        px = in ? px : 0.0f;
        py = in ? py : 0.0f;
        pz = in ? pz : 0.0f;
        return in ? e : 0.0f;
    }
    return e;
}

// cal_e_f_tile (bfgs.cuh:221-394): energy under the curl cap v_cap and the
// per-atom gradient F.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float energy_forces(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, float v_cap, float slope, Forces<APL>& F) {
    SceneArg& S = C.S();
    const int ln = tlane<TW>();
    const int n3 = TW * APL;
    const int lx = C.lx(), lf = lx + 4 * TW * APL;
    float* fx = F.fx;
    float* fy = F.fy;
    float* fz = F.fz;
    float e = 0.0f;
    C.evals++;
    // coordinates and radii to LDS for the pair loop
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = ln + TW * k;
        reinterpret_cast<float4*>(s_lds + lx)[a] = make_float4(P.x[k], P.y[k], P.z[k], C.rad[k]);
    }
    // inter-molecular term with the per-atom curl, and the box penalty
#pragma unroll
    for (int k = 0; k < APL; k++) {
        fx[k] = fy[k] = fz[k] = 0.0f;
        if (!heavy(C, k)) continue;
        float ea = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
        if (C.mode == kGrid) {
            ea = grid_eval(S, C.slot[k], P.x[k], P.y[k], P.z[k], gx, gy, gz);
        } else {
            const float ri = C.rad[k];
            for_reach(S, reach_of(S, P.x[k], P.y[k], P.z[k]), [&](float qx, float qy, float qz, uint32_t word) {
                const float rx = qx - P.x[k], ry = qy - P.y[k], rz = qz - P.z[k];
                const float rr = sq_dist(rx, ry, rz);
                if (rr < kR2Cut) {
                    float d = fsqrt(rr), dd;
                    ea += eval_ef(d - (ri + word_radius(word)), int(C.lut[k] >> word_flags2(word)) & 3, &dd);
                    d = fmaxf(d, kEps);
                    const float fdr = dd * frcp(d);
                    gx -= fdr * rx; gy -= fdr * ry; gz -= fdr * rz;
                }
            });
        }
        if (ea > 0.0f) {
            float s = v_cap * frcp(v_cap + ea);
            ea *= s;
            s *= s;
            gx *= s; gy *= s; gz *= s;
        }
        e += ea;
        // cal_box_penalty (bfgs.cuh:196-218)
        float pen = 0.0f;
        if (P.x[k] < S.box_lo[0]) { pen += S.box_lo[0] - P.x[k]; gx -= slope; }
        if (P.x[k] > S.box_hi[0]) { pen += P.x[k] - S.box_hi[0]; gx += slope; }
        if (P.y[k] < S.box_lo[1]) { pen += S.box_lo[1] - P.y[k]; gy -= slope; }
        if (P.y[k] > S.box_hi[1]) { pen += P.y[k] - S.box_hi[1]; gy += slope; }
        if (P.z[k] < S.box_lo[2]) { pen += S.box_lo[2] - P.z[k]; gz -= slope; }
        if (P.z[k] > S.box_hi[2]) { pen += P.z[k] - S.box_hi[2]; gz += slope; }
        e += pen * slope;
        fx[k] = gx; fy[k] = gy; fz[k] = gz;
    }
    wave_lds_fence();
    // The diagonals' masks are uniform: scalar loads, used as the lane condition directly.
    const unsigned long long* fm = C.L().fold_mask + C.d().fold_off;
    const float4* lx4 = reinterpret_cast<const float4*>(s_lds + lx);
    const int* lfl = reinterpret_cast<const int*>(s_lds + C.lfl());
    const int n = C.natom(), nfold = C.d().nfold;
    if constexpr (TW < kWave) {
        // A 32-lane tile (at most 32 atoms): the two diagonals dg and dg + 1 of a step are scored one
        // after the other by the same lanes, with the sums the whole-wave path forms over its two
        // halves: lane a adds both pair gradients of its atom and the partner shares from lanes
        // (a - dg) and (a - dg - 1) mod natom, and the energies of the two diagonals are kept apart
        // and summed row by row in the whole-wave order, so a chain computes the same bits either way.
        const int a = ln;
        const float4 xa = lx4[a];
        int q0 = a + 1 >= n ? a + 1 - n : a + 1;       // partner of atom a on diagonal 1
        int q1 = a + 2;                                // ... on diagonal 2 (mod natom)
        q1 = q1 >= n ? q1 - n : q1;
        q1 = q1 >= n ? q1 - n : q1;
        int s0 = a - 1 < 0 ? a - 1 + n : a - 1;        // the lane whose partner on diagonal dg is a
        int s1 = a - 2 < 0 ? a - 2 + n : a - 2;        // ... on diagonal dg + 1
        s0 = s0 < 0 ? s0 + n : s0;
        s1 = s1 < 0 ? s1 + n : s1;
        const int tb = tbase<TW>();
        float ax = 0.0f, ay = 0.0f, az = 0.0f, e1 = 0.0f;
#pragma unroll 1
        for (int dg = 1; dg <= nfold; dg += 2) {
            const unsigned long long m0 = uload(fm + dg - 1);
            const unsigned long long m1 = dg < nfold ? uload(fm + dg) : 0ull;
            float px0 = 0.0f, py0 = 0.0f, pz0 = 0.0f, px1 = 0.0f, py1 = 0.0f, pz1 = 0.0f;
            if (__builtin_amdgcn_inverse_ballot_w64(tmask<TW>(m0)))
                e += pair_grad(xa.x, xa.y, xa.z, xa.w, C.lut[0], lx4[q0], lfl[q0], v_cap, px0, py0, pz0);
            if (__builtin_amdgcn_inverse_ballot_w64(tmask<TW>(m1)))
                e1 += pair_grad(xa.x, xa.y, xa.z, xa.w, C.lut[0], lx4[q1], lfl[q1], v_cap, px1, py1, pz1);
            const int b0 = lane_addr(tb + s0), b1 = lane_addr(tb + s1);
            const float b0x = bperm(b0, px0), b0y = bperm(b0, py0), b0z = bperm(b0, pz0);
            const float b1x = bperm(b1, px1), b1y = bperm(b1, py1), b1z = bperm(b1, pz1);
            ax += (px0 + px1) - (b0x + b1x);
            ay += (py0 + py1) - (b0y + b1y);
            az += (pz0 + pz1) - (b0z + b1z);
            q0 = q0 + 2 >= n ? q0 + 2 - n : q0 + 2;
            q1 = q1 + 2 >= n ? q1 + 2 - n : q1 + 2;
            s0 = s0 - 2 < 0 ? s0 - 2 + n : s0 - 2;
            s1 = s1 - 2 < 0 ? s1 - 2 + n : s1 - 2;
        }
        fx[0] += ax; fy[0] += ay; fz[0] += az;
        if (C.biased()) e += bias_forces(C, P, F);
        const float r0 = row_sum(e), r1 = row_sum(e1);
        const float lo = ((rdl(r0, 0) + rdl(r0, 16)) + rdl(r1, 0)) + rdl(r1, 16);
        const float hi = ((rdl(r0, 32) + rdl(r0, 48)) + rdl(r1, 32)) + rdl(r1, 48);
        return (__lane_id() & 32) ? hi : lo;
    } else if constexpr (APL == 1) {
        // intra-molecular pairs with the per-pair curl, each pair once, in the packed steps of
        // LigSetDev::pack: a lane scores at most one pair per step, and the atoms collect their shares from
        // the wave's pair-force tile, so no LDS atomics are needed. Lanes past natom collect what is never
        // read. The next step's entry is loaded while this one is scored (a step past the last is there).
        // A step is bound by VALU issue (about 210 cycles of a SIMD) next to the LDS pipe (about 90
        // cycles of a CU with the two 16-byte coordinate reads): the entries hold LDS offsets and flag
        // constants, so that nothing is decoded or selected per pair, and twelve (nine) ds_bpermute per
        // step, at 6 cycles of the LDS pipe each, are three writes and paired reads.
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        const char* tile = reinterpret_cast<const char*>(s_lds + lx);
        const char* pk = reinterpret_cast<const char*>(C.L().pack + (size_t)C.d().pack_off * kWave);
        const int npack = C.d().npack;
        uint32_t at = uint32_t(sizeof(uint4)) * uint32_t(ln);
        uint4 t = *reinterpret_cast<const uint4*>(pk + at);
        if (n <= kWave / 2) {
            // up to 32 atoms: two folded diagonals per step, lanes 0-31 the pairs {a, (a + d) mod natom} of
            // diagonal d, lanes 32-63 those of d + 1, a the lane mod 32; lane a collects its atom's own share
            // from lane a + 32 and the partner shares of both diagonals
            const float4 xa = lx4[ln & 31];
            const uint32_t own = 4u * uint32_t((ln & 31) + 32);
#pragma unroll 1
            for (int st = 0; st < npack; st++) {
                at += uint32_t(sizeof(uint4)) * kWave;
                const uint4 tn = *reinterpret_cast<const uint4*>(pk + at);
                float px = 0.0f, py = 0.0f, pz = 0.0f;
                const float4 xj = *reinterpret_cast<const float4*>(tile + (t.x & 0xffffu));
                const float rx = xa.x - xj.x, ry = xa.y - xj.y, rz = xa.z - xj.z;
                const float rr = sq_dist(rx, ry, rz), rs = opaque(xa.w + xj.w);
                if (__uint_as_float(t.z) < kRampNoPair && rr < kR2Cut)
                    e += pair_core(rx, ry, rz, rr, rs, __uint_as_float(t.z), __uint_as_float(t.w), v_cap, px,
                                   py, pz);
                share_put(lf, ln, px, py, pz);
                const float3 o = share_get(lf, own), b0 = share_get(lf, t.y & 0xffu),
                             b1 = share_get(lf, (t.y >> 8) & 0xffu);
                ax += (px + o.x) - (b0.x + b1.x);
                ay += (py + o.y) - (b0.y + b1.y);
                az += (pz + o.z) - (b0.z + b1.z);
                t = tn;
            }
        } else {
            // 33-64 atoms: up to 63 pairs {i, j} of a step, lane l scores the one of its entry, and atom l
            // collects +p from the (at most two) lanes where it is i and -p from those where it is j; lane
            // 63 scores nothing and stands for no lane
#pragma unroll 1
            for (int st = 0; st < npack; st++) {
                at += uint32_t(sizeof(uint4)) * kWave;
                const uint4 tn = *reinterpret_cast<const uint4*>(pk + at);
                float px = 0.0f, py = 0.0f, pz = 0.0f;
                const float4 xi = *reinterpret_cast<const float4*>(tile + (t.x & 0xffffu)),
                             xj = *reinterpret_cast<const float4*>(tile + (t.x >> 16));
                const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
                // the radii with the coordinates, as 16-byte loads (12 bytes take the LDS pipe longer than 16)
                const float rr = sq_dist(rx, ry, rz), rs = opaque(xi.w + xj.w);
                if (__uint_as_float(t.z) < kRampNoPair && rr < kR2Cut)
                    e += pair_core(rx, ry, rz, rr, rs, __uint_as_float(t.z), __uint_as_float(t.w), v_cap, px,
                                   py, pz);
                share_put(lf, ln, px, py, pz);
                const float3 a0 = share_get(lf, t.y & 0xffu), a1 = share_get(lf, (t.y >> 8) & 0xffu);
                const float3 b0 = share_get(lf, (t.y >> 16) & 0xffu), b1 = share_get(lf, t.y >> 24);
                ax += (a0.x + a1.x) - (b0.x + b1.x);
                ay += (a0.y + a1.y) - (b0.y + b1.y);
                az += (a0.z + a1.z) - (b0.z + b1.z);
                t = tn;
            }
        }
        fx[0] += ax; fy[0] += ay; fz[0] += az;
        if (C.biased()) e += bias_forces(C, P, F);
        return uni(wave_sum(e));
    }
    // intra-molecular pairs with the per-pair curl, each pair once, as folded diagonals over the
    // atom slots: on diagonal d atom a scores the pair {a, (a + d) mod natom} and keeps the pair
    // gradient on itself; the partner's share is staged in the pair-force tile (one plain write per
    // atom slot, every slot written on every diagonal) and atom c reads it back from the slot of atom
    // (c - d) mod natom, so no LDS atomics are needed
    if constexpr (APL == 2) {
        // two slots: the second holds the atoms from 64 on, often few. It is scored for 4 (2) diagonals at once where
        // they fit 16 (32) lanes each, group g of the wave those of the g-th, from the coordinate tile; the
        // gradients reach the pair-force tile when their diagonal's turn comes, and their energies the
        // atoms' own lanes, so that every sum is formed in the order of the diagonals, with the bits of one slot
        // after the other. A slot of its own for each diagonal left 48-63 of 64 lanes idle in half the work of a
        // ligand of 65-80 atoms: 256 plain ligands of 10-80 atoms (58 of them past 64) 566 -> 511 ms.
        const int extra = n - kWave, gs = extra <= 16 ? 4 : extra <= 32 ? 5 : 6, per = kWave >> gs;
        const int la = ln & ((1 << gs) - 1), g = ln >> gs, a1 = kWave + la;
        const float4 x1 = lx4[a1];
        const uint32_t lut1 = uint32_t(__shfl(int(C.lut[1]), la));
        float ax0 = 0.0f, ay0 = 0.0f, az0 = 0.0f, ax1 = 0.0f, ay1 = 0.0f, az1 = 0.0f;
#pragma unroll 1
        for (int d0 = 1; d0 <= nfold; d0 += per) {
            const int cnt = nfold - d0 + 1 < per ? nfold - d0 + 1 : per;
            unsigned long long m1 = uload(fm + (d0 - 1) * 2 + 1);
            for (int i = 1; i < cnt; i++) m1 |= uload(fm + (d0 + i - 1) * 2 + 1) << (i << gs);
            float bx = 0.0f, by = 0.0f, bz = 0.0f, e1 = 0.0f;
            if (__builtin_amdgcn_inverse_ballot_w64(m1)) {
                const uint32_t q = uint32_t(a1 + d0 + g);
                const int j = int(min(q, q - uint32_t(n)));  // mod n
                e1 = pair_grad(x1.x, x1.y, x1.z, x1.w, lut1, lx4[j], lfl[j], v_cap, bx, by, bz);
            }
#pragma unroll 1
            for (int i = 0; i < cnt; i++) {
                const int dg = d0 + i;
                const unsigned long long m0 = uload(fm + (dg - 1) * 2);
                float px = 0.0f, py = 0.0f, pz = 0.0f;
                if (__builtin_amdgcn_inverse_ballot_w64(m0)) {
                    const uint32_t q = uint32_t(ln + dg);
                    const int j = int(min(q, q - uint32_t(n)));
                    e += pair_grad(P.x[0], P.y[0], P.z[0], C.rad[0], C.lut[0], lx4[j], lfl[j], v_cap, px, py, pz);
                }
                s_lds[lf + ln] = px;
                s_lds[lf + n3 + ln] = py;
                s_lds[lf + 2 * n3 + ln] = pz;
                if (g == i) {
                    s_lds[lf + a1] = bx;
                    s_lds[lf + n3 + a1] = by;
                    s_lds[lf + 2 * n3 + a1] = bz;
                }
                const float es = bperm(lane_addr(la + (i << gs)), e1);
                e += g == 0 ? es : 0.0f;
                wave_lds_fence();
                // lanes past the last atom read slots that mean nothing and collect what is never read
                const uint32_t c = uint32_t(ln - dg);
                const int src = int(min(c, c + uint32_t(n)));
                const float* f = s_lds + lf;
                ax0 = (ax0 + px) - f[src];
                ay0 = (ay0 + py) - f[n3 + src];
                az0 = (az0 + pz) - f[2 * n3 + src];
                ax1 = (ax1 + f[kWave + ln]) - f[kWave + ln - dg];
                ay1 = (ay1 + f[n3 + kWave + ln]) - f[n3 + kWave + ln - dg];
                az1 = (az1 + f[2 * n3 + kWave + ln]) - f[2 * n3 + kWave + ln - dg];
                wave_lds_fence();
            }
        }
        fx[0] += ax0; fy[0] += ay0; fz[0] += az0;
        fx[1] += ax1; fy[1] += ay1; fz[1] += az1;
    } else {
        float ax[APL], ay[APL], az[APL];
#pragma unroll
        for (int k = 0; k < APL; k++) ax[k] = ay[k] = az[k] = 0.0f;
#pragma unroll 1
        for (int dg = 1; dg <= nfold; dg++) {
#pragma unroll
            for (int k = 0; k < APL; k++) {
                const unsigned long long m = uload(fm + (dg - 1) * APL + k);
                const int a = ln + TW * k;
                float px = 0.0f, py = 0.0f, pz = 0.0f;
                if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                    const int q = a + dg < n ? a + dg : a + dg - n;
                    e += pair_grad<false>(P.x[k], P.y[k], P.z[k], C.rad[k], C.lut[k], lx4[q], lfl[q], v_cap, px, py, pz);
                }
                ax[k] += px; ay[k] += py; az[k] += pz;
                s_lds[lf + a] = px;
                s_lds[lf + n3 + a] = py;
                s_lds[lf + 2 * n3 + a] = pz;
            }
            wave_lds_fence();
#pragma unroll
            for (int k = 0; k < APL; k++) {
                const int c = ln + TW * k;
                if (c < n) {
                    const int src = c - dg >= 0 ? c - dg : c - dg + n;
                    ax[k] -= s_lds[lf + src];
                    ay[k] -= s_lds[lf + n3 + src];
                    az[k] -= s_lds[lf + 2 * n3 + src];
                }
            }
            wave_lds_fence();
        }
#pragma unroll
        for (int k = 0; k < APL; k++) {
            fx[k] += ax[k]; fy[k] += ay[k]; fz[k] += az[k];
        }
    }
    if (C.biased()) e += bias_forces(C, P, F);
    return uni(wave_sum(e));
}

// cal_grad_tile (bfgs.cuh:69-193): the pose gradient from the per-atom gradient,
// returned lane-distributed (lane k = component k).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float pose_grad(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, const Forces<APL>& F) {
    const int ln = tlane<TW>();
    const float* fx = F.fx;
    const float* fy = F.fy;
    const float* fz = F.fz;

    // gradient (cal_grad_tile, bfgs.cuh:69-193): centre = sum of heavy-atom gradients;
    // orientation from the torque about the centre (see orient_grad); torsions below.
    float sgx = 0.0f, sgy = 0.0f, sgz = 0.0f, tqx = 0.0f, tqy = 0.0f, tqz = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        if (!heavy(C, k)) continue;
        sgx += fx[k]; sgy += fy[k]; sgz += fz[k];
        const float wx = P.x[k] - P.c0, wy = P.y[k] - P.c1, wz = P.z[k] - P.c2;
        tqx += msub2(wy, fz[k], wz, fy[k]);
        tqy += msub2(wz, fx[k], wx, fz[k]);
        tqz += msub2(wx, fy[k], wy, fx[k]);
    }
    const float rg = tsum4<TW>(ln, sgx, sgy, sgz, tqx), rt = tsum4<TW>(ln, tqy, tqz, tqy, tqz);
    float gout = rg;  // lanes 0-2
    {
        const float3 og = orient_grad(P.r0, P.r1, P.r2, trdl<TW>(rg, 3), trdl<TW>(rt, 0), trdl<TW>(rt, 1));
        gout = ln == 3 ? og.x : gout;
        gout = ln == 4 ? og.y : gout;
        gout = ln == 5 ? og.z : gout;
    }
    // Torsions. Lane t forms torsion t's unit axis from the LDS coordinate tile, which still holds this pose (the
    // energy of P was the last evaluation), and stages it with the pivot and the heavy atoms it
    // rotates in the pair-force tile, idle by now; the torques about the axes are then summed four at a time. Bound by
    // VALU issue where waves are many and by the serial chain where they are few: every lane forming every
    // axis, and a wave sum and two lane selects per torsion, took 46 instructions per torsion, this 21:
    // 1,048,576 evaluations of 40 atoms and 8 torsions 4.13 -> 3.83 ms, 256 plain ligands 582 -> 566 ms.
    const float4* lx4 = reinterpret_cast<const float4*>(s_lds + C.lx());
    const int nt = C.ntors(), lt = C.lt(), lf = C.lx() + 4 * TW * APL;
    constexpr int RE = (6 + 2 * APL + 3) & ~3, CAP = 3 * TW * APL / RE;
    static_assert(CAP % 4 == 0, "whole groups of four torsions");
    unsigned long long hv[APL];
#pragma unroll
    for (int k = 0; k < APL; k++) hv[k] = tballot<TW>(heavy(C, k));
#pragma unroll 1
    for (int t0 = 0; t0 < nt; t0 += CAP) {
        const int t1 = nt < t0 + CAP ? nt : t0 + CAP;
        wave_lds_fence();
        if (ln >= t0 && ln < t1) {
            const TorsEnt te = tors_ent_at<APL>(lt, ln);
            const float4 xt = lx4[te.to], xf = lx4[te.from];
            float ux = xt.x - xf.x, uy = xt.y - xf.y, uz = xt.z - xf.z;
            const float inv = frsq(sq_dist(ux, uy, uz));
            ux *= inv; uy *= inv; uz *= inv;
            float* r = s_lds + lf + (ln - t0) * RE;
            *reinterpret_cast<float4*>(r) = make_float4(ux, uy, uz, xt.x);
            r[4] = xt.y;
            r[5] = xt.z;
#pragma unroll
            for (int k = 0; k < APL; k++) {
                const unsigned long long m = tors_mask_at<APL>(lt, ln, k) & hv[k];
                r[6 + 2 * k] = __uint_as_float(uint32_t(m));
                r[7 + 2 * k] = __uint_as_float(uint32_t(m >> 32));
            }
        }
        wave_lds_fence();
        // this lane's part of the torque about the axis of record i; past the last torsion whatever the tile
        // holds, which ends up on lanes past the gradient
        const auto torque = [&](int i) {
            const float* r = s_lds + lf + i * RE;
            const float4 u = *reinterpret_cast<const float4*>(r), w = *reinterpret_cast<const float4*>(r + 4);
            float st = 0.0f;
#pragma unroll
            for (int k = 0; k < APL; k++) {
                const uint32_t lo = __builtin_amdgcn_readfirstlane(__float_as_uint(k == 0 ? w.z : r[6 + 2 * k]));
                const uint32_t hi = __builtin_amdgcn_readfirstlane(__float_as_uint(k == 0 ? w.w : r[7 + 2 * k]));
                const float lx = P.x[k] - u.w, ly = P.y[k] - w.x, lz = P.z[k] - w.y;
                const float cx = msub2(ly, fz[k], lz, fy[k]), cy = msub2(lz, fx[k], lx, fz[k]),
                            cz = msub2(lx, fy[k], ly, fx[k]);
                const float q = madd3(cx, u.x, cy, u.y, cz, u.z);
                const bool in = __builtin_amdgcn_inverse_ballot_w64(tmask<TW>((unsigned long long)lo | ((unsigned long long)hi << 32)));
                st = in ? st + q : st;
            }
            return st;
        };
#pragma unroll 1
        for (int t = t0; t < t1; t += 4) {
            // torsion t + i belongs on lane 6 + t + i, which takes value (i + 2) mod 4 of a sum of four
            const float s0 = torque(t - t0), s1 = torque(t - t0 + 1);
            float s2 = 0.0f, s3 = 0.0f;
            if (t + 2 < t1) {
                s2 = torque(t - t0 + 2);
                s3 = torque(t - t0 + 3);
            }
            const float v = tsum4<TW>(ln, s2, s3, s0, s1);
            gout = ln >= 6 + t ? v : gout;
        }
        wave_lds_fence();
    }
    gout = ln < 6 + nt ? gout : 0.0f;
    // constraint docking (bfgs.cuh:176): the rigid components are never written and
    // keep the zeros the reference's gradient buffers start with
    if (C.L().constraint && ln < 6) gout = 0.0f;
    return gout;
}

// cal_e_grad_tile (bfgs.cuh:397-410).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float energy_grad(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, float v_cap, float slope,
                                             float& g) {
    Forces<APL> F;
    const float e = energy_forces(C, P, v_cap, slope, F);
    g = pose_grad(C, P, F);
    return e;
}

// A lower bound of energy_forces' value at P without the bias terms, for any curl cap: the box penalty
// of the heavy atoms as energy_forces sums it, less the largest attraction any heavy atom can feel from
// the receptor (every receptor heavy atom at its most attractive distance: the gauss, hydrophobic and
// hydrogen-bond terms together stay below 0.67 kcal/mol per pair, and a grid value interpolates such
// sums) and any intra pair can add (the curl only shrinks repulsion).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float energy_lower_bound(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P, float slope) {
    SceneArg& S = C.S();
    float pen = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        if (!heavy(C, k)) continue;
        pen += fmaxf(S.box_lo[0] - P.x[k], 0.0f) + fmaxf(P.x[k] - S.box_hi[0], 0.0f);
        pen += fmaxf(S.box_lo[1] - P.y[k], 0.0f) + fmaxf(P.y[k] - S.box_hi[1], 0.0f);
        pen += fmaxf(S.box_lo[2] - P.z[k], 0.0f) + fmaxf(P.z[k] - S.box_hi[2], 0.0f);
    }
    return tuni<TW>(tsum<TW>(pen) * slope - 0.67f * (float(S.nrec) * float(C.nheavy()) + float(C.npair())));
}

// How many waves run a chain. Solo: one. Team: the four of a block, each with the chain's whole state in its own
// registers and LDS slice and computing the same bits, so that they take the same branches; a line search
// evaluates four trial steps at a time, one per wave, and every wave goes on with the one the sequential
// search would have ended on. sh: the block's shared area in LDS (floats).
struct Solo {};
struct Team {
    int wave, sh;      // team_floats(APL) at sh: two sets of codes, the queue item, then a pose, its gradient and energy
    mutable int flip;  // which of the two sets of trial codes the next round uses
};
// Trial codes: how a trial of the line search ended.
constexpr int kTrialRejected = 0, kTrialScreened = 1, kTrialTaken = 2, kTrialNotFinite = 3, kTrialLast = 4;
constexpr int kTrials = 10;

// line_search_tile (bfgs.cuh:623-670). A trial whose energy is certain to fail the sufficient-decrease
// test is not evaluated: when the gradient is dominated by the box penalty (p . g below -1e4, a pose
// partly outside the box at slope 1e6), the trial pose's penalty alone can exceed the test's bound by
// far, and such a trial is rejected from energy_lower_bound (with a margin of 1e-4 of the magnitudes
// involved, far above the rounding of either side). The trials, their steps and the pose the search ends
// on are the same as with every trial evaluated; the last trial is always evaluated, since its energy and
// forces are the search's result.
// The search fails, returning false with x_new = x, g_new = g, e_out = e0 and alpha 0, on a direction
// with a non-finite p . g or at a trial pose with a non-finite coordinate. Both come from a search that
// has walked a pose some 1e7 A or more out of the box (after a negative step-0 diagonal rescale, say),
// where FP32 rounds bonded atoms onto one point: a torsion axis of zero length turns its gradient and
// its rotated atoms into NaN. The reference searches on, and can keep a pose of NaN coordinates, which
// every energy term skips (their comparisons fail), so it scores finite; hydrogens are never scored.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ bool pose_finite(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P) {
    bool bad = false;
#pragma unroll
    for (int k = 0; k < APL; k++)
        bad |= C.type[k] >= 0 &&
               !(__builtin_isfinite(P.x[k]) && __builtin_isfinite(P.y[k]) && __builtin_isfinite(P.z[k]));
    return tballot<TW>(bad) == 0ull;
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ bool line_search(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& x, float g, float p, float e0, float v_cap,
                            float slope, WPose<APL>& x_new, float& g_new, float& e_out, float& alpha_out,
                            const Solo& = Solo()) {
    const float pg = tuni<TW>(tsum<TW>(p * g));
    const auto fail = [&]() {
        x_new = x;
        g_new = g;
        e_out = e0;
        alpha_out = 0.0f;
        return false;
    };
    if (!__builtin_isfinite(pg)) return fail();
    const bool screen = pg < -1e4f && !(C.biased());
    float alpha = 1.0f, e_new = 0.0f;
    Forces<APL> F;
    for (int trial = 0; trial < 10; trial++) {
        x_new = x;
        apply_update(C, x_new, p, alpha);
        if (!pose_finite(C, x_new)) return fail();
        if (screen && trial < 9) {
            const float bound = 1e-4f * alpha * pg;
            const float lb = energy_lower_bound(C, x_new, slope);
            if ((lb - e0) - bound > 1e-4f * (fabsf(lb) + fabsf(e0) + fabsf(bound)) + 1.0f) {
                alpha *= 0.5f;
                continue;
            }
        }
        e_new = energy_forces(C, x_new, v_cap, slope, F);
        if (e_new - e0 < 1e-4f * alpha * pg) break;
        alpha *= 0.5f;
    }
    // only the gradient of the trial the search ends on is ever used (bfgs.cuh:641-667)
    g_new = pose_grad(C, x_new, F);
    e_out = e_new;
    alpha_out = alpha;
    return true;
}

// line_search by a team. The trials of a round are independent; what is counted as evaluated is what the sequential
// search evaluates.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ bool line_search(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& x, float g, float p, float e0,
                                            float v_cap, float slope, WPose<APL>& x_new, float& g_new, float& e_out,
                                            float& alpha_out, const Team& T) {
    static_assert(TW == kWave, "a team's chain takes whole waves");
    const int ln = tlane<TW>();
    const float pg = uni(wave_sum(p * g));
    const int ev0 = C.evals;
    int ev = 0, first = 0, code = 0, winner = 0;
    float e_new = 0.0f;
    Forces<APL> F;
    bool failed = !__builtin_isfinite(pg);
    if (!failed) {
        const bool screen = pg < -1e4f && !C.biased();
        for (; ; first += kWavesPerBlock) {
            const int trial = first + T.wave;
            int mine = kTrialScreened;  // past the last trial: never looked at
            if (trial < kTrials) {
                const float alpha = __uint_as_float(uint32_t(127 - trial) << 23);  // 2^-trial
                x_new = x;
                apply_update(C, x_new, p, alpha);
                bool skip = false;
                if (!pose_finite(C, x_new)) {
                    mine = kTrialNotFinite;
                } else {
                    if (screen && trial < kTrials - 1) {
                        const float bound = 1e-4f * alpha * pg;
                        const float lb = energy_lower_bound(C, x_new, slope);
                        skip = (lb - e0) - bound > 1e-4f * (fabsf(lb) + fabsf(e0) + fabsf(bound)) + 1.0f;
                    }
                    if (!skip) {
                        e_new = energy_forces(C, x_new, v_cap, slope, F);
                        mine = e_new - e0 < 1e-4f * alpha * pg ? kTrialTaken
                               : trial == kTrials - 1          ? kTrialLast
                                                               : kTrialRejected;
                    }
                }
            }
            int* codes = reinterpret_cast<int*>(s_lds + T.sh) + kWavesPerBlock * T.flip;
            T.flip ^= 1;
            if (ln == 0) codes[T.wave] = mine;
            __syncthreads();
            winner = -1;
#pragma unroll
            for (int w = 0; w < kWavesPerBlock; w++) {
                const int c = __builtin_amdgcn_readfirstlane(codes[w]);
                if (winner < 0) {
                    ev += c != kTrialScreened && c != kTrialNotFinite;
                    if (c >= kTrialTaken) {
                        winner = w;
                        code = c;
                    }
                }
            }
            if (winner >= 0) break;
        }
        failed = code == kTrialNotFinite;
    }
    C.evals = ev0 + ev;
    if (failed) {
        x_new = x;
        g_new = g;
        e_out = e0;
        alpha_out = 0.0f;
        return false;
    }
    float* s = s_lds + T.sh + 12;
    if (T.wave == winner) {
        g_new = pose_grad(C, x_new, F);
#pragma unroll
        for (int k = 0; k < APL; k++) {
            s[(3 * k) * kWave + ln] = x_new.x[k];
            s[(3 * k + 1) * kWave + ln] = x_new.y[k];
            s[(3 * k + 2) * kWave + ln] = x_new.z[k];
        }
        s[3 * APL * kWave + ln] = x_new.dihe;
        s[(3 * APL + 1) * kWave + ln] = g_new;
        float* u = s + (3 * APL + 2) * kWave;
        if (ln == 0) {
            u[0] = x_new.c0; u[1] = x_new.c1; u[2] = x_new.c2;
            u[3] = x_new.r0; u[4] = x_new.r1; u[5] = x_new.r2;
            u[6] = e_new;
        }
    }
    __syncthreads();
    if (T.wave != winner) {
#pragma unroll
        for (int k = 0; k < APL; k++) {
            x_new.x[k] = s[(3 * k) * kWave + ln];
            x_new.y[k] = s[(3 * k + 1) * kWave + ln];
            x_new.z[k] = s[(3 * k + 2) * kWave + ln];
        }
        x_new.dihe = s[3 * APL * kWave + ln];
        g_new = s[(3 * APL + 1) * kWave + ln];
        const float* u = s + (3 * APL + 2) * kWave;
        x_new.c0 = uni(u[0]); x_new.c1 = uni(u[1]); x_new.c2 = uni(u[2]);
        x_new.r0 = uni(u[3]); x_new.r1 = uni(u[4]); x_new.r2 = uni(u[5]);
        x_new.e = x.e;
        e_new = uni(u[6]);
    }
    const int taken = first + winner;
    e_out = e_new;
    // after the last trial failed, the step is halved once more
    alpha_out = __uint_as_float(uint32_t(127 - taken - (code == kTrialLast ? 1 : 0)) << 23);
    return true;
}

__device__ __forceinline__ int row_lane_clamped(int ln, int dim) { return ln < dim ? ln : dim - 1; }

// A lane-distributed vector (component k on lane k) written to LDS at offset o, for broadcast reads.
template <int TW>
__device__ __forceinline__ void stage_vec(int o, float v) { s_lds[o + tlane<TW>()] = v; }

// Row of the inverse Hessian (at LDS offset hrow) times the vector staged at LDS offset vo, over dim
// components: four columns per pass with independent partial sums, the vector's four components by
// one broadcast load, so the reads are in flight together. Every lane reads a real row (callers mask
// lanes past dim).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float hess_row_dot(const Ctx<APL, TW, LAZY>& C, int hrow, int dim, int vo) {
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    int j = 0;
    for (; j + 4 <= dim; j += 4) {
        const float4 v = *reinterpret_cast<const float4*>(s_lds + vo + j);
        const float* h = s_lds + hrow + j;
        s0 += h[0] * v.x;
        s1 += h[1] * v.y;
        s2 += h[2] * v.z;
        s3 += h[3] * v.w;
    }
    for (; j < dim; j++) s0 += s_lds[hrow + j] * s_lds[vo + j];
    return (s0 + s1) + (s2 + s3);
}

// bfgs_tile (bfgs.cuh:729-829): the inverse Hessian lives in the wave's LDS
// tile (lane i owns row i) and the start pose is parked in LDS for the
// restore at the end (the energy went up, or a line search failed). The vectors the Hessian products read (g, y, p, -Hy) are staged in
// the coordinate tile, idle between a line search and the next one.
template <int APL, int TW, bool LAZY, class Crew = Solo>
__device__ __forceinline__ void bfgs(const Ctx<APL, TW, LAZY>& C, WPose<APL>& x, int max_steps, float v_cap, float slope,
                                     const Crew& crew = Crew()) {
    float g;
    const float E_ori = energy_grad(C, x, v_cap, slope, g);
    float E = E_ori, E1 = 0.0f, alpha = 0.0f;
    {
        const int ln = tlane<TW>(), dim = C.dim(), hrow = C.lh() + ln * C.ld;
        if (ln < dim)
            for (int j = 0; j < dim; j++) s_lds[hrow + j] = (j == ln) ? 1.0f : 0.0f;
    }
    float g_new = g;
    WPose<APL> x_new = x;
    save_pose(C, x);
    float p = g;
    bool failed = false;
    for (int step = 0; step < max_steps; step++) {
        // rows beyond dim are masked: their lanes read the last row
        {
            const int ln = tlane<TW>(), dim = C.dim(), v0 = C.lx();
            stage_vec<TW>(v0, g);
            wave_lds_fence();
            const float s = hess_row_dot(C, C.lh() + row_lane_clamped(ln, dim) * C.ld, dim, v0);
            p = ln < dim ? -s : 0.0f;
            wave_lds_fence();
        }
        if (!line_search(C, x, g, p, E, v_cap, slope, x_new, g_new, E1, alpha, crew)) {
            failed = true;
            break;
        }
        const float y = g_new - g;
        E = E1;
        x = x_new;
        const float gg = tsum<TW>(g * g);
        if (sqrtf(gg) < 1e-5f) break;
        g = g_new;
        const int ln = tlane<TW>(), dim = C.dim(), hrow = C.lh() + ln * C.ld;
        const int v0 = C.lx(), vp = v0 + TW, vm = v0 + 2 * TW;
        const bool row = ln < dim;
        if (step == 0) {
            const float yy = tuni<TW>(tsum<TW>(y * y));
            if (fabsf(yy) > kEps) {
                const float yp0 = tsum<TW>(y * p);
                if (row) s_lds[hrow + ln] = alpha * yp0 / yy;
            }
        }
        const float yp = tuni<TW>(tsum<TW>(y * p));
        if (alpha * yp < kEps) continue;
        stage_vec<TW>(v0, y);
        wave_lds_fence();
        const float hy = hess_row_dot(C, C.lh() + row_lane_clamped(ln, dim) * C.ld, dim, v0);
        const float mhy = row ? -hy : 0.0f;
        const float yhy = -tsum<TW>(y * mhy);
        const float r = 1.0f / (alpha * yp);
        const float a1 = tuni<TW>(alpha * r), a2 = tuni<TW>(alpha * alpha * fmaf_(r * r, yhy, r));
        const float a2p = a2 * p;
        stage_vec<TW>(vp, p);
        stage_vec<TW>(vm, mhy);
        wave_lds_fence();
        // four columns per pass: their reads are in flight together
        int j = 0;
        for (; j + 4 <= dim; j += 4) {
            const float4 pj = *reinterpret_cast<const float4*>(s_lds + vp + j);
            const float4 mj = *reinterpret_cast<const float4*>(s_lds + vm + j);
            if (row) {
                float* h = s_lds + hrow + j;
                const float h0 = h[0], h1 = h[1], h2 = h[2], h3 = h[3];
                h[0] = h0 + madd2(a1, madd2(mhy, pj.x, mj.x, p), a2p, pj.x);
                h[1] = h1 + madd2(a1, madd2(mhy, pj.y, mj.y, p), a2p, pj.y);
                h[2] = h2 + madd2(a1, madd2(mhy, pj.z, mj.z, p), a2p, pj.z);
                h[3] = h3 + madd2(a1, madd2(mhy, pj.w, mj.w, p), a2p, pj.w);
            }
        }
        for (; j < dim; j++) {
            const float pj = s_lds[vp + j], mj = s_lds[vm + j];
            if (row) s_lds[hrow + j] += madd2(a1, madd2(mhy, pj, mj, p), a2p, pj);
        }
        wave_lds_fence();
    }
    if (failed || E > E_ori) {  // a failed line search: the start pose, as when the energy went up
        restore_pose(C, x);
        E = E_ori;
    }
    x.e = tuni<TW>(E);
}

// ------------------------------------------------------------------ RNG
// Philox4x32-10 (Salmon et al., SC'11); the stream of a chain is keyed by
// (seed, ligand index) with counter (chain, draw, 0x55443244, 0).
__device__ __forceinline__ uint4 philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const uint32_t hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return make_uint4(c0, c1, c2, c3);
}

__device__ __forceinline__ float u01(uint32_t u) { return float((u >> 8) + 1u) * (1.0f / 16777216.0f); }

struct Rng {
    uint32_t k0, k1, chain, draw;
    __device__ uint4 next() { return philox(chain, draw++, 0x55443244u, 0u, k0, k1); }
    __device__ uint4 at(uint32_t d) const { return philox(chain, d, 0x55443244u, 0u, k0, k1); }
};

// gen_4_rand_in_sphere (E/src/cuda/common.cuh:90-103); the acceptance test is
// evaluated with rounded (uncontracted) float operations.
__device__ __forceinline__ float3 rand_in_ball(Rng& rng) {
    for (;;) {
        const uint4 b = rng.next();
        const float a0 = (u01(b.x) - 0.5f) * 2.0f, a1 = (u01(b.y) - 0.5f) * 2.0f, a2 = (u01(b.z) - 0.5f) * 2.0f;
        const float r2 = __fadd_rn(__fadd_rn(__fmul_rn(a0, a0), __fmul_rn(a1, a1)), __fmul_rn(a2, a2));
        if (r2 < 1.0f) return make_float3(a0, a1, a2);
    }
}

// gyration_radius (common.cuh:106-122).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ float gyration(const Ctx<APL, TW, LAZY>& C, const WPose<APL>& P) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++)
        if (heavy(C, k)) {
            const float dx = P.x[k] - P.c0, dy = P.y[k] - P.c1, dz = P.z[k] - P.c2;
            s += sq_dist(dx, dy, dz);
        }
    s = tsum<TW>(s);
    const float r = C.nheavy() > 0 ? sqrtf(s / float(C.nheavy())) : 0.0f;
    return tuni<TW>(r > 0.0f ? r : 1.0f);
}

// What a mutation did: kind 0 translation, 1 rotation, 2 torsion; magnitude
// |d| / 2 A, rotation angle / pi or |torsion change| / pi; moved = fraction of
// heavy atoms displaced. The plain MC ignores it; the learned proposal feeds it
// to its network.
struct Move {
    int kind;
    float mag, moved;
};

// mutate_pose_tile (E/src/cuda/mc.cu:146-256).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ Move mutate(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, Rng& rng) {
    SceneArg& S = C.S();
    const uint4 b = rng.next();
    // constraint docking draws a torsion only; a rigid ligand then stays put (mc.cu:159-166)
    int which;
    if (C.L().constraint) which = C.ntors() > 0 ? 2 + int(b.x % uint32_t(C.ntors())) : -1;
    else which = int(b.x % uint32_t(2 + C.ntors()));
    Move mv;
    if (which < 0) {
        mv.kind = 2;
        mv.mag = 0.0f;
        mv.moved = 0.0f;
    } else if (which == 0) {
        const float3 a = rand_in_ball(rng);
        const float d0 = tuni<TW>(fminf(fmaxf(2.0f * a.x + P.c0, S.box_lo[0]), S.box_hi[0]) - P.c0);
        const float d1 = tuni<TW>(fminf(fmaxf(2.0f * a.y + P.c1, S.box_lo[1]), S.box_hi[1]) - P.c1);
        const float d2 = tuni<TW>(fminf(fmaxf(2.0f * a.z + P.c2, S.box_lo[2]), S.box_hi[2]) - P.c2);
        P.c0 = tuni<TW>(P.c0 + d0); P.c1 = tuni<TW>(P.c1 + d1); P.c2 = tuni<TW>(P.c2 + d2);
#pragma unroll
        for (int k = 0; k < APL; k++)
            if (valid(C, k)) { P.x[k] += d0; P.y[k] += d1; P.z[k] += d2; }
        mv.kind = 0;
        mv.mag = 0.5f * sqrtf(sq_dist(d0, d1, d2));
        mv.moved = 1.0f;
    } else if (which == 1) {
        const float3 a = rand_in_ball(rng);
        const float gr = gyration(C, P);
        const float v0 = tuni<TW>(2.0f / gr * a.x), v1 = tuni<TW>(2.0f / gr * a.y), v2 = tuni<TW>(2.0f / gr * a.z);
        const float4 q = rotvec_to_quat(v0, v1, v2);
        P.r0 = v0; P.r1 = v1; P.r2 = v2;
        rigid_move(C, P, q, P.c0, P.c1, P.c2, P.c0, P.c1, P.c2);
        mv.kind = 1;
        mv.mag = sqrtf(sq_dist(v0, v1, v2)) * (1.0f / kPi);
        mv.moved = 1.0f;
    } else {
        const int t = which - 2;
        const uint4 bb = rng.next();
        const TorsEnt te = tors_ent(C, t);
        int i = int(ceilf(__fsub_rn(__fmul_rn(u01(bb.x), float(te.nrange)), 1.0f)));
        i = i < 0 ? 0 : (i > te.nrange - 1 ? te.nrange - 1 : i);
        float2 r = make_float2(te.lo, te.hi);
        if (i > 0) r = C.L().ranges[C.L().tors_range[C.d().tors_off + t].x + i];
        const float target = r.x + (r.y - r.x) * u01(bb.y);
        const float inc = target - tread<TW>(P.dihe, t);
        apply_torsion(C, P, t, inc);
        centroid(C, P);
        int nmoved = 0;
#pragma unroll
        for (int k = 0; k < APL; k++) nmoved += __popcll(tors_mask(C, t, k) & tballot<TW>(heavy(C, k)));
        mv.kind = 2;
        mv.mag = fabsf(normalize_angle(inc)) * (1.0f / kPi);
        mv.moved = C.nheavy() > 0 ? float(nmoved) / float(C.nheavy()) : 0.0f;
    }
    return mv;
}

// randomize_pose_tile (mc.cu:18-104): centre drawn in the box, super-Fibonacci
// orientation by chain index, each torsion drawn in a random allowed range;
// applied through apply_update with alpha = 1. Constraint docking keeps centre
// and orientation (:27-35), the align bias keeps the centre (:36-39); the centre
// block is drawn either way.
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void randomize(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P, Rng& rng, int idx, int n) {
    SceneArg& S = C.S();
    const int ln = tlane<TW>();
    const uint4 b = rng.next();
    const float gc0 = (S.box_lo[0] + (S.box_hi[0] - S.box_lo[0]) * u01(b.x)) - P.c0;
    const float gc1 = (S.box_lo[1] + (S.box_hi[1] - S.box_lo[1]) * u01(b.y)) - P.c1;
    const float gc2 = (S.box_lo[2] + (S.box_hi[2] - S.box_lo[2]) * u01(b.z)) - P.c2;
    // super-Fibonacci sample idx of n (Alexa, CVPR'22): angles 2 pi s / phi and
    // 2 pi s / psi, reduced to one turn before the hardware sin / cos
    const float s = float(idx) + 0.5f;
    const float r = fsqrt(s / float(n)), R = fsqrt(1.0f - s / float(n));
    const float fa = s * (1.0f / 1.4142135623730951f), fb = s * (1.0f / 1.5337511687552043f);
    float sa, ca, sb, cb;
    __sincosf(2.0f * kPi * (fa - floorf(fa)), &sa, &ca);
    __sincosf(2.0f * kPi * (fb - floorf(fb)), &sb, &cb);
    const float3 rv = quat_to_rotvec(make_float4(r * sa, r * ca, R * sb, R * cb));
    // torsion t draws block (draw + t) on lane t: a range, then a value in it
    float tv = 0.0f;
    if (ln < C.ntors()) {
        const uint4 bt = rng.at(rng.draw + ln);
        const int2 rr = C.L().tors_range[C.d().tors_off + ln];
        int j = int(__fmul_rn(u01(bt.x), float(rr.y)));
        j = j > rr.y - 1 ? rr.y - 1 : j;
        const float2 rg = C.L().ranges[rr.x + j];
        tv = (rg.x + (rg.y - rg.x) * u01(bt.y)) - P.dihe;
    }
    rng.draw += C.ntors();
    // direction vector: lanes 0..5 rigid part, lane 6 + t torsion t
    const float sh = tshfl<TW>(tv, ln - 6);
    float d = (ln >= 6 && ln < 6 + C.ntors()) ? sh : 0.0f;
    const bool keep_c = C.L().constraint || C.L().bias_type == 2, keep_o = C.L().constraint;
    d = ln == 0 ? (keep_c ? 0.0f : gc0) : d;
    d = ln == 1 ? (keep_c ? 0.0f : gc1) : d;
    d = ln == 2 ? (keep_c ? 0.0f : gc2) : d;
    d = ln == 3 ? (keep_o ? 0.0f : rv.x) : d;
    d = ln == 4 ? (keep_o ? 0.0f : rv.y) : d;
    d = ln == 5 ? (keep_o ? 0.0f : rv.z) : d;
    apply_update(C, P, d, 1.0f);
}

// ---------------------------------------------------------- pose buffers
template <int APL>
__device__ __forceinline__ void load_pose(const Ctx<APL>& C, Karg<PoseBufs>& B, int lig, int chain, WPose<APL>& P) {
    KLig& d = C.d();
    const int natom = d.natom, ntors = d.ntors, nchain = B.nchain;
    const size_t xo = ((size_t)d.atom_off * nchain + (size_t)chain * natom) * 3;
    const size_t po = (size_t)lig * nchain + chain;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = lane() + kWave * k;
        if (a < natom) { P.x[k] = B.x[xo + 3 * a]; P.y[k] = B.x[xo + 3 * a + 1]; P.z[k] = B.x[xo + 3 * a + 2]; }
        else { P.x[k] = P.y[k] = P.z[k] = 0.0f; }
    }
    P.c0 = B.c[po * 3]; P.c1 = B.c[po * 3 + 1]; P.c2 = B.c[po * 3 + 2];
    P.r0 = B.rv[po * 3]; P.r1 = B.rv[po * 3 + 1]; P.r2 = B.rv[po * 3 + 2];
    const size_t dof = (size_t)d.tors_off * nchain + (size_t)chain * ntors;
    P.dihe = lane() < ntors ? B.dihe[dof + lane()] : 0.0f;
    P.e = B.e[po];
}

template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void store_pose(const Ctx<APL, TW, LAZY>& C, Karg<PoseBufs>& B, int lig, int chain,
                                           const WPose<APL>& P) {
    KLig& d = C.d();
    const int natom = d.natom, ntors = d.ntors, nchain = B.nchain;
    const size_t xo = ((size_t)d.atom_off * nchain + (size_t)chain * natom) * 3;
    const size_t po = (size_t)lig * nchain + chain;
    const int ln = tlane<TW>();
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = ln + TW * k;
        if (a < natom) { B.x[xo + 3 * a] = P.x[k]; B.x[xo + 3 * a + 1] = P.y[k]; B.x[xo + 3 * a + 2] = P.z[k]; }
    }
    if (ln == 0) { B.c[po * 3] = P.c0; B.rv[po * 3] = P.r0; B.e[po] = P.e; }
    if (ln == 1) { B.c[po * 3 + 1] = P.c1; B.rv[po * 3 + 1] = P.r1; }
    if (ln == 2) { B.c[po * 3 + 2] = P.c2; B.rv[po * 3 + 2] = P.r2; }
    const size_t dof = (size_t)d.tors_off * nchain + (size_t)chain * ntors;
    if (ln < ntors) B.dihe[dof + ln] = P.dihe;
}

// Input conformation of a ligand: coordinates, dihedrals, centroid, rot_vec = 0,
// energy 999 (E/src/cuda/task.cu:94-108).
template <int APL, int TW, bool LAZY>
__device__ __forceinline__ void initial_pose(const Ctx<APL, TW, LAZY>& C, WPose<APL>& P) {
    KLig& d = C.d();
    LigArg& L = C.L();
    const int ln = tlane<TW>();
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = ln + TW * k;
        if (a < d.natom) { const float4 v = L.atom_x0[d.atom_off + a]; P.x[k] = v.x; P.y[k] = v.y; P.z[k] = v.z; }
        else { P.x[k] = P.y[k] = P.z[k] = 0.0f; }
    }
    P.dihe = ln < d.ntors ? L.tors_dihe0[d.tors_off + ln] : 0.0f;
    centroid(C, P);
    P.r0 = P.r1 = P.r2 = 0.0f;
    P.e = 999.0f;
}

}  // namespace ud2
