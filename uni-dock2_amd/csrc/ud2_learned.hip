// Learned-proposal Monte Carlo search (no reference counterpart; the plain
// search is mc_kernel, after E/src/cuda/mc.cu:275-398).
//
// lmc_kernel is persistent like mc_kernel: each wave takes (ligand, chain)
// items from a size-sorted queue and runs the whole chain with its state in
// registers and LDS. One MC step, by policy:
//   plain    one random mutation (the reference's step);
//   exact    n_cand mutations all scored with the exact search energy, the
//            best one kept;
//   learned  n_cand mutations described by 80 pooled grid-map features each
//            (bf16 rows in LDS), scored together by the network on MFMA
//            (one 16-candidate group per wave), the top_k rescored exactly and
//            the best kept;
//   collect  n_cand mutations whose features and BFGS-refined energies are
//            written out as training data; the chain continues with
//            candidate 0, i.e. the plain trajectory.
// The kept candidate is BFGS-refined and goes through the reference's
// Metropolis test (mc.cu:340-392). A candidate is identified by the Philox
// block where its mutation starts, so rebuilding it replays the same draws.
// While candidates are drawn and scored, the LDS that the energy and BFGS use
// is idle: the candidate rows take the coordinate / force / BFGS-start area
// and the feature scratch and the network's hidden layer take the Hessian's.
#include "ud2_device.h"
#include "ud2_mlp.h"

namespace ud2 {

// Feature class of each XS type (E/src/constants/constants.h:48-68); -1 = hydrogen.
static __constant__ int c_fclass[kNumTypes] = {-1, 1, 0, 1, 2, 3, 4, 3, 5, 6, 5, 6, 0, 1, 7, 7, 0, 0, 0, 0, 7};

// Features of pose P (80 bf16 into xrow). Per heavy atom: its own map's value e
// and gradient g at its position, statistics [1, min(e,0), clamp(e,0,1),
// log1p(max(e,0)), e < -0.3, min(box overshoot,4), min(|g|,8)(e<=0),
// min(|g|,8)(e>0)] pooled by feature class into xrow[8 class + stat]; move
// globals in xrow[64..79]. The per-atom rows go through the LDS scratch at
// `sc` (8 floats per atom) and lane j sums feature j.
template <int APL>
__device__ __forceinline__ void pose_features(const Ctx<APL>& C, const WPose<APL>& P, const Move& mv, float e_acc, int sc,
                              uint16_t* xrow) {
    SceneArg& S = C.S();
    const int ln = tlane<kWave>(), natom = C.natom();
    float curl = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = ln + kWave * k;
        float cls = -1.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f, p4 = 0.0f, p5 = 0.0f, p6 = 0.0f, p7 = 0.0f;
        if (heavy(C, k)) {
            const int t = C.type[k];
            const int slot = S.slot_tab[t];
            float gx = 0.0f, gy = 0.0f, gz = 0.0f, e = 0.0f;
            if (slot >= 0) e = grid_eval(S, slot, P.x[k], P.y[k], P.z[k], gx, gy, gz);
            const float over = fmaxf(S.box_lo[0] - P.x[k], 0.0f) + fmaxf(P.x[k] - S.box_hi[0], 0.0f) +
                               fmaxf(S.box_lo[1] - P.y[k], 0.0f) + fmaxf(P.y[k] - S.box_hi[1], 0.0f) +
                               fmaxf(S.box_lo[2] - P.z[k], 0.0f) + fmaxf(P.z[k] - S.box_hi[2], 0.0f);
            const float gc = fminf(sqrtf(gx * gx + gy * gy + gz * gz), 8.0f);
            const float ep = fmaxf(e, 0.0f);
            cls = float(c_fclass[t]);
            p1 = fminf(e, 0.0f);
            p2 = fminf(ep, 1.0f);
            p3 = log1pf(fminf(ep, 1e30f));
            p4 = e < -0.3f ? 1.0f : 0.0f;
            p5 = fminf(over, 4.0f);
            p6 = e <= 0.0f ? gc : 0.0f;
            p7 = e > 0.0f ? gc : 0.0f;
            curl += e > 0.0f ? e / (1.0f + e) : e;
        }
        if (a < natom) {
            float* r = s_lds + sc + 8 * a;
            r[0] = cls; r[1] = p1; r[2] = p2; r[3] = p3; r[4] = p4; r[5] = p5; r[6] = p6; r[7] = p7;
        }
    }
    wave_lds_fence();
    const float my_cls = float(ln >> 3);
    const int st = ln & 7;
    float f = 0.0f;
#pragma unroll 4
    for (int a = 0; a < natom; a++) {
        const float c = s_lds[sc + 8 * a];
        const float v = st == 0 ? 1.0f : s_lds[sc + 8 * a + st];
        f += c == my_cls ? v : 0.0f;
    }
    xrow[ln] = f2bf(f);
    curl = wave_sum(curl);
    if (ln < 16) {
        float g = 0.0f;
        if (ln == 0) g = mv.kind == 0 ? 1.0f : 0.0f;
        if (ln == 1) g = mv.kind == 1 ? 1.0f : 0.0f;
        if (ln == 2) g = mv.kind == 2 ? 1.0f : 0.0f;
        if (ln == 3) g = mv.mag;
        if (ln == 4) g = float(C.nheavy()) / 64.0f;
        if (ln == 5) g = float(C.ntors()) / 16.0f;
        if (ln == 6) g = fminf(fmaxf(e_acc, -20.0f), 20.0f) / 10.0f;
        if (ln == 7) g = mv.moved;
        if (ln == 8) g = fminf(fmaxf(curl, -20.0f), 20.0f) / 10.0f;
        xrow[kPooled + ln] = f2bf(g);
    }
    wave_lds_fence();
}

__device__ __forceinline__ MlpDev network(Karg<MlpDev>& w) {
    MlpDev W;
    W.w1 = w.w1; W.w1s = w.w1s; W.w2t = w.w2t; W.w2s = w.w2s; W.w2 = w.w2;
    W.b1 = w.b1; W.b2 = w.b2; W.w3 = w.w3; W.b3 = w.b3;
    W.mu = w.mu; W.inv_sigma = w.inv_sigma;
    return W;
}

// Persistent learned-proposal MC kernel. One-atom-per-lane ligands fit six
// waves per SIMD in LDS when at most 8 candidates are scored per group (8 hidden
// rows staged, partly in the slice's idle coordinate / force / BFGS-start area;
// 16 rows of ligands with 15 torsions need 832 B per block more than a quarter
// of the CU's 160 KB, and run three waves per SIMD); the occupancy hint holds
// the register allocation to the 80 VGPRs that six waves allow, which measured
// 6 % faster than four waves at 128 VGPRs despite the spills, and four waves faster
// than three; at six it is bound by VALU issue (1.04 of the FMA probe's rate). POL >= 0 compiles one
// policy only, on grid maps (the learned search); POL = -1 takes policy and inter term from the arguments. Wider ligands run at
// three waves per SIMD (two slots) or two (three and four), as the MC kernel does.
template <int APL, int POL>
__global__ __launch_bounds__(kWave* kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(APL == 1 ? 6 : APL == 2 ? 3 : 2)))
void lmc_kernel(LmcArgs) {
    Karg<LmcArgs>* const K = kernel_args<LmcArgs>();
    const int policy = POL >= 0 ? POL : K->policy;
    const int w = threadIdx.x / kWave;
    const int base = w * reread(K)->lds_floats_per_wave;
    const int nchain = reread(K)->P.nchain;
    const int n_items = reread(K)->n_order * nchain;
    const int ln = lane();
    uint16_t* xl = reinterpret_cast<uint16_t*>(s_lds + base + reread(K)->lfeat);
    uint16_t* a1l = reinterpret_cast<uint16_t*>(s_lds + base + reread(K)->la1);
    uint16_t* a1lb = reinterpret_cast<uint16_t*>(s_lds + base + reread(K)->la1b);
    for (;;) {
        int item = 0;
        if (ln == 0) item = atomicAdd(reread(K)->counter, 1);
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= n_items) break;
        const int lig = reread(K)->order[item / nchain];
        const int chain = item % nchain;
        const size_t pid = (size_t)lig * nchain + chain;
        Ctx<APL> C;
        load_ctx(C, (KHead*)K, lig, POL >= 0 ? int(kGrid) : reread(K)->mode, base, reread(K)->hdim_ld);
        Rng rng{reread(K)->seed, uint32_t(lig + reread(K)->lig_index_base), uint32_t(chain), 0u};
        C.evals = 0;
        int n_feat = 0;
        WPose<APL> acc;
        initial_pose(C, acc);
        // step -1 is the start pre-screen: n_start randomised starts (super-Fibonacci
        // orientations spread over n_start * nchain) go through the same candidate code
        // as the MC steps' mutations, and the chain starts from the best one (network,
        // or exact energy for the plain / exact policies)
        const int ns = reread(K)->n_start;
        const bool prescreen = reread(K)->randomize && ns > 1;
        if (reread(K)->randomize && !prescreen) randomize(C, acc, rng, chain, nchain);
        store_pose(C, reread(K)->P, lig, chain, acc);
        save_pose(C, acc, 1);  // the accepted pose lives in LDS between steps
        float best = 1e9f;
        for (int step = prescreen ? -1 : 0; step < reread(K)->mc_steps; step++) {
            const bool pre = step < 0;
            WPose<APL> cand;
            restore_pose(C, cand, 1);
            const float acc_e = cand.e;
            const size_t crow = ((size_t)(pre ? 0 : step) * reread(K)->n_pose + pid) * kGroup;
            if (pre && policy != kPolicyLearned) {
                float be = INFINITY;
                uint32_t bs = rng.draw;
                int bk = 0;
                for (int k = 0; k < ns; k++) {
                    const uint32_t start = rng.draw;
                    WPose<APL> t;
                    restore_pose(C, t, 1);
                    randomize(C, t, rng, chain * ns + k, nchain * ns);
                    Forces<APL> F;
                    const float e = energy_forces(C, t, kVCap, kSlope, F);
                    if (e < be || k == 0) { be = e; bs = start; bk = k; }
                }
                Rng r3 = rng;
                r3.draw = bs;
                randomize(C, cand, r3, chain * ns + bk, nchain * ns);
                store_pose(C, reread(K)->P, lig, chain, cand);
                save_pose(C, cand, 1);
                continue;
            }
            if (policy == kPolicyPlain) {
                mutate(C, cand, rng);
            } else if (policy == kPolicyExact) {
                float be = INFINITY;
                uint32_t bs = rng.draw;
                for (int c = 0; c < reread(K)->n_cand; c++) {
                    const uint32_t start = rng.draw;
                    WPose<APL> t;
                    restore_pose(C, t, 1);
                    mutate(C, t, rng);
                    Forces<APL> F;
                    const float e = energy_forces(C, t, kVCap, kSlope, F);
                    if (e < be || c == 0) { be = e; bs = start; }
                }
                Rng r3 = rng;
                r3.draw = bs;
                restore_pose(C, cand, 1);
                mutate(C, cand, r3);
            } else {
                // candidate c starts at Philox block my_start of lane c
                const int nc = pre ? ns : reread(K)->n_cand;
                uint32_t my_start = 0;
                // the candidate rows sit in the coordinate / pair-force area: randomised starts must
                // not stage their torsion steps there
                C.stage = false;
                for (int c = 0; c < nc; c++) {
                    if (ln == c) my_start = rng.draw;
                    WPose<APL> t;
                    restore_pose(C, t, 1);
                    Move mv;
                    if (pre) {
                        randomize(C, t, rng, chain * ns + c, nchain * ns);
                        mv.kind = 0; mv.mag = 1.0f; mv.moved = 1.0f;
                    } else {
                        mv = mutate(C, t, rng);
                    }
                    uint16_t* dst = policy == kPolicyCollect ? reread(K)->collect_x + (crow + c) * kFeat : xl + c * kFeat;
                    pose_features(C, t, mv, pre ? 999.0f : acc_e, base + reread(K)->lscr, dst);
                }
                n_feat += nc;
                C.stage = true;  // no pose update until the network has read the rows
                if (policy == kPolicyLearned) {
                    wave_lds_fence();
                    const MlpDev W = network(reread(K)->W);
                    float p = mlp_group_scores_lds(W, xl, a1l, a1lb, reread(K)->a1_split, reread(K)->a1_rows);  // lane 16 q + r: score of candidate r
                    p = (ln < nc && p == p) ? p : INFINITY;
                    int rank = 0;
                    float pmin = INFINITY;
                    for (int j = 0; j < nc; j++) {
                        const float pj = rdl(p, j);
                        rank += (pj < p || (pj == p && j < ln)) ? 1 : 0;
                        pmin = fminf(pmin, pj);
                    }
                    float be = INFINITY;
                    uint32_t bs = 0;
                    int pick = 0;
                    if (pre) {
                        pick = __ffsll((long long)__ballot(ln < nc && rank == 0)) - 1;
                        bs = uint32_t(rdl_i(int(my_start), pick));
                        Rng r3 = rng;
                        r3.draw = bs;
                        restore_pose(C, cand, 1);
                        randomize(C, cand, r3, chain * ns + pick, nchain * ns);
                        store_pose(C, reread(K)->P, lig, chain, cand);
                        save_pose(C, cand, 1);
                        continue;
                    }
                    if (reread(K)->sel_temp > 0.0f) {
                        // one candidate drawn with p ~ exp(-(score - min) / T); no exact rescoring
                        const float w = (ln < nc && pmin < INFINITY) ? __expf(-(p - pmin) / reread(K)->sel_temp) : 0.0f;
                        float wsum = 0.0f;
                        for (int j = 0; j < nc; j++) wsum += rdl(w, j);
                        const float target = u01(rng.next().x) * wsum;
                        float cum = 0.0f;
                        for (int j = 0; j < nc; j++) {
                            cum += rdl(w, j);
                            if (cum < target) pick = j + 1;
                        }
                        pick = pick < nc ? pick : nc - 1;
                        bs = uint32_t(rdl_i(int(my_start), pick));
                    }
                    for (int r = 0; reread(K)->sel_temp <= 0.0f && r < reread(K)->top_k; r++) {
                        const unsigned long long m = __ballot(ln < nc && rank == r);
                        const int c = __ffsll((long long)m) - 1;
                        const uint32_t start = uint32_t(rdl_i(int(my_start), c));
                        Rng r2 = rng;
                        r2.draw = start;
                        WPose<APL> t;
                        restore_pose(C, t, 1);
                        mutate(C, t, r2);
                        Forces<APL> F;
                        const float e = energy_forces(C, t, kVCap, kSlope, F);
                        if (e < be || r == 0) { be = e; bs = start; }
                    }
                    Rng r3 = rng;
                    r3.draw = bs;
                    restore_pose(C, cand, 1);
                    mutate(C, cand, r3);
                } else {
                    // collect: every other candidate refined for its label
                    for (int c = nc - 1; c >= 1; c--) {
                        Rng r2 = rng;
                        r2.draw = uint32_t(rdl_i(int(my_start), c));
                        WPose<APL> t;
                        restore_pose(C, t, 1);
                        mutate(C, t, r2);
                        if (reread(K)->collect_e0) {
                            Forces<APL> F;
                            const float e0 = energy_forces(C, t, kVCap, kSlope, F);
                            if (ln == 0) reread(K)->collect_e0[crow + c] = e0;
                        }
                        bfgs(C, t, reread(K)->opt_steps, kVCap, kSlope);
                        if (ln == 0) reread(K)->collect_y[crow + c] = t.e;
                    }
                    Rng r2 = rng;
                    r2.draw = uint32_t(rdl_i(int(my_start), 0));
                    restore_pose(C, cand, 1);
                    mutate(C, cand, r2);
                    if (reread(K)->collect_e0) {
                        Forces<APL> F;
                        const float e0 = energy_forces(C, cand, kVCap, kSlope, F);
                        if (ln == 0) reread(K)->collect_e0[crow] = e0;
                    }
                }
            }
            if (reread(K)->opt_steps == 0) {
                float gd;
                cand.e = energy_grad(C, cand, kVCap, kSlope, gd);
            } else {
                bfgs(C, cand, reread(K)->opt_steps, kVCap, kSlope);
            }
            if (policy == kPolicyCollect && ln == 0) reread(K)->collect_y[crow] = cand.e;
            const uint4 b = rng.next();
            const bool accepted = (cand.e < acc_e) || (u01(b.x) < __expf((acc_e - cand.e) / 1.2f));
            if (step == 0 || accepted) {
                if (cand.e < best) {
                    if (reread(K)->opt_steps > 0) bfgs(C, cand, reread(K)->opt_steps, kVCapAuth, kSlope);
                    if (cand.e < best) {
                        store_pose(C, reread(K)->P, lig, chain, cand);
                        best = cand.e;
                    }
                }
                save_pose(C, cand, 1);
            }
        }
        if (reread(K)->stats && ln == 0) {
            const unsigned long long ev = (unsigned long long)C.evals;
            const unsigned long long nh = (unsigned long long)C.nheavy();
            atomicAdd(&reread(K)->stats[0], ev);
            atomicAdd(&reread(K)->stats[1], (ev + (unsigned long long)n_feat) * 32ull * nh);
            atomicAdd(&reread(K)->stats[2], ev * (unsigned long long)C.npair());
            atomicAdd(&reread(K)->stats[3], 1ull);
        }
    }
}

// Features of selected poses (no move: kind -1, accepted energy 0).
template <int APL>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void features_kernel(FeatArgs) {
    Karg<FeatArgs>* const K = kernel_args<FeatArgs>();
    Karg<FeatArgs>& A = *K;
    const int w = threadIdx.x / kWave;
    const int s = blockIdx.x * kWavesPerBlock + w;
    if (s >= A.n_sel) return;
    const int pid = A.sel[s];
    const int lig = pid / A.P.nchain, chain = pid % A.P.nchain;
    Ctx<APL> C;
    load_ctx(C, (KHead*)K, lig, kGrid, w * A.lds_floats_per_wave, A.hdim_ld);
    WPose<APL> p;
    load_pose<APL>(C, A.P, lig, chain, p);
    Move mv;
    mv.kind = -1; mv.mag = 0.0f; mv.moved = 0.0f;
    pose_features(C, p, mv, 0.0f, C.lh(), A.x + (size_t)s * kFeat);
}

// ------------------------------------------------------------- launchers
#define UD2_APL_SWITCH(apl, CALL) \
    switch (apl) {                \
        case 1: CALL(1);          \
        case 2: CALL(2);          \
        case 3: CALL(3);          \
        case 4: CALL(4);          \
        default: return hipErrorInvalidValue; \
    }

// Whether the build of lmc_kernel for the learned policy runs a search: it holds the grid inter term only.
static bool lmc_learned_build(int policy, int mode) { return policy == kPolicyLearned && mode == kGrid; }

template <int APL>
static hipError_t launch_lmc_t(const LmcArgs& a, int n_blocks, hipStream_t s) {
    const size_t lds = (size_t)a.lds_floats_per_wave * kWavesPerBlock * sizeof(float);
    if (lmc_learned_build(a.policy, a.mode))
        hipLaunchKernelGGL((lmc_kernel<APL, kPolicyLearned>), dim3(n_blocks), dim3(kWave * kWavesPerBlock), lds, s, a);
    else
        hipLaunchKernelGGL((lmc_kernel<APL, -1>), dim3(n_blocks), dim3(kWave * kWavesPerBlock), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_lmc(LmcArgs a, int apl, int n_blocks, hipStream_t s) {
#define CALL(N) return launch_lmc_t<N>(a, n_blocks, s)
    UD2_APL_SWITCH(apl, CALL)
#undef CALL
}

template <int APL>
static hipError_t launch_feat_t(const FeatArgs& a, hipStream_t s) {
    const size_t lds = (size_t)a.lds_floats_per_wave * kWavesPerBlock * sizeof(float);
    const int nb = (a.n_sel + kWavesPerBlock - 1) / kWavesPerBlock;
    hipLaunchKernelGGL(features_kernel<APL>, dim3(nb), dim3(kWave * kWavesPerBlock), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_features(FeatArgs a, int apl, hipStream_t s) {
    if (a.n_sel <= 0) return hipSuccess;
#define CALL(N) return launch_feat_t<N>(a, s)
    UD2_APL_SWITCH(apl, CALL)
#undef CALL
}

template <int APL>
static int lmc_occ_t(int policy, int mode, int lds_bytes) {
    int nb = 0;
    const hipError_t e = lmc_learned_build(policy, mode)
                             ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lmc_kernel<APL, kPolicyLearned>,
                                                                            kWave * kWavesPerBlock, lds_bytes)
                             : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lmc_kernel<APL, -1>,
                                                                            kWave * kWavesPerBlock, lds_bytes);
    if (e != hipSuccess) return 1;
    return nb > 0 ? nb : 1;
}

int lmc_blocks_per_cu(int apl, int policy, int mode, int lds_bytes) {
    switch (apl) {
        case 1: return lmc_occ_t<1>(policy, mode, lds_bytes);
        case 2: return lmc_occ_t<2>(policy, mode, lds_bytes);
        case 3: return lmc_occ_t<3>(policy, mode, lds_bytes);
        default: return lmc_occ_t<4>(policy, mode, lds_bytes);
    }
}

}  // namespace ud2
