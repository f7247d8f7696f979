// HIP kernels of the docking hot path for gfx950 (CDNA4, wave64): Monte Carlo,
// per-pose optimisation hooks, pose-vector scoring, grid-map build, clustering
// and final scoring. The device building blocks and the execution model are
// described in ud2_device.h.
#include <type_traits>

#include "ud2_device.h"

namespace ud2 {

// --------------------------------------------------------------- kernels
// Persistent MC kernel: each wave takes (ligand, chain group) items from the queue and runs whole
// chains of mc_kernel (mc.cu:275-398), randomisation first. A wave runs 64 / TW chains of one ligand,
// one per tile of TW lanes: TW = 64 one chain per wave; TW = 32 (one atom per lane, at most 32 atoms
// and 14 torsions) two, chains 2 i and 2 i + 1 on lanes 0-31 and 32-63, each computed with the same
// bits as by a whole wave. With an odd chain count the last group's second tile repeats the last
// chain and stores nothing. The best pose goes to the pose buffers whenever it improves (the
// reference copies it to out_pose at the same points, mc.cu:389-392).
// OCC is the occupancy hint (waves per SIMD the register allocation must allow). One-atom-per-lane
// ligands fit six waves per SIMD in LDS; the whole-wave kernel runs at six (80 VGPRs, 39 spilled): five
// waves with 96 VGPRs and none spilled measure the same on 256 ligands, and the learned kernel 3 % slower.
// The search is bound by VALU issue, the LDS pipe and latency together. The half-wave kernel (128-137 VGPRs, none
// spilled) comes at 4, 3 and 2 waves. The two-slot kernel runs at three waves per SIMD (127 VGPRs; its LDS
// allows three blocks per CU), the three- and four-slot kernels at two (145 and 171): on ligands of 65-80
// atoms three waves measured 25 % faster than two.
// MODE is the inter term: the grid builds hold nothing of the direct sum and the other way round.
// TEAM: the four waves of a block run one chain (see Team). A search of few chains leaves most of the chip's 1,024
// SIMDs idle and lasts as long as one chain's serial work, 2.4 energies per line search; a team's rounds of four
// trials make that 1.2, with two barriers each: on one GPU, one ligand of 24 atoms at 128 chains and 10 steps 10.1 -> 5.2 ms,
// in direct mode (5 steps) 13.0 -> 6.7 ms, one of 80 atoms 41.3 -> 21.7 and 47.5 -> 21.8 ms.
template <int APL, int TW, int OCC, int MODE, bool TEAM = false>
__global__ __launch_bounds__(kWave* kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(OCC)))
void mc_kernel(McArgs) {
    Karg<McArgs>* const K = kernel_args<McArgs>();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    using Crew = std::conditional_t<TEAM, Team, Solo>;
    Crew crew;
    if constexpr (TEAM) crew = Team{wave, kWavesPerBlock * K->lds_floats_per_wave, 0};
    constexpr int CPW = kWave / TW;  // chains per wave
    const int h = CPW == 1 ? 0 : __lane_id() / TW;
    for (;;) {
        Karg<McArgs>& A = *reread(K);
        const int base = wave * A.lds_floats_per_wave + h * (A.lds_floats_per_wave / CPW);
        const int nchain = A.P.nchain;
        const int ngroup = (nchain + CPW - 1) / CPW;
        const int n_items = A.n_order * ngroup;
        int item = 0;
        if constexpr (TEAM) {
            int* slot = reinterpret_cast<int*>(s_lds + crew.sh) + 2 * kWavesPerBlock;
            __syncthreads();  // every wave has read the last item
            if (threadIdx.x == 0) *slot = atomicAdd(A.counter, 1);
            __syncthreads();
            item = *slot;
        } else {
            if (lane() == 0) item = atomicAdd(A.counter, 1);
        }
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= n_items) break;
        const int lig = A.order[item / ngroup];
        const int c = CPW * (item % ngroup) + h;
        const bool real = CPW == 1 ? !TEAM || wave == 0 : c < nchain;  // who stores
        const int chain = CPW == 1 || real ? c : nchain - 1;
        Ctx<APL, TW, (OCC > 2) && !TEAM> C;
        load_ctx(C, (KHead*)K, lig, MODE, base, A.hdim_ld);
        Rng rng{A.seed, uint32_t(lig + A.lig_index_base), uint32_t(chain), 0u};
        WPose<APL> acc;
        initial_pose(C, acc);
        if (A.randomize) randomize(C, acc, rng, chain, nchain);
        if (A.mc_steps == 0) {
            Forces<APL> F;
            acc.e = energy_forces(C, acc, kVCap, kSlope, F);
            if (real) store_pose(C, reread(K)->P, lig, chain, acc);
            continue;
        }
        if (real) store_pose(C, reread(K)->P, lig, chain, acc);
        save_pose(C, acc, 1);  // the accepted pose lives in LDS between steps
        float best = 1e9f;
        C.evals = 0;
        for (int step = 0; step < reread(K)->mc_steps; step++) {
            WPose<APL> cand;
            restore_pose(C, cand, 1);
            const float acc_e = cand.e;
            mutate(C, cand, rng);
            const int opt_steps = reread(K)->opt_steps;
            if (opt_steps == 0) {
                float gd;
                cand.e = energy_grad(C, cand, kVCap, kSlope, gd);
            } else {
                bfgs(C, cand, opt_steps, kVCap, kSlope, crew);
            }
            const uint4 b = rng.next();
            const bool accepted = (cand.e < acc_e) || (u01(b.x) < __expf((acc_e - cand.e) / 1.2f));
            if (step == 0 || accepted) {
                if (cand.e < best) {
                    if (opt_steps > 0) bfgs(C, cand, opt_steps, kVCapAuth, kSlope, crew);
                    if (cand.e < best) {
                        if (real) store_pose(C, reread(K)->P, lig, chain, cand);
                        best = cand.e;
                    }
                }
                save_pose(C, cand, 1);
            }
        }
        unsigned long long* stats = reread(K)->stats;
        if (stats && tlane<TW>() == 0 && real) {
            const unsigned long long ev = (unsigned long long)C.evals;
            atomicAdd(&stats[0], ev);
            atomicAdd(&stats[1], ev * 32ull * (unsigned long long)C.nheavy());
            atomicAdd(&stats[2], ev * (unsigned long long)C.npair());
            atomicAdd(&stats[3], 1ull);
        }
    }
}

// Per-pose operations on selected poses: BFGS (optimize_cu, E/src/cuda/optimize.cu:14-58),
// energy + gradient, one pose update, one line search from H = I
// (line_search_one_gpu, E/src/cuda/bfgs_wrapper.cu:12-48), or a reset to the
// input conformation.
template <int APL, int MODE>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void opt_kernel(OptArgs) {
    Karg<OptArgs>* const K = kernel_args<OptArgs>();
    Karg<OptArgs>& A = *K;
    const int w = threadIdx.x / kWave;
    const int s = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerBlock + w);
    if (s >= A.n_sel) return;
    const int pid = A.sel ? A.sel[s] : A.few[s];
    const int lig = pid / A.P.nchain, chain = pid % A.P.nchain;
    const int o = A.sel ? A.pos[s] : A.few_pos[s];
    Ctx<APL> C;
    load_ctx(C, (KHead*)K, lig, MODE, w * A.lds_floats_per_wave, A.hdim_ld);
    WPose<APL> P;
    const int ln = lane();
    if (A.op == 4) {
        initial_pose(C, P);
        store_pose(C, A.P, lig, chain, P);
        return;
    }
    load_pose(C, A.P, lig, chain, P);
    if (A.op == 0) {
        bfgs(C, P, A.max_steps, A.v_cap, A.slope);
        store_pose(C, A.P, lig, chain, P);
        if (A.out_e && ln == 0) A.out_e[o] = P.e;
    } else if (A.op == 1) {
        float g;
        const float e = energy_grad(C, P, A.v_cap, A.slope, g);
        if (A.out_e && ln == 0) A.out_e[o] = e;
        if (A.out_g && ln < C.dim()) A.out_g[(size_t)o * kWave + ln] = g;
    } else if (A.op == 2) {
        const float d = ln < C.dim() ? A.dir[(size_t)o * kWave + ln] : 0.0f;
        apply_update(C, P, d, A.alpha);
        store_pose(C, A.P, lig, chain, P);
    } else {
        float g;
        const float e0 = energy_grad(C, P, A.v_cap, A.slope, g);
        const float p = ln < C.dim() ? -g : 0.0f;
        WPose<APL> xn;
        float gn, e1, al;
        line_search(C, P, g, p, e0, A.v_cap, A.slope, xn, gn, e1, al);
        xn.e = e1;
        store_pose(C, A.P, lig, chain, xn);
        if (A.out_e && ln == 0) A.out_e[o] = al;
        if (A.out_g && ln < C.dim()) A.out_g[(size_t)o * kWave + ln] = gn;
    }
}

// Energy + gradient of pose vectors [centre, quaternion (w, x, y, z), torsions]
// of one ligand: torsions set on its input conformation in index order, then
// the conformer rotated by q about its centroid and moved to the centre;
// rot_vec = rotvec(q).
template <int APL, int MODE>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void posevec_kernel(PoseVecArgs) {
    Karg<PoseVecArgs>* const K = kernel_args<PoseVecArgs>();
    Karg<PoseVecArgs>& A = *K;
    const int w = threadIdx.x / kWave;
    Ctx<APL> C;
    load_ctx(C, (KHead*)K, A.lig, MODE, w * A.lds_floats_per_wave, A.hdim_ld);
    WPose<APL> P0;
    initial_pose(C, P0);
    const int ln = lane();
    const int nt = C.ntors(), dimv = 7 + nt, dimg = 6 + nt;
    const int64_t stride = (int64_t)gridDim.x * kWavesPerBlock;
    for (int64_t i = (int64_t)blockIdx.x * kWavesPerBlock + w; i < A.n; i += stride) {
        const float* pv = A.pv + i * dimv;
        const float mine = ln < dimv ? pv[ln] : 0.0f;
        WPose<APL> P = P0;
        for (int t = 0; t < nt; t++) apply_torsion(C, P, t, rdl(mine, 7 + t) - rdl(P.dihe, t));
        if (nt > 0) centroid(C, P);
        const float4 q = make_float4(rdl(mine, 3), rdl(mine, 4), rdl(mine, 5), rdl(mine, 6));
        const float n0 = rdl(mine, 0), n1 = rdl(mine, 1), n2 = rdl(mine, 2);
        rigid_move(C, P, q, P.c0, P.c1, P.c2, n0, n1, n2);
        P.c0 = n0; P.c1 = n1; P.c2 = n2;
        const float3 rv = quat_to_rotvec(q);
        P.r0 = uni(rv.x); P.r1 = uni(rv.y); P.r2 = uni(rv.z);
        float g;
        const float e = energy_grad(C, P, A.v_cap, A.slope, g);
        if (ln == 0) A.e[i] = e;
        if (ln < dimg) A.g[i * dimg + ln] = g;
    }
}

// Whether a receptor atom can be within the cutoff of a point of the box lo .. hi.
__device__ __forceinline__ bool in_reach(const float4& r, const float lo[3], const float hi[3]) {
    const float ex = fmaxf(fmaxf(lo[0] - r.x, r.x - hi[0]), 0.0f);
    const float ey = fmaxf(fmaxf(lo[1] - r.y, r.y - hi[1]), 0.0f);
    const float ez = fmaxf(fmaxf(lo[2] - r.z, r.z - hi[2]), 0.0f);
    return sq_dist(ex, ey, ez) < kR2Reach;
}

// The atoms rec[c0 .. c0 + kNearChunk) in reach of the box lo .. hi, compacted in receptor order into near (x, y, z,
// atom_word) by a block of 256 threads; returns their number. wave_n: the counts of 64 atoms each.
constexpr int kNearChunk = 1024;
__device__ __forceinline__ int near_atoms(const float4* rec, int nrec, int c0, const float lo[3], const float hi[3],
                                          float4* near, int* wave_n) {
    const int tid = threadIdx.x, ln = lane(), w = tid / kWave;
    // atom c0 + 256 i + tid on thread tid
    float4 r[kNearChunk / 256];
    unsigned long long keep[kNearChunk / 256];
#pragma unroll
    for (int i = 0; i < kNearChunk / 256; i++) {
        const int j = c0 + 256 * i + tid;
        r[i] = rec[j < nrec ? j : nrec - 1];
        keep[i] = __ballot(j < nrec && in_reach(r[i], lo, hi));
        if (ln == 0) wave_n[4 * i + w] = __popcll(keep[i]);
    }
    __syncthreads();
    int n = 0;
#pragma unroll
    for (int i = 0; i < kNearChunk / 256; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (v == w && ((keep[i] >> ln) & 1ull))
                near[n + __popcll(keep[i] & ((1ull << ln) - 1ull))] = r[i];
            n += wave_n[4 * i + v];
        }
    __syncthreads();
    return n;
}

// Grid maps: one thread per grid point, all probe types at once, a block of 8 x 8 x 4 points (a wave 8 x 4
// x 2, so that its lanes mostly agree on which receptor atoms are in reach). The block first compacts, in
// receptor order, the atoms within the cutoff of its bounding box into LDS (about 190 of 2,000 at
// 0.021 atoms / A^3), kNearChunk receptor atoms at a time; each point then sums those in the cutoff in
// the receptor's order, which gives the bits of the sum over the whole receptor. The slots come
// sorted by probe radius: the terms that depend on the distance alone are formed once per radius (4 for the 8
// default types), and the flag terms per slot from scalar registers. Bound by VALU issue and the two
// exponentials per radius. The loop over the whole receptor for every point, with every term per type,
// took 785 us for 81^3 points, 8 types and 2,000 atoms.
__global__ __launch_bounds__(256) void grid_kernel(GridArgs A) {
    const SceneDev& S = A.S;
    __shared__ float4 near[kNearChunk];  // x, y, z, atom_word
    __shared__ int wave_n[kNearChunk / kWave];
    const int tid = threadIdx.x, ln = lane(), w = tid / kWave;
    const int nb[2] = {(S.gn[0] + 7) / 8, (S.gn[1] + 7) / 8};
    const int b0[3] = {int(blockIdx.x % nb[0]) * 8, int((blockIdx.x / nb[0]) % nb[1]) * 8,
                       int(blockIdx.x / (nb[0] * nb[1])) * 4};
    const int ix = b0[0] + (ln & 7), iy = b0[1] + 4 * (w & 1) + ((ln >> 3) & 3), iz = b0[2] + 2 * (w >> 1) + (ln >> 5);
    const float px = S.gorigin[0] + S.gspacing * float(ix);
    const float py = S.gorigin[1] + S.gspacing * float(iy);
    const float pz = S.gorigin[2] + S.gspacing * float(iz);
    float lo[3], hi[3];
    constexpr int kSide[3] = {7, 7, 3};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        lo[d] = S.gorigin[d] + S.gspacing * float(b0[d]);
        hi[d] = S.gorigin[d] + S.gspacing * float(b0[d] + kSide[d]);
    }
    constexpr int kMaxSlots = kNumTypes;
    float acc[kMaxSlots];
#pragma unroll
    for (int k = 0; k < kMaxSlots; k++) acc[k] = 0.0f;
    for (int c0 = 0; c0 < S.nrec; c0 += kNearChunk) {
        const int n = near_atoms(S.rec, S.nrec, c0, lo, hi, near, wave_n);
        for (int j = 0; j < n; j++) {
            const float4 q = near[j];
            const float dx = q.x - px, dy = q.y - py, dz = q.z - pz;
            const float rr = dx * dx + dy * dy + dz * dz;
            const uint32_t word = __builtin_amdgcn_readfirstlane(__float_as_uint(q.w));
            if (rr < kR2Cut) {
                const float dist = sqrtf(rr), rj = word_radius(word);
                float e0 = 0.0f, h = 0.0f, b = 0.0f;
#pragma unroll
                for (int k = 0; k < kMaxSlots; k++) {
                    if (k < A.nslot) {
                        if (k == 0 || A.radius[k] != A.radius[k - 1]) e0 = eval_radial(dist - (A.radius[k] + rj), h, b);
                        const int fl = int(A.lut[k] >> word_flags2(word)) & 3;
                        acc[k] += add_flag_terms(e0, h, b, fl);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (ix >= S.gn[0] || iy >= S.gn[1] || iz >= S.gn[2]) return;
    const size_t npt = (size_t)S.gn[0] * S.gn[1] * S.gn[2];
    const size_t id = ((size_t)iz * S.gn[1] + iy) * S.gn[0] + ix;
#pragma unroll
    for (int k = 0; k < kMaxSlots; k++)
        if (k < A.nslot) A.maps[(size_t)A.slot[k] * npt + id] = acc[k];
}

// Candidates of one round whose RMSDs a thread forms together.
constexpr int kClusterCand = 4;

// RMSDs of pose xo (this thread's; `live` threads only) with kClusterCand poses xc, the same for the
// whole wave: bit k set where the RMSD to xc[k] is below limit. cal_rmsd_pair_warp (cluster.cu:16-37)
// over the heavy atoms in float with rounded operations in atom order, so that each is bit-identical to a
// scalar float loop on the host. The partial sums only grow, so a wave stops at the first four atoms after
// which every sum has passed `cut`, a value of the sum from which the rounded RMSD is not below limit.
__device__ __forceinline__ uint32_t rmsd_below(const float* xo, const float* const xc[kClusterCand], bool live,
                                               const unsigned long long heavy[kMaxApl], int natom, int n, float cut,
                                               float limit) {
    float s[kClusterCand];
#pragma unroll
    for (int k = 0; k < kClusterCand; k++) s[k] = live ? 0.0f : INFINITY;
    for (int a0 = 0; a0 < natom; a0 += 4) {
        const uint32_t hv = uint32_t(heavy[a0 / kWave] >> (a0 % kWave)) & 15u;  // no bits past natom
        if (hv == 0) continue;
        float o[12];
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((hv >> i) & 1u) {
                const float* p = xo + 3 * (a0 + i);
                o[3 * i] = p[0]; o[3 * i + 1] = p[1]; o[3 * i + 2] = p[2];
            }
#pragma unroll
        for (int k = 0; k < kClusterCand; k++) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if ((hv >> i) & 1u) {
                    const float* p = xc[k] + 3 * (a0 + i);
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const float d = __fsub_rn(o[3 * i + c], uload(p + c));
                        s[k] = __fadd_rn(s[k], __fmul_rn(d, d));
                    }
                }
        }
        bool open = false;
#pragma unroll
        for (int k = 0; k < kClusterCand; k++) open |= s[k] < cut;
        if (__ballot(open) == 0ull) return 0u;
    }
    uint32_t below = 0u;
#pragma unroll
    for (int k = 0; k < kClusterCand; k++)
        if (live && __fsqrt_rn(__fdiv_rn(s[k], float(n))) < limit) below |= 1u << k;
    return below;
}

// Greedy leader clustering of one ligand per block (cluster_cu, cluster.cu:93-129):
// poses ranked by ascending energy (ties by index), a pose becomes a leader when
// its RMSD to every current leader is >= limit.
// The remaining poses are kept compacted in rank order, and a round takes the first of them as
// candidates, 4 per group of threads: every remaining pose is measured against every candidate (a
// thread holds one pose and reads its group's candidates by scalar loads), the candidates are resolved
// among themselves in rank order, and the poses near a new leader drop out. As the poses get fewer, the
// block splits into more groups (up to 8, 32 candidates a round). The RMSDs are a serial sum per pair,
// so what bounds the kernel is the latency of those sums and how many run at once. One pose at a time
// against the leaders so far (a thread per leader, three barriers a pose) took 4,410 us for 64 ligands
// of 512 poses; this takes 290 us. Blocks of 512 threads took 315 us. With up to 64 poses the block
// (a power of two, blockDim.x) is what the first round can use, a wave for every four poses: 4,096 ligands of
// 1 / 8 / 32 poses take 20 / 73 / 228 us, in blocks of 1,024 threads 326 / 373 / 520 us (one pose at a time 19 / 170 / 940).
constexpr int kClusterThreads = 1024;
__global__ __launch_bounds__(kClusterThreads) void cluster_kernel(ClusterArgs A) {
    const int nt = blockDim.x;
    const int lig = blockIdx.x;
    if (lig >= A.n_lig) return;
    const int E = A.nchain, tid = threadIdx.x, ln = lane();
    const int n_words = (E + kWave - 1) / kWave;
    float* es = s_lds;                                          // [E], until the poses are ranked
    uint32_t* near = reinterpret_cast<uint32_t*>(s_lds);        // [E] then: candidates near each remaining pose
    unsigned long long* left = reinterpret_cast<unsigned long long*>(s_lds + cluster_near_words(E));  // ranks remaining
    uint16_t* order = reinterpret_cast<uint16_t*>(left + n_words);  // [E] pose of each rank
    uint16_t* list = order + E;                                     // [E] remaining ranks, compacted
    const DevLig d = A.L.ligs[lig];
    const float* e = A.e + (size_t)lig * E;
    for (int i = tid; i < E; i += nt) {
        const float ei = e[i];
        es[i] = ei != ei ? INFINITY : ei;
    }
    for (int w = tid; w < n_words; w += nt) {
        const int m = E - w * kWave;
        left[w] = m >= kWave ? ~0ull : (1ull << m) - 1ull;
    }
    unsigned long long heavy[kMaxApl];
    int n = 0;
#pragma unroll
    for (int k = 0; k < kMaxApl; k++) {
        const int a = ln + kWave * k;
        heavy[k] = __ballot(a < d.natom && __float_as_int(A.L.atom_x0[d.atom_off + (a < d.natom ? a : 0)].w) != kTypeH);
        n += __popcll(heavy[k]);
    }
    __syncthreads();
    for (int i = tid; i < E; i += nt) {
        const float ei = es[i];
        int rank = 0;
        for (int j = 0; j < E; j++) {
            const float ej = es[j];
            rank += (ej < ei) || (ej == ei && j < i);
        }
        order[rank] = uint16_t(i);
    }
    // sums from which sqrt(sum / n) is not below limit whatever the roundings (a few 1e-7); no cut for
    // limits whose square loses precision
    float cut = A.limit * A.limit * float(n) * 1.00001f;
    if (!(cut > 1e-30f)) cut = A.limit > 0.0f && n > 0 ? INFINITY : 0.0f;
    const float* xb = A.x + (size_t)d.atom_off * E * 3;
    const size_t stride = (size_t)d.natom * 3;
    int n_lead = 0;
    __syncthreads();
    for (;;) {
        // compact the remaining ranks
        int total = 0;
        for (int w = 0; w < n_words; w++) total += __popcll(left[w]);
        if (total == 0) break;
        for (int r = tid; r < E; r += nt) {
            const unsigned long long m = left[r / kWave];
            if ((m >> (r % kWave)) & 1ull) {
                int at = __popcll(m & ((1ull << (r % kWave)) - 1ull));
                for (int w = 0; w < r / kWave; w++) at += __popcll(left[w]);
                list[at] = uint16_t(r);
                near[at] = 0u;
            }
        }
        __syncthreads();
        int groups = 1;
        while (groups < 8 && (2 * groups) * ((total + kWave - 1) / kWave) * kWave <= nt) groups *= 2;
        const int per = nt / groups, g = __builtin_amdgcn_readfirstlane(tid >> (31 - __clz(per)));
        const int n_cand = min(kClusterCand * groups, total);
        if (total > 1 && kClusterCand * g < n_cand) {  // the last pose left leads, whatever it is near
            const float* xc[kClusterCand];
#pragma unroll
            for (int k = 0; k < kClusterCand; k++) {
                const int i = min(kClusterCand * g + k, n_cand - 1);
                xc[k] = xb + stride * (size_t)__builtin_amdgcn_readfirstlane(int(order[list[i]]));
            }
            const uint32_t real = (1u << min(kClusterCand, n_cand - kClusterCand * g)) - 1u;
            for (int q0 = tid & (per - 1) & ~(kWave - 1); q0 < total; q0 += per) {
                const int q = q0 + ln;
                const bool live = q < total;
                const float* xo = xb + stride * (size_t)order[list[live ? q : 0]];
                const uint32_t b = rmsd_below(xo, xc, live, heavy, d.natom, n, cut, A.limit) & real;
                if (b) atomicOr(&near[q], b << (kClusterCand * g));
            }
        }
        __syncthreads();
        // the candidates in rank order: one becomes a leader unless a leader before it is near
        const uint32_t mine = ln < n_cand ? near[ln] : 0u;
        uint32_t lead = 0u;
        for (int i = 0; i < n_cand; i++)
            if ((uint32_t(rdl_i(int(mine), i)) & lead) == 0u) lead |= 1u << i;
        if (tid < n_cand && ((lead >> tid) & 1u))
            A.leaders[(size_t)lig * E + n_lead + __popc(lead & ((1u << tid) - 1u))] = order[list[tid]];
        n_lead += __popc(lead);
        for (int q = tid; q < total; q += nt)
            if (q < n_cand || (near[q] & lead)) {
                const int r = list[q];
                atomicAnd(&left[r / kWave], ~(1ull << (r % kWave)));
            }
        __syncthreads();
    }
    if (tid == 0) A.nleaders[lig] = n_lead;
}

// Weighted Vina terms of one heavy pair at surface distance d (Vina::eval_decomp,
// E/src/score/vina.h:256-274): gauss1, gauss2, repulsion, hydrophobic, hbond,
// with the expressions of eval_ef.
__device__ __forceinline__ void eval_terms(float d, int flags, float t[5]) {
    t[0] = -0.035579f * __expf(-4.0f * d * d);
    const float t2 = (d - 3.0f) * 0.5f;
    t[1] = -0.005156f * __expf(-t2 * t2);
    const float dn = fminf(d, 0.0f);
    t[2] = 0.840245f * dn * dn;
    t[3] = (flags & 1) ? -0.035069f * fminf(fmaxf(1.5f - d, 0.0f), 1.0f) : 0.0f;
    t[4] = (flags & 2) ? -0.587439f * fminf(fmaxf(-d * (1.0f / 0.7f), 0.0f), 1.0f) : 0.0f;
}

// Final re-score of selected poses, score() (E/src/score/score.cpp:12-108):
// no curl, intra pairs once, direct inter sum, penalty at the fixed slope, bias
// sites. DECOMP: instead, the per-atom split of the inter sum into its five
// terms, score_decomp() (score.cpp:115-147).
template <int APL, bool DECOMP>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void final_score_kernel(ScoreArgs A) {
    const int w = threadIdx.x / kWave;
    const int s = blockIdx.x * kWavesPerBlock + w;
    if (s >= A.n_sel) return;
    const int pid = A.sel[s];
    const int lig = pid / A.nchain, chain = pid % A.nchain;
    const DevLig d = A.L.ligs[lig];
    const float* xb = A.x + ((size_t)d.atom_off * A.nchain + (size_t)chain * d.natom) * 3;
    SceneArg& S = kernel_args<ScoreArgs>()->S;
    LigArg& L = kernel_args<ScoreArgs>()->L;
    const int ln = lane();
    float e_inter = 0.0f, e_pen = 0.0f, e_intra = 0.0f, e_bias = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; k++) {
        const int a = ln + kWave * k;
        if (a >= d.natom) continue;
        const int ti = __float_as_int(L.atom_x0[d.atom_off + a].w);
        const float px = xb[3 * a], py = xb[3 * a + 1], pz = xb[3 * a + 2];
        if (!DECOMP && L.bias_type != 0 && L.bias_start) {
            const int j1 = L.bias_start[d.atom_off + a + 1];
            for (int j = L.bias_start[d.atom_off + a]; j < j1; j++) {
                const float4 b = L.bias_site[j];
                float sdummy;
                e_bias += bias_site_energy(L.bias_type, L.bias_k, b, L.bias_r2[j], ti, b.x - px, b.y - py, b.z - pz,
                                           sdummy);
            }
        }
        float t5[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (ti != kTypeH) {
            const float ri = c_vdw[ti];
            const uint32_t lut = pair_lut(c_tflags[ti]);
            for_reach(S, reach_of(S, px, py, pz), [&](float qx, float qy, float qz, uint32_t word) {
                const float rx = qx - px, ry = qy - py, rz = qz - pz;
                const float rr = rx * rx + ry * ry + rz * rz;
                if (rr < kR2Cut) {
                    const float dist = sqrtf(rr) - (ri + word_radius(word));
                    const int fl = int(lut >> word_flags2(word)) & 3;
                    if (DECOMP) {
                        float t[5];
                        eval_terms(dist, fl, t);
#pragma unroll
                        for (int q = 0; q < 5; q++) t5[q] += t[q];
                    } else {
                        float dd;
                        e_inter += eval_ef(dist, fl, &dd);
                    }
                }
            });
            if (px < S.box_lo[0]) e_pen += S.box_lo[0] - px;
            if (px > S.box_hi[0]) e_pen += px - S.box_hi[0];
            if (py < S.box_lo[1]) e_pen += S.box_lo[1] - py;
            if (py > S.box_hi[1]) e_pen += py - S.box_hi[1];
            if (pz < S.box_lo[2]) e_pen += S.box_lo[2] - pz;
            if (pz > S.box_hi[2]) e_pen += pz - S.box_hi[2];
        }
        if (DECOMP) {
            float* o = A.decomp + ((size_t)s * A.decomp_stride + a) * 5;
#pragma unroll
            for (int q = 0; q < 5; q++) o[q] = t5[q];
        }
    }
    if (DECOMP) return;
    const uint2* pr = L.pairs + d.pair_off;
    for (int p = ln; p < d.npair; p += kWave) {
        const uint2 rec = pr[p];
        const int i = rec.x & 255, j = (rec.x >> 8) & 255, fl = (rec.x >> 16) & 3;
        float rx = xb[3 * j] - xb[3 * i], ry = xb[3 * j + 1] - xb[3 * i + 1], rz = xb[3 * j + 2] - xb[3 * i + 2];
        float rr = rx * rx + ry * ry + rz * rz;
        if (rr < kR2Cut) {
            float dd;
            e_intra += eval_ef(sqrtf(rr) - __uint_as_float(rec.y), fl, &dd);
        }
    }
    e_inter = wave_sum(e_inter);
    e_pen = wave_sum(e_pen) * kSlope;
    e_intra = wave_sum(e_intra);
    e_bias = wave_sum(e_bias);
    if (ln == 0 && A.out4) {
        A.out4[(size_t)s * 4] = e_intra;
        A.out4[(size_t)s * 4 + 1] = e_inter;
        A.out4[(size_t)s * 4 + 2] = e_pen;
        A.out4[(size_t)s * 4 + 3] = e_bias;
    }
}

__global__ void fill_i32_kernel(int32_t* p, int32_t v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------------- launchers
// Pair steps of the ligands of at most 32 atoms (LigSetDev::pack) from their folded diagonals (mask bit l of diagonal
// d: the pair {l, (l + d) mod natom} is scored), a ligand per block, a lane per entry. On the GPU, where a table is
// written in its 64 lanes' order; formed on the host and copied, they made a set of 1,000 ligands of 12-31 atoms
// take 5.4 ms instead of 3.7.
__global__ __launch_bounds__(kWave) void pack_diagonals_kernel(LigSetDev L, uint4* __restrict__ pack) {
    const DevLig d = L.ligs[blockIdx.x];
    if (d.natom > kWave / 2) return;
    const int ln = lane(), a = ln & 31, na = d.natom;
    const auto type = [&](int i) { return __float_as_int(L.atom_x0[d.atom_off + i].w); };
    for (int s = 0; s < d.npack; s++) {
        const int dg = 2 * s + 1, dl = dg + (ln >> 5);
        uint4 t = make_uint4(0u, 0u, __float_as_uint(kRampNoPair), 0u);
        if (a < na) {
            const int j = (a + dl) % na;
            if (dl <= d.nfold && ((L.fold_mask[d.fold_off + dl - 1] >> a) & 1ull)) {
                const int fl = pair_flags(type(a), type(j));
                t.z = __float_as_uint(ramp_hyd(fl));
                t.w = __float_as_uint(ramp_hb(fl));
            }
            t.x = uint32_t(16 * j);
            t.y = uint32_t(4 * ((a + na - dg % na) % na)) | (uint32_t(4 * (32 + (a + na - (dg + 1) % na) % na)) << 8);
        }
        pack[(size_t)(d.pack_off + s) * kWave + ln] = t;
    }
}

hipError_t launch_pack_diagonals(const LigSetDev& L, int n_lig, uint4* pack, hipStream_t s) {
    hipLaunchKernelGGL(pack_diagonals_kernel, dim3(n_lig), dim3(kWave), 0, s, L, pack);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int32_t* p, int32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

// Reach lists. A block takes a brick of 4 x 4 x 2 cells, eight per wave: it compacts the receptor atoms in reach of the
// brick into LDS, kNearChunk receptor atoms at a time, and every wave keeps, in receptor order, those
// within reach of each of its cells' cubes (widened a little for points that round into them). The first launch
// counts and gives every wave's lists their place, the second writes them. Bound by latency, at few waves: 2,000 atoms and
// 15,625 cells take 18 + 16 us. A wave per cell over the whole receptor took 27 + 46 us.
constexpr int kReachBrick[3] = {4, 4, 2}, kReachPerWave = 4 * 4 * 2 / kWavesPerBlock;
template <bool FILL>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void reach_kernel(ReachArgs A) {
    __shared__ float4 near[kNearChunk];
    __shared__ int wave_n[kNearChunk / kWave];
    const int ln = lane(), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int nb[2] = {(A.rn[0] + kReachBrick[0] - 1) / kReachBrick[0], (A.rn[1] + kReachBrick[1] - 1) / kReachBrick[1]};
    const int b0[3] = {int(blockIdx.x % nb[0]) * kReachBrick[0], int((blockIdx.x / nb[0]) % nb[1]) * kReachBrick[1],
                       int(blockIdx.x / (nb[0] * nb[1])) * kReachBrick[2]};
    const auto low = [&](int d, int c) { return A.rorigin[d] + A.edge * float(c) - 1e-3f; };
    const auto high = [&](int d, int c) { return A.rorigin[d] + A.edge * float(c + 1) + 1e-3f; };
    float lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        lo[d] = low(d, b0[d]);
        hi[d] = high(d, b0[d] + kReachBrick[d] - 1);
    }
    int cell[kReachPerWave], n[kReachPerWave], at[kReachPerWave];  // cell -1: none
    const auto place = [&](int k, int c[3]) {
        const int i = kReachPerWave * w + k;
        c[0] = b0[0] + i % kReachBrick[0];
        c[1] = b0[1] + i / kReachBrick[0] % kReachBrick[1];
        c[2] = b0[2] + i / (kReachBrick[0] * kReachBrick[1]);
    };
#pragma unroll
    for (int k = 0; k < kReachPerWave; k++) {
        int c[3];
        place(k, c);
        cell[k] = c[0] < A.rn[0] && c[1] < A.rn[1] && c[2] < A.rn[2] ? (c[2] * A.rn[1] + c[1]) * A.rn[0] + c[0] : -1;
        n[k] = 0;
        at[k] = FILL && cell[k] >= 0 ? A.off[cell[k]].x : 0;
    }
    for (int c0 = 0; c0 < A.nrec; c0 += kNearChunk) {
        const int m = near_atoms(A.rec, A.nrec, c0, lo, hi, near, wave_n);
#pragma unroll
        for (int k = 0; k < kReachPerWave; k++) {
            if (cell[k] < 0) continue;
            int c[3];
            place(k, c);
            float clo[3], chi[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                clo[d] = low(d, c[d]);
                chi[d] = high(d, c[d]);
            }
            for (int j0 = 0; j0 < m; j0 += kWave) {
                const int j = j0 + ln;
                const float4 r = near[j < m ? j : m - 1];
                const unsigned long long keep = __ballot(j < m && in_reach(r, clo, chi));
                if (FILL && ((keep >> ln) & 1ull)) A.reach[at[k] + n[k] + __popcll(keep & ((1ull << ln) - 1ull))] = r;
                n[k] += __popcll(keep);
            }
        }
        __syncthreads();  // before the next chunk overwrites near
    }
    if (FILL) {
#pragma unroll
        for (int k = 0; k < kReachPerWave; k++)
            if (cell[k] >= 0 && ln < (kReachPad - n[k] % kReachPad) % kReachPad)
                A.reach[at[k] + n[k] + ln] = make_float4(1e18f, 1e18f, 1e18f, 0.0f);
        return;
    }
    // one atomic per block: a thousand on one word take 15 us
    __shared__ unsigned long long base[kWavesPerBlock + 1];
    unsigned long long sum = 0;
#pragma unroll
    for (int k = 0; k < kReachPerWave; k++) sum += (n[k] + kReachPad - 1) / kReachPad * kReachPad;
    if (ln == 0) base[w] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        sum = 0;
        for (int v = 0; v < kWavesPerBlock; v++) sum += base[v];
        base[kWavesPerBlock] = atomicAdd(A.total, sum);
    }
    __syncthreads();
    if (ln != 0) return;
    unsigned long long next = base[kWavesPerBlock];
    for (int v = 0; v < w; v++) next += base[v];
#pragma unroll
    for (int k = 0; k < kReachPerWave; k++) {
        if (cell[k] < 0) continue;
        const int len = (n[k] + kReachPad - 1) / kReachPad * kReachPad;
        A.off[cell[k]] = make_int2(int(next), int(next) + len);  // lists of more than kReachEntries are not used
        next += len;
    }
}

hipError_t launch_reach(const ReachArgs& a, bool fill, hipStream_t s) {
    int64_t n = 1;
    for (int d = 0; d < 3; d++) n *= (a.rn[d] + kReachBrick[d] - 1) / kReachBrick[d];
    if (n <= 0) return hipSuccess;
    const dim3 grid((unsigned)n), block(kWave * kWavesPerBlock);
    if (fill) hipLaunchKernelGGL(reach_kernel<true>, grid, block, 0, s, a);
    else hipLaunchKernelGGL(reach_kernel<false>, grid, block, 0, s, a);
    return hipGetLastError();
}

// Cell-major copy of the maps: one thread per cell and map.
__global__ __launch_bounds__(256) void brick_kernel(BrickArgs A) {
    const int cx = A.gn[0] - 1, cy = A.gn[1] - 1, cz = A.gn[2] - 1;
    const int64_t ncell = (int64_t)cx * cy * cz;
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= ncell * A.nslot) return;
    const int slot = int(id / ncell);
    const int64_t c = id % ncell;
    const int ix = int(c % cx), iy = int((c / cx) % cy), iz = int(c / ((int64_t)cx * cy));
    const int nx = A.gn[0], nxy = A.gn[0] * A.gn[1];
    const float* m = A.maps + (size_t)slot * (size_t)nxy * A.gn[2] + (size_t)iz * nxy + (size_t)iy * nx + ix;
    A.cells[2 * id] = make_float4(m[0], m[1], m[nx], m[nx + 1]);
    A.cells[2 * id + 1] = make_float4(m[nxy], m[nxy + 1], m[nxy + nx], m[nxy + nx + 1]);
}

hipError_t launch_brick(const BrickArgs& a, hipStream_t s) {
    const int64_t n = (int64_t)(a.gn[0] - 1) * (a.gn[1] - 1) * (a.gn[2] - 1) * a.nslot;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(brick_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// Random-gather probe over the cell-major maps: each thread reads kProbePerThread cells drawn by an
// integer hash from the first `span` cells (two float4 per cell, one 32-byte sector, as the search's
// trilinear gathers read them) and writes the sum of what it read. It measures the bandwidth that
// scattered 32-byte gathers over this footprint can reach on the device.
__global__ __launch_bounds__(256) void gather_probe_kernel(const float4* cells, uint32_t span, uint32_t seed,
                                                           float* out, int64_t n_threads) {
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n_threads) return;
    float acc = 0.0f;
    uint32_t h = uint32_t(id) ^ (uint32_t(id >> 32) * 0x85EBCA6Bu) ^ seed;
#pragma unroll 8
    for (int k = 0; k < kProbePerThread; k++) {
        // murmur3's 32-bit finaliser of (h + k)
        uint32_t x = h + uint32_t(k) * 0x9E3779B9u;
        x ^= x >> 16; x *= 0x85EBCA6Bu; x ^= x >> 13; x *= 0xC2B2AE35u; x ^= x >> 16;
        const uint32_t c = uint32_t((uint64_t(x) * span) >> 32);  // < span
        const float4 a = cells[2 * (size_t)c], b = cells[2 * (size_t)c + 1];
        acc += (a.x + a.y + a.z + a.w) + (b.x + b.y + b.z + b.w);
    }
    out[id] = acc;
}

hipError_t launch_gather_probe(const float4* cells, uint32_t span, uint32_t seed, float* out, int64_t n_threads,
                               hipStream_t s) {
    if (n_threads <= 0) return hipSuccess;
    hipLaunchKernelGGL(gather_probe_kernel, dim3((unsigned)((n_threads + 255) / 256)), dim3(256), 0, s, cells, span,
                       seed, out, n_threads);
    return hipGetLastError();
}

// VALU probe: each thread runs kValuChains independent FP32 FMA chains of `iters` steps and writes their
// sum. Enough waves in flight hide each chain's latency, so the launch measures the rate at which the
// chip issues plain (unpacked) FP32 VALU instructions: the VALU ceiling of the search kernels, which
// are built without packed FP32 instructions.
constexpr int kValuChains = 8;
__global__ __launch_bounds__(256) void valu_probe_kernel(float* out, int iters, int64_t n_threads) {
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n_threads) return;
    float a[kValuChains];
#pragma unroll
    for (int k = 0; k < kValuChains; k++) a[k] = float(id & 1023) * 1e-6f + float(k);
    const float m = 0.9999f, c = 1e-7f;
    for (int i = 0; i < iters; i++) {
#pragma unroll
        for (int k = 0; k < kValuChains; k++) a[k] = __builtin_fmaf(a[k], m, c);
    }
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < kValuChains; k++) s += a[k];
    out[id] = s;
}

hipError_t launch_valu_probe(float* out, int iters, int64_t n_threads, hipStream_t s) {
    if (n_threads <= 0) return hipSuccess;
    hipLaunchKernelGGL(valu_probe_kernel, dim3((unsigned)((n_threads + 255) / 256)), dim3(256), 0, s, out, iters,
                       n_threads);
    return hipGetLastError();
}

hipError_t launch_grid_build(const GridArgs& a, hipStream_t s) {
    const int64_t nb = (int64_t)((a.S.gn[0] + 7) / 8) * ((a.S.gn[1] + 7) / 8) * ((a.S.gn[2] + 3) / 4);
    hipLaunchKernelGGL(grid_kernel, dim3((unsigned)nb), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <int APL, int TW, int OCC, int MODE = kGrid>
static hipError_t launch_mc_t(const McArgs& a, int n_blocks, hipStream_t s) {
    size_t lds = (size_t)a.lds_floats_per_wave * kWavesPerBlock * sizeof(float);
    hipLaunchKernelGGL((mc_kernel<APL, TW, OCC, MODE>), dim3(n_blocks), dim3(kWave * kWavesPerBlock), lds, s, a);
    return hipGetLastError();
}

// A team launch (n_blocks chains at a time, four waves each) of a one- or two-slot class; lds_floats_per_wave as ever,
// the team's shared area after the four slices.
hipError_t launch_mc_team(McArgs a, int apl, int n_blocks, hipStream_t s) {
    const size_t lds = ((size_t)a.lds_floats_per_wave * kWavesPerBlock + team_floats(apl)) * sizeof(float);
    const dim3 grid(n_blocks), block(kWave * kWavesPerBlock);
    const bool direct = a.mode == kDirect;
    if (apl == 1 && !direct) hipLaunchKernelGGL((mc_kernel<1, kWave, 4, kGrid, true>), grid, block, lds, s, a);
    else if (apl == 1) hipLaunchKernelGGL((mc_kernel<1, kWave, 4, kDirect, true>), grid, block, lds, s, a);
    else if (apl == 2 && !direct) hipLaunchKernelGGL((mc_kernel<2, kWave, 3, kGrid, true>), grid, block, lds, s, a);
    else if (apl == 2) hipLaunchKernelGGL((mc_kernel<2, kWave, 3, kDirect, true>), grid, block, lds, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// waves: the most waves per SIMD the launch can keep resident (2, 4 or more). The one-slot whole-wave
// search runs the build held to that many: with few other waves to hide its latency behind, a chain is
// faster with fewer spills (128 chains, one wave each: 32.4 ligands/s on the six-wave build, 33.9 on the
// four-wave one). On maps the four-wave build serves two waves per SIMD too (it spills nothing); most such searches
// run on teams.
hipError_t launch_mc(McArgs a, int apl, int variant, int n_blocks, int waves, hipStream_t s) {
    if (variant != kMcWhole && apl != 1) return hipErrorInvalidValue;
    if (a.mode == kDirect) {  // whole waves at two or four waves per SIMD (one slot), as below otherwise
        if (variant != kMcWhole) return hipErrorInvalidValue;
        switch (apl) {
            case 1:
                return waves <= 2 ? launch_mc_t<1, kWave, 2, kDirect>(a, n_blocks, s)
                                  : launch_mc_t<1, kWave, 4, kDirect>(a, n_blocks, s);
            case 2: return launch_mc_t<2, kWave, 3, kDirect>(a, n_blocks, s);
            case 3: return launch_mc_t<3, kWave, 2, kDirect>(a, n_blocks, s);
            case 4: return launch_mc_t<4, kWave, 2, kDirect>(a, n_blocks, s);
            default: return hipErrorInvalidValue;
        }
    }
    switch (variant) {
        case kMcHalf4: return launch_mc_t<1, kTileNarrow, 4>(a, n_blocks, s);
        case kMcHalf3: return launch_mc_t<1, kTileNarrow, 3>(a, n_blocks, s);
        case kMcHalf2: return launch_mc_t<1, kTileNarrow, 2>(a, n_blocks, s);
        case kMcWhole: break;
        default: return hipErrorInvalidValue;
    }
    switch (apl) {
        case 1:
            return waves <= 4 ? launch_mc_t<1, kWave, 4>(a, n_blocks, s)
                              : launch_mc_t<1, kWave, 6>(a, n_blocks, s);
        case 2: return launch_mc_t<2, kWave, 3>(a, n_blocks, s);
        case 3: return launch_mc_t<3, kWave, 2>(a, n_blocks, s);
        case 4: return launch_mc_t<4, kWave, 2>(a, n_blocks, s);
        default: return hipErrorInvalidValue;
    }
}

template <int APL>
static hipError_t launch_opt_t(const OptArgs& a, hipStream_t s) {
    size_t lds = (size_t)a.lds_floats_per_wave * kWavesPerBlock * sizeof(float);
    int nb = (a.n_sel + kWavesPerBlock - 1) / kWavesPerBlock;
    if (a.mode == kDirect)
        hipLaunchKernelGGL((opt_kernel<APL, kDirect>), dim3(nb), dim3(kWave * kWavesPerBlock), lds, s, a);
    else
        hipLaunchKernelGGL((opt_kernel<APL, kGrid>), dim3(nb), dim3(kWave * kWavesPerBlock), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_opt(OptArgs a, int apl, hipStream_t s) {
    if (a.n_sel <= 0) return hipSuccess;
    switch (apl) {
        case 1: return launch_opt_t<1>(a, s);
        case 2: return launch_opt_t<2>(a, s);
        case 3: return launch_opt_t<3>(a, s);
        case 4: return launch_opt_t<4>(a, s);
        default: return hipErrorInvalidValue;
    }
}

template <int APL>
static hipError_t launch_posevec_t(const PoseVecArgs& a, int n_blocks, hipStream_t s) {
    size_t lds = (size_t)a.lds_floats_per_wave * kWavesPerBlock * sizeof(float);
    if (a.mode == kDirect)
        hipLaunchKernelGGL((posevec_kernel<APL, kDirect>), dim3(n_blocks), dim3(kWave * kWavesPerBlock), lds, s, a);
    else
        hipLaunchKernelGGL((posevec_kernel<APL, kGrid>), dim3(n_blocks), dim3(kWave * kWavesPerBlock), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_posevec(PoseVecArgs a, int apl, int n_blocks, hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    switch (apl) {
        case 1: return launch_posevec_t<1>(a, n_blocks, s);
        case 2: return launch_posevec_t<2>(a, n_blocks, s);
        case 3: return launch_posevec_t<3>(a, n_blocks, s);
        case 4: return launch_posevec_t<4>(a, n_blocks, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_cluster(const ClusterArgs& a, hipStream_t s) {
    if (a.n_lig <= 0) return hipSuccess;
    // up to 64 poses: a wave for every four of them
    int threads = kClusterThreads;
    if (a.nchain <= kWave) {
        threads = kWave;
        while (threads < 8 * kWave && threads / kWave * kClusterCand < a.nchain) threads *= 2;
    }
    hipLaunchKernelGGL(cluster_kernel, dim3(a.n_lig), dim3(threads), cluster_lds_bytes(a.nchain), s, a);
    return hipGetLastError();
}

template <int APL>
static hipError_t launch_score_t(const ScoreArgs& a, bool decomp, hipStream_t s) {
    int nb = (a.n_sel + kWavesPerBlock - 1) / kWavesPerBlock;
    if (decomp) hipLaunchKernelGGL((final_score_kernel<APL, true>), dim3(nb), dim3(kWave * kWavesPerBlock), 0, s, a);
    else hipLaunchKernelGGL((final_score_kernel<APL, false>), dim3(nb), dim3(kWave * kWavesPerBlock), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_final_score(const ScoreArgs& a, int apl, bool decomp, hipStream_t s) {
    if (a.n_sel <= 0) return hipSuccess;
    switch (apl) {
        case 1: return launch_score_t<1>(a, decomp, s);
        case 2: return launch_score_t<2>(a, decomp, s);
        case 3: return launch_score_t<3>(a, decomp, s);
        case 4: return launch_score_t<4>(a, decomp, s);
        default: return hipErrorInvalidValue;
    }
}

template <int APL, int TW, int OCC, int MODE = kGrid>
static int mc_occ(int lds_bytes) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, mc_kernel<APL, TW, OCC, MODE>, kWave * kWavesPerBlock, lds_bytes) !=
        hipSuccess)
        return 1;
    return nb > 0 ? nb : 1;
}

int mc_blocks_per_cu(int apl, int variant, int mode, int lds_bytes) {
    if (mode == kDirect) switch (apl) {
            case 1: return mc_occ<1, kWave, 4, kDirect>(lds_bytes);
            case 2: return mc_occ<2, kWave, 3, kDirect>(lds_bytes);
            case 3: return mc_occ<3, kWave, 2, kDirect>(lds_bytes);
            default: return mc_occ<4, kWave, 2, kDirect>(lds_bytes);
        }
    switch (variant) {
        case kMcHalf4: return mc_occ<1, kTileNarrow, 4>(lds_bytes);
        case kMcHalf3: return mc_occ<1, kTileNarrow, 3>(lds_bytes);
        case kMcHalf2: return mc_occ<1, kTileNarrow, 2>(lds_bytes);
        default: break;
    }
    switch (apl) {
        case 1: return mc_occ<1, kWave, 6>(lds_bytes);
        case 2: return mc_occ<2, kWave, 3>(lds_bytes);
        case 3: return mc_occ<3, kWave, 2>(lds_bytes);
        default: return mc_occ<4, kWave, 2>(lds_bytes);
    }
}

template <int APL>
static int pv_occ(int mode, int lds_bytes) {
    int nb = 0;
    const hipError_t e =
        mode == kDirect ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, posevec_kernel<APL, kDirect>,
                                                                       kWave * kWavesPerBlock, lds_bytes)
                        : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, posevec_kernel<APL, kGrid>,
                                                                       kWave * kWavesPerBlock, lds_bytes);
    return e == hipSuccess && nb > 0 ? nb : 1;
}

int posevec_blocks_per_cu(int apl, int mode, int lds_bytes) {
    switch (apl) {
        case 1: return pv_occ<1>(mode, lds_bytes);
        case 2: return pv_occ<2>(mode, lds_bytes);
        case 3: return pv_occ<3>(mode, lds_bytes);
        default: return pv_occ<4>(mode, lds_bytes);
    }
}

}  // namespace ud2
