// Internal structures shared by the host API (ud2_api.cpp) and the kernels
// (ud2_kernels.hip). Not part of the C-ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace ud2 {

constexpr int kWave = 64;
constexpr int kMaxApl = 4;                  // atoms per lane: natom <= 256
constexpr int kMaxAtoms = kWave * kMaxApl;  // pair records pack atom indices in 8 bits
constexpr int kMaxTors = 57;                // 7 + ntors <= 64: one pose-vector / BFGS component per lane
constexpr int kWavesPerBlock = 4;
constexpr int kXcds = 8;                    // blocks are dealt round the chip's XCDs, each with its own L2 cache
// The narrow tile of the MC search: two chains of a ligand per wave, one per 32 lanes, for ligands of
// at most kTileNarrow atoms and kTileNarrowTors torsions (every torsion step of a pose update staged
// in the tile's LDS, as a whole wave stages them, so both round alike).
constexpr int kTileNarrow = 32;
constexpr int kTileNarrowTors = 14;
// MC kernel variants: one chain per wave, or two per wave with an occupancy hint of 4, 3 or 2 waves
// per SIMD (the register budget the allocation is held to).
constexpr int kMcWhole = 0, kMcHalf4 = 1, kMcHalf3 = 2, kMcHalf2 = 3, kMcVariants = 4;
__host__ __device__ constexpr int mc_variant_tw(int v) { return v == kMcWhole ? kWave : kTileNarrow; }
// Queue heads of one MC search: one per variant of the one-atom-per-lane class, one per wider class.
constexpr int kMcHeads = kMcVariants + kMaxApl - 1;
constexpr int kNumTypes = 21;

// A pair's flag terms as two constants of eval_ramps: kh is 1.5 for a hydrophobic pair, else so low that the
// hydrophobic ramp clamp(kh - d) is zero at any distance; kb is -1 / 0.7 for a hydrogen-bond pair,
// else 0, and the ramp clamp(kb d) with it.
constexpr float kRampHyd = 1.5f, kRampNone = -1e30f, kRampHb = -(1.0f / 0.7f);
constexpr float kRampNoPair = 4.0f;  // kh of a lane that scores no pair (packed steps)
__host__ __device__ constexpr float ramp_hyd(int flags) { return (flags & 1) ? kRampHyd : kRampNone; }
__host__ __device__ constexpr float ramp_hb(int flags) { return (flags & 2) ? kRampHb : 0.0f; }

// A receptor atom's vdW radius and type flags in one word: the radius is in [1, 4), so its bits less
// those of 1.0 take 24 bits; the doubled flags (as pair_lut takes them) take the bits above.
constexpr uint32_t atom_word(uint32_t radius_bits, uint32_t flags) {
    return (radius_bits - 0x3F800000u) | (2 * flags) << 24;
}

// One ligand of a ligand set on the device.
struct DevLig {
    int32_t natom, ntors, npair, nheavy;
    int32_t atom_off;   // into atom_x0 (atoms)
    int32_t tors_off;   // into tors_* (torsions)
    int32_t pair_off;   // into pairs
    int32_t apl;        // ceil(natom / 64)
    int32_t leaf_first; // 1: the torsions have a leaf-first application order (tors_axis .y >> 16)
    int32_t fold_off;   // into fold_mask
    int32_t nfold;      // natom / 2 folded pair diagonals, apl mask words each
    int32_t pack_off;   // into pack (steps of 64 lanes)
    int32_t npack;      // pair steps of its table (LigSetDev::pack; ligands of at most 64 atoms)
};

// Device view of a ligand set.
struct LigSetDev {
    const DevLig* ligs;
    const float4* atom_x0;                 // x, y, z, type (int bits)
    const int2* tors_axis;                 // (from | rank << 16, to | order << 16); entry t's order = the torsion
                                           // applied t-th, leaf first; its rank = when torsion t is applied
    const float* tors_dihe0;               // input dihedral (radians)
    const int2* tors_range;                // (global offset into ranges, count)
    const float2* ranges;                  // (lo, hi) radians
    const unsigned long long* tors_mask;   // [ntors_total][kMaxApl] rotated-atom bit masks
    const uint2* pairs;                    // {i | j << 8 | hyd << 16 | hbond << 17, bits of R_i + R_j}
    // Folded pair diagonals: for d = 1 .. natom / 2, apl words per diagonal; bit a % 64 of word
    // (d - 1) * apl + a / 64 is set when the pair {a, (a + d) mod natom} is a scored (heavy) intra
    // pair (for even natom, diagonal natom / 2 only for atoms below natom / 2, so every pair
    // appears once).
    const unsigned long long* fold_mask;
    // Pair steps of the one-atom-per-lane ligands, one entry per lane and step. Lane l scores the pair {i, j}
    // (gradient +p on i, -p on j) of .x = 16 i | 16 j << 16 (their LDS offsets), with the flag constants
    // kh = .z and kb = .w (ramp_hyd, ramp_hb; kh = kRampNoPair: no pair), and collects the p of the lanes
    // whose byte offsets 4 * lane .y holds.
    // 33-64 atoms: up to 63 pairs per step in any order, lanes 0 .. 62; every atom is i of at most two and j of at
    // most two: bytes 0-1 of .y the lanes where atom l is i, bytes 2-3 those where it is j, lane 63, which
    // scores nothing, for none.
    // Up to 32 atoms: the folded diagonals 2 s + 1 (lanes 0-31) and 2 s + 2 (lanes 32-63) in step s, i the lane mod
    // 32 and .x = 16 j; bytes 0-1 of .y the two lanes where atom l is j.
    const uint4* pack;
    // Bias sites (FlexParamVina::inds_bias / params_bias, E/src/cuda/task.cu:157-168)
    // and the task options that change the search (DockParam, E/src/model/model.h:151-168).
    const int32_t* bias_start;             // [atoms + 1] CSR over the set's atoms; null: no sites
    const float4* bias_site;               // x, y, z, V (well depth, or affinity for align)
    const float* bias_r2;                  // Gaussian width r2 of each site (pos)
    int32_t bias_type;                     // 0 no, 1 pos, 2 align (BiasType, model.h:145-149)
    float bias_k;                          // scale of V
    int32_t constraint;                    // constraint docking: no rigid degrees of freedom
};

// Device view of a scene: receptor, box and (optional) grid maps.
struct SceneDev {
    const float4* rec;  // [nrec + 1] heavy receptor atoms: x, y, z, atom_word; the last one means nothing
    int32_t nrec;
    float box_lo[3], box_hi[3];
    const float4* cells;  // maps cell-major: [slot][cz][cy][cx] x {c000 c100 c010 c110}, {c001 c101 c011 c111}
    int32_t gn[3];
    float gorigin[3];
    float gspacing, ginv;
    const int32_t* slot_tab;  // [kNumTypes] map of each XS type (-1 = none), device memory
    // Reach lists of the direct sum: the space around the box in cells of edge 1 / rinv from rorigin, and per
    // cell the receptor atoms that a point in it can have within the cutoff, in receptor order: entries
    // reach_off[cell].x .. reach_off[cell].y of reach (as rec), their number padded to a
    // multiple of 4 with atoms out of any reach. Beyond rec_lo .. rec_hi no receptor atom is in reach.
    const float4* reach;
    const int2* reach_off;
    int32_t rn[3];
    float rorigin[3], rinv;
    float rec_lo[3], rec_hi[3];
};

// Pose buffers of a ligand set with nchain poses per ligand, laid out by
// ligand: x at (atom_off * nchain + chain * natom) * 3, dihedrals at
// tors_off * nchain + chain * ntors, centre / rot_vec at (lig * nchain + chain) * 3,
// energy at lig * nchain + chain.
struct PoseBufs {
    float* x;
    float* c;
    float* rv;
    float* dihe;
    float* e;
    int32_t nchain;
};

enum InterMode : int32_t { kDirect = 0, kGrid = 1 };

// What the arguments of every kernel that works on poses begin with.
struct ArgHead {
    LigSetDev L;
    SceneDev S;
};

struct McArgs {
    LigSetDev L;
    SceneDev S;
    PoseBufs P;
    const int32_t* order;  // ligands in the work order of this launch
    int32_t n_order;
    int32_t* counter;      // work-queue head, zero at launch
    int32_t mode;
    int32_t mc_steps, opt_steps, randomize;
    uint32_t seed;
    int32_t lig_index_base;
    int32_t lds_floats_per_wave;
    int32_t hdim_ld;       // leading dimension of the per-wave Hessian (odd)
    unsigned long long* stats;  // optional: evals, gather bytes, pair evals, chains
};

constexpr int kOptFew = 64;  // selections up to this long travel with the kernel's arguments
struct OptArgs {
    LigSetDev L;
    SceneDev S;
    PoseBufs P;
    const int32_t* sel;  // selected poses: lig * nchain + chain (null: they are in few)
    const int32_t* pos;  // output slot of each selected pose
    int32_t n_sel;
    int32_t mode;
    int32_t max_steps;
    float v_cap, slope;
    int32_t lds_floats_per_wave;
    int32_t hdim_ld;
    float* out_e;   // energy of each selected pose (may be null)
    float* out_g;   // [n_sel][64] gradient (may be null)
    const float* dir;   // [n_sel][64] update direction (pose-update hook)
    float alpha;
    int32_t op;     // 0 BFGS, 1 energy+gradient, 2 pose update, 3 line search from H = I, 4 reset
    int32_t few[kOptFew], few_pos[kOptFew];  // a short selection and its output slots
};

struct PoseVecArgs {
    LigSetDev L;
    SceneDev S;
    int32_t lig;
    int64_t n;
    const float* pv;   // [n][7 + ntors]
    float* e;          // [n]
    float* g;          // [n][6 + ntors]
    float v_cap, slope;
    int32_t mode;
    int32_t lds_floats_per_wave;
    int32_t hdim_ld;   // sizes the torsion table (>= 6 + ntors)
};

struct ClusterArgs {
    LigSetDev L;
    const float* x;
    const float* e;
    int32_t nchain;
    int32_t n_lig;
    float limit;
    int32_t* leaders;   // [n_lig][nchain]
    int32_t* nleaders;  // [n_lig]
};

// 32-bit words of the clustering kernel's first LDS array (one per pose, an even number of them), and the bytes of all:
// that, a bit per rank, and two 16-bit indices per pose.
__host__ __device__ constexpr size_t cluster_near_words(int nchain) { return size_t(nchain + 1) & ~size_t(1); }
__host__ __device__ constexpr size_t cluster_lds_bytes(int nchain) {
    return cluster_near_words(nchain) * sizeof(uint32_t) + size_t((nchain + kWave - 1) / kWave) * sizeof(uint64_t) +
           2 * size_t(nchain) * sizeof(uint16_t);
}
constexpr int kClusterMaxPoses = 8192;
static_assert(kClusterMaxPoses <= 65536 && cluster_lds_bytes(kClusterMaxPoses) <= 160 * 1024,
              "a ligand's poses are ranked in 16 bits, in the LDS of one block");

struct ScoreArgs {
    LigSetDev L;
    SceneDev S;
    const float* x;
    int32_t nchain;
    const int32_t* sel;
    int32_t n_sel;
    float* out4;          // [n_sel][4]: intra, inter, penalty, bias (may be null)
    float* decomp;        // [n_sel][decomp_stride][5] per-atom inter terms (decomposition launch)
    int32_t decomp_stride;
};

// Reach lists (SceneDev::reach): every cell's place among the entries (fill false), or the entries.
struct ReachArgs {
    const float4* rec;
    int32_t nrec;
    int32_t rn[3];
    float rorigin[3], edge;
    int2* off;                  // [cells]
    unsigned long long* total;  // entries of all lists, zero at first
    float4* reach;
};
constexpr int kReachPad = 4;  // a list's length is a multiple of this

struct GridArgs {
    SceneDev S;
    // the maps in order of their probe radius
    float radius[kNumTypes];
    uint32_t lut[kNumTypes];     // pair flags with a partner of doubled type flags f: (lut >> f) & 3
    int32_t slot[kNumTypes];     // place in maps
    int32_t nslot;
    float* maps;
};

// Cell-major copy of the maps (SceneDev::cells): the 8 corners of a grid cell are one
// aligned 32-byte sector, so a trilinear gather reads two float4 instead of 8 scattered floats.
struct BrickArgs {
    const float* maps;  // [nslot][nz][ny][nx]
    float4* cells;      // [nslot][nz-1][ny-1][nx-1][2]
    int32_t gn[3];
    int32_t nslot;
};

// ---------------------------------------------------------- learned proposal
constexpr int kFeat = 80;     // network inputs of one candidate
constexpr int kPooled = 64;   // 8 feature classes x 8 statistics
constexpr int kHidden = 256;
constexpr int kGroup = 16;    // candidates of one MC state = MFMA tile width
constexpr int kA1Stride = kHidden + 8;  // bf16 per staged hidden row; padding spreads rows over the LDS banks
constexpr int kMaxCand = 16;
constexpr int kMlpNParam = kFeat * kHidden + kHidden + kHidden * kHidden + kHidden + kHidden + 1;
constexpr int kMlpNNorm = 2 * kFeat;
// canonical parameter offsets: W1[80][256], b1, W2[256][256], b2, w3, b3; then mu[80], inv_sigma[80]
constexpr int kOffW1 = 0, kOffB1 = kFeat * kHidden, kOffW2 = kOffB1 + kHidden, kOffB2 = kOffW2 + kHidden * kHidden,
              kOffW3 = kOffB2 + kHidden, kOffB3 = kOffW3 + kHidden;

// Place of A[row][k] of a weight matrix in its fragments of 16 rows by 16 or 32 k, nk fragments along k: lane l of a
// fragment holds row l % 16 and the 4 or 8 k from 4 (l / 16) or 8 (l / 16) on.
__host__ __device__ constexpr int frag16(int row, int k, int nk) {
    return ((row / 16 * nk + k / 16) * kWave + 16 * (k % 16 / 4) + row % 16) * 4 + k % 4;
}
__host__ __device__ constexpr int frag32(int row, int k, int nk) {
    return ((row / 16 * nk + k / 32) * kWave + 16 * (k % 32 / 8) + row % 16) * 8 + k % 8;
}

// Device copies of the network used by the MFMA kernels.
struct MlpDev {
    // bf16 weights as A operands, fragment by fragment: the 64 lanes' values of one MFMA lie together, in the
    // order of the lanes (frag16, frag32), so that a wave's load is 512 or 1,024 consecutive bytes
    const uint16_t* w1;   // [16 tiles][5 K blocks] 16x16x16 fragments of W1 transposed (rows: hidden units)
    const uint16_t* w1s;  // [16][3] 16x16x32 fragments of it, zero past feature 79 (scoring)
    const uint16_t* w2t;  // [16][16] 16x16x16 fragments of W2 transposed (rows: out-units)
    const uint16_t* w2s;  // [16][8] 16x16x32 fragments of it, the in-units in the K = 32 order (k32_slot) (scoring)
    const uint16_t* w2;   // [16][16] 16x16x16 fragments of W2 (rows: in-units) (backward)
    const float* b1;      // [256]
    const float* b2;      // [256]
    const float* w3;      // [256], values rounded to bf16
    const float* b3;      // [1]
    const float* mu;      // [80]
    const float* inv_sigma;  // [80]
};

// Training buffers of one minibatch of n_groups groups (rows = 16 * n_groups).
struct MlpTrain {
    const uint16_t* x;       // dataset features [*][80]
    const int32_t* groups;   // dataset group of each minibatch group (null: identity)
    int32_t n_groups;
    const float* label;      // dataset labels [*], for the loss
    const float* dy;         // [rows] d loss / d y_hat; null: of the loss
    // operands of the weight-gradient GEMMs in bf16: 16x16x16 fragments [tiles of 16 units][groups] with the units as
    // rows and the group's 16 candidates as k (frag16)
    uint16_t* xn;            // normalised inputs, 5 tiles
    uint16_t* a1;            // 16 tiles each
    uint16_t* dz1;
    uint16_t* dz2;
    float* part;             // [n_groups][kPartStride]: partial sums of dw3, db2, db1, db3 and the loss
};
constexpr int kPartStride = 3 * kHidden + 16;  // whole blocks of 16 sums
constexpr int kGradW = kFeat * kHidden + kHidden * kHidden;  // weights with GEMM gradients: W1, then W2

constexpr int kW1sSize = kHidden * 96;  // W1's 16x16x32 fragments: three K blocks

// bf16 copies of the weights that an update writes (MlpDev).
struct MlpPack {
    uint16_t *w1, *w1s, *w2t, *w2s, *w2;
    float* w3r;
};

// Adam's state and settings, and where the loss goes (may be null).
struct MlpAdam {
    float *p, *m, *v;
    float lr, beta1, beta2, eps, c1, c2;
    float* loss;
    float loss_scale;
};

enum LmcPolicy : int32_t { kPolicyPlain = 0, kPolicyExact = 1, kPolicyLearned = 2, kPolicyCollect = 3 };

// Persistent learned-proposal MC over the chains of one launch class.
struct LmcArgs {
    LigSetDev L;
    SceneDev S;
    PoseBufs P;              // best pose of each chain (the result)
    const int32_t* order;
    int32_t n_order;
    int32_t* counter;        // work-queue head, zero at launch
    int32_t mode;            // inter term of the search energy
    int32_t mc_steps, opt_steps, randomize;
    uint32_t seed;
    int32_t lig_index_base;
    int32_t lds_floats_per_wave;
    int32_t hdim_ld;
    int32_t lscr, lfeat;       // feature scratch, candidate rows (floats from the slice start)
    int32_t la1, la1b, a1_split;  // hidden layer: rows below a1_split at la1, the others at la1b
    int32_t a1_rows;         // hidden rows staged: 8 when at most 8 candidates / starts are scored, else 16
    int32_t policy, n_cand, top_k;
    float sel_temp;          // learned: > 0 draws one candidate with p ~ exp(-score / sel_temp)
    int32_t n_start;         // > 1: randomised starts per chain, the best kept (network or exact energy)
    MlpDev W;
    int64_t n_pose;
    uint16_t* collect_x;     // collect: [mc_steps][n_pose][16][80] features
    float* collect_y;        // collect: [mc_steps][n_pose][16] energies after BFGS
    float* collect_e0;       // collect (optional): [mc_steps][n_pose][16] energies before BFGS
    unsigned long long* stats;
};

struct FeatArgs {
    LigSetDev L;
    SceneDev S;
    PoseBufs P;
    const int32_t* sel;
    int32_t n_sel;
    uint16_t* x;             // [n_sel][80]
    int32_t lds_floats_per_wave;
    int32_t hdim_ld;         // sizes the torsion table (>= 6 + ntors of every selected ligand)
};

template <class T>
constexpr bool begins_with_head() { return offsetof(T, L) == offsetof(ArgHead, L) && offsetof(T, S) == offsetof(ArgHead, S); }
static_assert(begins_with_head<McArgs>() && begins_with_head<OptArgs>() && begins_with_head<PoseVecArgs>() &&
                  begins_with_head<LmcArgs>() && begins_with_head<FeatArgs>(),
              "kernels read the ligand set and the scene through ArgHead");

// Launchers (ud2_kernels.hip); each returns a hipError_t.
hipError_t launch_grid_build(const GridArgs& a, hipStream_t s);
hipError_t launch_brick(const BrickArgs& a, hipStream_t s);
hipError_t launch_reach(const ReachArgs& a, bool fill, hipStream_t s);
constexpr int kProbePerThread = 16;  // gathers per thread of the gather probe
hipError_t launch_gather_probe(const float4* cells, uint32_t span, uint32_t seed, float* out, int64_t n_threads,
                               hipStream_t s);
hipError_t launch_valu_probe(float* out, int iters, int64_t n_threads, hipStream_t s);
hipError_t launch_mc(McArgs a, int apl, int variant, int n_blocks, int waves, hipStream_t s);
hipError_t launch_mc_team(McArgs a, int apl, int n_blocks, hipStream_t s);
hipError_t launch_opt(OptArgs a, int apl, hipStream_t s);
hipError_t launch_posevec(PoseVecArgs a, int apl, int n_blocks, hipStream_t s);
hipError_t launch_cluster(const ClusterArgs& a, hipStream_t s);
hipError_t launch_final_score(const ScoreArgs& a, int apl, bool decomp, hipStream_t s);
hipError_t launch_pack_diagonals(const LigSetDev& L, int n_lig, uint4* pack, hipStream_t s);
hipError_t launch_fill_i32(int32_t* p, int32_t v, int64_t n, hipStream_t s);
int mc_blocks_per_cu(int apl, int variant, int mode, int lds_bytes_per_block);
// LDS floats of a wave slice before its torsion table: coordinates + pair forces (7 * 64 * apl) and two
// parked poses (64 * (3 * apl + 1) + 8 each), lds_flags_offset; a multiple of 4, so the table after it
// stays 16-byte aligned. A tile of tw < 64 lanes (one chain of a wave that runs 64 / tw chains) has the
// same layout with tw in place of 64.
__host__ __device__ constexpr int lds_flags_offset(int apl, int tw = kWave) { return 7 * tw * apl + 2 * (tw * (3 * apl + 1) + 8); }
// ... and then each atom's doubled type flags (one int per atom slot, tw * apl)
__host__ __device__ constexpr int lds_fixed_floats(int apl, int tw = kWave) { return lds_flags_offset(apl, tw) + tw * apl; }
// Torsion table of the wave's ligand, filled once per work item: per torsion {from | to << 16,
// number of allowed ranges, first range lo, hi} and the rotated-atom mask word pairs of each
// atom slot, padded to 16 bytes. ld (the Hessian's leading dimension) >= 6 + ntors sizes it.
__host__ __device__ constexpr int tors_entry_floats(int apl) { return apl <= 2 ? 8 : 12; }
__host__ __device__ constexpr int lds_tors_floats(int apl, int ld) { return (ld > 6 ? ld - 6 : 0) * tors_entry_floats(apl); }
// LDS floats of a wave (or tile) slice before its Hessian tile (or feature scratch).
__host__ __device__ constexpr int lds_head_floats(int apl, int ld, int tw = kWave) {
    return lds_fixed_floats(apl, tw) + lds_tors_floats(apl, ld);
}
// Shared area of a block whose four waves run one chain, after their slices (Team).
__host__ __device__ constexpr int team_floats(int apl) { return 12 + kWave * (3 * apl + 2) + 8; }
// Per-wave slices are rounded to 4 floats so every slice starts 16-byte aligned.
__host__ __device__ constexpr int lds_round4(int n) { return (n + 3) & ~3; }
int posevec_blocks_per_cu(int apl, int mode, int lds_bytes_per_block);
// LDS floats per wave of the features kernel: the head and 8 floats per atom of feature scratch.
__host__ __device__ constexpr int lds_prop_floats(int apl, int ld) { return lds_head_floats(apl, ld) + 8 * kWave * apl; }

// Learned proposal (ud2_learned.hip) and network (ud2_mlp.hip) launchers.
hipError_t launch_lmc(LmcArgs a, int apl, int n_blocks, hipStream_t s);
hipError_t launch_features(FeatArgs a, int apl, hipStream_t s);
int lmc_blocks_per_cu(int apl, int policy, int mode, int lds_bytes_per_block);
hipError_t launch_mlp_forward(const MlpDev& W, const uint16_t* x, const int32_t* groups, int64_t n_groups, float* y,
                              hipStream_t s);
hipError_t launch_mlp_train(const MlpDev& W, const MlpTrain& T, int splits, float* gpart, hipStream_t s);
hipError_t launch_mlp_update(const float* gpart, int splits, const float* part, int n_groups, float* grad,
                             const MlpAdam& O, const MlpPack& D, hipStream_t s);
hipError_t launch_mlp_pack(const float* params, const MlpPack& D, hipStream_t s);

}  // namespace ud2
