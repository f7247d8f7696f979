// Host side of libud2.so: the C ABI declared in include/ud2.h.
//
// Owns the device copies of the receptor / grid maps (ud2_scene) and of a
// batch of ligand topologies (ud2_ligset), validates every input before a
// kernel sees it, and launches the kernels of ud2_kernels.hip. Errors become
// return codes with a per-thread message; nothing throws across the ABI.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <functional>
#include <mutex>
#include <numeric>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/ud2.h"
#include "ud2_internal.h"

using namespace ud2;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define UD2_HIP(call)                                                                                  \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess) return fail(UD2_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

const float kVdwHost[kNumTypes] = {1.1f, 1.92f, 1.9f, 1.9f, 1.8f, 1.8f, 1.8f, 1.8f, 1.7f, 1.7f, 1.7f,
                                   1.7f, 1.5f, 2.2f, 2.1f, 2.0f, 1.8f, 2.0f, 2.2f, 2.3f, 1.2f};
const int kFlagsHost[kNumTypes] = {0, 0, 1, 0, 0, 4, 2, 6, 0, 4, 2, 6, 1, 0, 0, 0, 1, 1, 1, 0, 4};

int pair_flags_host(int ti, int tj) {
    int a = kFlagsHost[ti], b = kFlagsHost[tj];
    int hyd = a & b & 1;
    int hb = (((a >> 1) & (b >> 2)) | ((a >> 2) & (b >> 1))) & 1;
    return hyd | (hb << 1);
}

// pair_lut of an atom type: its pair flags with a partner of flags b at bits 2 b.
uint32_t pair_lut_host(int type) {
    const int a = kFlagsHost[type];
    uint32_t t = 0;
    for (int b = 0; b < 8; b++) {
        const int hb = (((a >> 1) & (b >> 2)) | ((a >> 2) & (b >> 1))) & 1;
        t |= uint32_t((a & b & 1) | (hb << 1)) << (2 * b);
    }
    return t;
}

uint32_t float_bits(float v) {
    uint32_t u;
    std::memcpy(&u, &v, sizeof(u));
    return u;
}

// Entry of a lane without a pair, and a pair's part of an entry (LigSetDev::pack).
const uint4 kNoPair = make_uint4(0u, 0u, float_bits(kRampNoPair), 0u);
void set_pair(uint4& t, int i, int j, const int32_t* types) {
    const int fl = pair_flags_host(types[i], types[j]);
    t.x = uint32_t(16 * i) | (uint32_t(16 * j) << 16);
    t.z = float_bits(ramp_hyd(fl));
    t.w = float_bits(ramp_hb(fl));
}

// Packed pair steps of a ligand of 33-64 atoms (LigSetDev::pack). Each step holds at most 63 pairs,
// one per lane, with every atom i (gradient +p) of at most two of them and j (-p) of at most two, so
// an atom collects its shares with four lane reads. Greedy first fit, the pairs of the busiest atoms
// first, each pair in the first step where either orientation fits. Appends the steps' entries and
// returns their number, or -1 if the steps do not cover the pairs.
int pack_pairs(int na, const std::vector<std::pair<int, int>>& pl, const int32_t* types, std::vector<uint4>& pack) {
    constexpr int kSlots = 2, kLanes = kWave - 1, kNone = kLanes * 4;
    std::vector<int> deg(na, 0);
    for (auto& ij : pl) {
        deg[ij.first]++;
        deg[ij.second]++;
    }
    std::vector<int> order(pl.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int c) {
        return deg[pl[a].first] + deg[pl[a].second] > deg[pl[c].first] + deg[pl[c].second];
    });
    struct Step {
        std::vector<std::pair<int, int>> lanes;  // (i, j) per lane
        std::vector<int> as_i, as_j;
    };
    std::vector<Step> steps;
    for (int k : order) {
        const int a = pl[k].first, c = pl[k].second;
        bool placed = false;
        for (Step& st : steps) {
            if (int(st.lanes.size()) >= kLanes) continue;
            for (int o = 0; o < 2 && !placed; o++) {
                const int i = o ? c : a, j = o ? a : c;
                if (st.as_i[i] < kSlots && st.as_j[j] < kSlots) {
                    st.lanes.push_back({i, j});
                    st.as_i[i]++;
                    st.as_j[j]++;
                    placed = true;
                }
            }
            if (placed) break;
        }
        if (!placed) {
            Step st;
            st.as_i.assign(na, 0);
            st.as_j.assign(na, 0);
            st.lanes.push_back({a, c});
            st.as_i[a]++;
            st.as_j[c]++;
            steps.push_back(std::move(st));
        }
    }
    size_t covered = 0;
    for (const Step& st : steps) {
        uint32_t src_i[kWave] = {}, src_j[kWave] = {};
        int ni[kWave] = {}, nj[kWave] = {};
        const size_t base = pack.size();
        pack.resize(base + kWave, kNoPair);
        for (int l = 0; l < int(st.lanes.size()); l++) {
            const int i = st.lanes[l].first, j = st.lanes[l].second;
            set_pair(pack[base + l], i, j, types);
            src_i[i] |= uint32_t(4 * l) << (8 * ni[i]++);
            src_j[j] |= uint32_t(4 * l) << (8 * nj[j]++);
            covered++;
        }
        for (int a = 0; a < kWave; a++) {
            for (int k = ni[a]; k < kSlots; k++) src_i[a] |= uint32_t(kNone) << (8 * k);
            for (int k = nj[a]; k < kSlots; k++) src_j[a] |= uint32_t(kNone) << (8 * k);
            pack[base + a].y = src_i[a] | (src_j[a] << 16);
        }
    }
    return covered == pl.size() ? int(steps.size()) : -1;
}

template <class T>
int upload(T** d, const std::vector<T>& h) {
    size_t n = std::max<size_t>(h.size(), 1);
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(d), n * sizeof(T)));
    if (!h.empty()) UD2_HIP(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return UD2_OK;
}

int n_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    return n;
}

int odd_ld(int dim) { return (dim % 2 == 1) ? dim : dim + 1; }

// ------------------------------------------------------------ tile tuning
// Which MC kernel variant (kMcWhole: one chain per wave; kMcHalf4 / 3 / 2: two chains per wave on
// 32-lane tiles, at an occupancy hint of 4, 3 or 2 waves per SIMD) runs a one-atom-per-lane ligand,
// by (natom, ntors) bucket: natom 1-8, 9-16, 17-24, 25-32 by ntors 0-3, 4-7, 8-11, 12-14.
// Ligands past those sizes always run one chain per wave. The table starts with every bucket on
// kMcWhole (on MI355X two chains per wave measured slower for every bucket of the 1,024-ligand
// screening batch: the chains' line searches, acceptances and refinements diverge, and the
// per-chain values that a whole wave keeps in scalar registers take vector registers) and is
// replaced by ud2_autotune's measurements; the policy can force a variant.
constexpr int kTuneAtomBuckets = 4, kTuneTorsBuckets = 4;
constexpr int kTuneBuckets = kTuneAtomBuckets * kTuneTorsBuckets;
static_assert(kTuneBuckets == UD2_TUNE_BUCKETS && kMcVariants == UD2_MC_VARIANTS, "tuning table sizes");

struct TuneState {
    std::mutex mu;
    int policy = UD2_TILE_AUTO;
    int forced = kMcHalf4;               // the half-wave variant UD2_TILE_ALWAYS runs
    int8_t variant[kTuneBuckets];
    float ms[kTuneBuckets][kMcVariants];  // probe search time per variant; -1 unmeasured
    std::atomic<int64_t> version{1};
    TuneState() {
        for (int b = 0; b < kTuneBuckets; b++) {
            variant[b] = kMcWhole;
            for (int v = 0; v < kMcVariants; v++) ms[b][v] = -1.0f;
        }
    }
};
TuneState g_tune;

// Bucket of a ligand that can run on a 32-lane tile, else -1.
int tune_bucket(int natom, int ntors) {
    if (natom < 1 || natom > kTileNarrow || ntors < 0 || ntors > kTileNarrowTors) return -1;
    return ((natom - 1) / 8) * kTuneTorsBuckets + std::min(ntors / 4, kTuneTorsBuckets - 1);
}

int mc_variant(const DevLig& d, int policy, int forced, const int8_t* table) {
    const int b = d.apl == 1 ? tune_bucket(d.natom, d.ntors) : -1;
    if (b < 0 || policy == UD2_TILE_NEVER) return kMcWhole;
    return policy == UD2_TILE_ALWAYS ? forced : table[b];
}

}  // namespace

namespace ud2 {
int set_error(int code, const std::string& msg) { return fail(code, msg); }
}  // namespace ud2

struct ud2_scene {
    int device = 0;
    float4* d_rec = nullptr;  // [nrec + 1]
    int32_t nrec = 0;
    float box_lo[3], box_hi[3];
    float* d_maps = nullptr;     // [types][nz][ny][nx]
    float4* d_cells = nullptr;   // cell-major copy the kernels gather from
    int32_t gn[3] = {0, 0, 0};
    float gorigin[3] = {0, 0, 0};
    float gspacing = 0;
    std::vector<int32_t> probe_types;
    int32_t slot_of_type[kNumTypes];
    int32_t* d_slot = nullptr;
    // reach lists of the direct sum (SceneDev::reach)
    float4* d_reach = nullptr;
    int2* d_reach_off = nullptr;
    int64_t reach_bytes = 0;
    int32_t rn[3] = {0, 0, 0};
    float rorigin[3] = {0, 0, 0}, redge = 1.0f;
    float rec_lo[3], rec_hi[3];

    SceneDev view() const {
        SceneDev s;
        s.rec = d_rec;
        s.nrec = nrec;
        for (int d = 0; d < 3; d++) {
            s.box_lo[d] = box_lo[d];
            s.box_hi[d] = box_hi[d];
            s.gn[d] = gn[d];
            s.gorigin[d] = gorigin[d];
            s.rn[d] = rn[d];
            s.rorigin[d] = rorigin[d];
            s.rec_lo[d] = rec_lo[d];
            s.rec_hi[d] = rec_hi[d];
        }
        s.reach = d_reach;
        s.reach_off = d_reach_off;
        s.rinv = 1.0f / redge;
        s.cells = d_cells;
        s.gspacing = gspacing;
        s.ginv = gspacing > 0 ? 1.0f / gspacing : 0.0f;
        s.slot_tab = d_slot;
        return s;
    }
};

struct ud2_ligset {
    int device = 0;
    int32_t n_lig = 0;
    std::vector<DevLig> h_ligs;
    std::vector<uint8_t> has_slot_type;  // union of heavy ligand types, per XS type
    DevLig* d_ligs = nullptr;
    float4* d_x0 = nullptr;
    int2* d_axis = nullptr;
    float* d_dihe0 = nullptr;
    int2* d_trange = nullptr;
    float2* d_ranges = nullptr;
    unsigned long long* d_mask = nullptr;
    uint2* d_pairs = nullptr;
    unsigned long long* d_fold = nullptr;
    uint4* d_pack = nullptr;
    int32_t* d_counter = nullptr;
    // Work order of the persistent search launches, fixed at creation: ligands by atoms-per-lane
    // class (widest first), within a class most expensive first, so each launch's tail holds the
    // cheapest chains. Class apl occupies order[cls_pos[apl] .. cls_pos[apl] + cls_cnt[apl]);
    // cls_dmax[apl] is its largest 6 + ntors.
    std::vector<int32_t> h_order;
    int32_t* d_order = nullptr;
    int32_t cls_pos[kMaxApl + 1] = {0}, cls_cnt[kMaxApl + 1] = {0}, cls_dmax[kMaxApl + 1] = {0};
    double load = 0.0;  // work of the set's ligands in units of the costliest one's
    // The one-atom-per-lane class split for the MC search by kernel variant: part v (the ligands
    // that variant v runs, in the work order above) at split[part_pos[v] .. + part_cnt[v]), its
    // largest 6 + ntors part_dmax[v]. Rebuilt when the tile policy or table changes (split_version).
    mutable std::vector<int32_t> h_split;
    int32_t* d_split = nullptr;
    mutable int32_t part_pos[kMcVariants] = {0}, part_cnt[kMcVariants] = {0}, part_dmax[kMcVariants] = {0};
    mutable int64_t split_version = 0;
    mutable bool split_forced = false;  // by UD2_TILE_ALWAYS
    int32_t* d_sel_all = nullptr; // scratch for all-pose selections
    int64_t sel_all_cap = 0;
    int32_t* d_bias_start = nullptr;  // [atoms + 1], null without sites
    float4* d_bias_site = nullptr;
    float* d_bias_r2 = nullptr;
    int32_t bias_type = 0;
    float bias_k = 0.1f;
    int32_t constraint = 0;

    LigSetDev view() const {
        LigSetDev v;
        v.ligs = d_ligs;
        v.atom_x0 = d_x0;
        v.tors_axis = d_axis;
        v.tors_dihe0 = d_dihe0;
        v.tors_range = d_trange;
        v.ranges = d_ranges;
        v.tors_mask = d_mask;
        v.pairs = d_pairs;
        v.fold_mask = d_fold;
        v.pack = d_pack;
        v.bias_start = d_bias_start;
        v.bias_site = d_bias_site;
        v.bias_r2 = d_bias_r2;
        v.bias_type = bias_type;
        v.bias_k = bias_k;
        v.constraint = constraint;
        return v;
    }
    int max_apl() const {
        int m = 1;
        for (auto& l : h_ligs) m = std::max(m, int(l.apl));
        return m;
    }
    int max_dim() const {
        int m = 6;
        for (auto& l : h_ligs) m = std::max(m, 6 + int(l.ntors));
        return m;
    }
};

namespace {

// Rebuilds the set's tile split when the tile policy or table changed since it was last built: a host
// copy on stream st, which is then synchronised (the host vector is the copy's source).
int refresh_split(const ud2_ligset* ls, hipStream_t st) {
    int policy = 0, forced = 0;
    int8_t table[kTuneBuckets];
    int64_t version = 0;
    {
        std::lock_guard<std::mutex> lock(g_tune.mu);
        version = g_tune.version.load();
        if (ls->split_version == version) return UD2_OK;
        policy = g_tune.policy;
        forced = g_tune.forced;
        std::memcpy(table, g_tune.variant, sizeof(table));
    }
    const int pos = ls->cls_pos[1], cnt = ls->cls_cnt[1];
    std::vector<int32_t> part[kMcVariants];
    int dmax[kMcVariants] = {0};
    for (int k = pos; k < pos + cnt; k++) {
        const int l = ls->h_order[k];
        const DevLig& d = ls->h_ligs[l];
        const int v = mc_variant(d, policy, forced, table);
        part[v].push_back(l);
        dmax[v] = std::max(dmax[v], 6 + int(d.ntors));
    }
    ls->h_split.clear();
    for (int v = 0; v < kMcVariants; v++) {
        ls->part_pos[v] = int32_t(ls->h_split.size());
        ls->part_cnt[v] = int32_t(part[v].size());
        ls->part_dmax[v] = dmax[v];
        ls->h_split.insert(ls->h_split.end(), part[v].begin(), part[v].end());
    }
    if (cnt > 0) {
        UD2_HIP(hipMemcpyAsync(ls->d_split, ls->h_split.data(), size_t(cnt) * sizeof(int32_t), hipMemcpyHostToDevice,
                               st));
        UD2_HIP(hipStreamSynchronize(st));
    }
    ls->split_version = version;
    ls->split_forced = policy == UD2_TILE_ALWAYS;
    return UD2_OK;
}

PoseBufs pose_view(const ud2_poses* P) {
    PoseBufs b;
    b.x = P->x_d;
    b.c = P->c_d;
    b.rv = P->rv_d;
    b.dihe = P->dihe_d;
    b.e = P->e_d;
    b.nchain = P->nchain;
    return b;
}

int check_poses(const ud2_ligset* ls, const ud2_poses* P) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    if (!P || !P->x_d || !P->c_d || !P->rv_d || !P->dihe_d || !P->e_d) return fail(UD2_ERR_ARG, "null pose buffer");
    if (P->nchain <= 0) return fail(UD2_ERR_ARG, "nchain must be positive");
    return UD2_OK;
}

int check_mode(const ud2_scene* sc, const ud2_ligset* ls, int32_t mode) {
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    if (mode != UD2_MODE_DIRECT && mode != UD2_MODE_GRID) return fail(UD2_ERR_ARG, "mode must be 0 (direct) or 1 (grid)");
    if (mode == UD2_MODE_GRID) {
        if (!sc->d_maps) return fail(UD2_ERR_STATE, "grid mode requested but the scene has no grid maps");
        for (int t = 1; t < kNumTypes; t++)
            if (ls->has_slot_type[t] && sc->slot_of_type[t] < 0)
                return fail(UD2_ERR_STATE, "grid mode: no map for ligand atom type " + std::to_string(t));
    }
    return UD2_OK;
}

int ensure_sel(ud2_ligset* ls, int64_t n) {
    if (n <= ls->sel_all_cap) return UD2_OK;
    ls->sel_all_cap = 0;
    if (ls->d_sel_all) UD2_HIP(hipFree(ls->d_sel_all));
    ls->d_sel_all = nullptr;
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(&ls->d_sel_all), size_t(n) * sizeof(int32_t)));
    ls->sel_all_cap = n;
    return UD2_OK;
}

// Runs one opt_kernel operation over the selected poses: the selection is
// regrouped by atoms-per-lane class and each class launched with its own LDS
// size; per-pose outputs stay at the pose's position in sel_d.
int run_opt(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel,
            int32_t mode, int op, int32_t max_steps, float v_cap, float slope, float* out_e, float* out_g,
            const float* dir, float alpha, hipStream_t st) {
    if (n_sel <= 0) return UD2_OK;
    if (!sel_d) return fail(UD2_ERR_ARG, "null selection");
    std::vector<int32_t> h(n_sel);
    // the selection may have been written by earlier work on the caller's stream (which need not
    // synchronise with the null stream): wait for it before reading
    UD2_HIP(hipStreamSynchronize(st));
    UD2_HIP(hipMemcpy(h.data(), sel_d, size_t(n_sel) * sizeof(int32_t), hipMemcpyDeviceToHost));
    const int64_t npose = int64_t(ls->n_lig) * P->nchain;
    // the poses by class, then their positions in the selection
    std::vector<int32_t> ids(size_t(2) * n_sel);
    std::vector<int> start(kMaxApl + 2, 0), dmax(kMaxApl + 1, 6);
    for (int32_t p : h) {
        if (p < 0 || p >= npose) return fail(UD2_ERR_ARG, "pose id out of range: " + std::to_string(p));
        const DevLig& d = ls->h_ligs[p / P->nchain];
        start[d.apl + 1]++;
        dmax[d.apl] = std::max(dmax[d.apl], 6 + int(d.ntors));
    }
    for (int apl = 1; apl <= kMaxApl; apl++) start[apl + 1] += start[apl];
    std::vector<int> at(start);
    for (int32_t s = 0; s < n_sel; s++) {
        const int k = at[ls->h_ligs[h[s] / P->nchain].apl]++;
        ids[k] = h[s];
        ids[n_sel + k] = s;
    }
    // Up to kOptFew poses go with the kernel's arguments: a handful of poses is evaluated in 10 us, and copying
    // their ids to the GPU twice, with a wait before, took 31 us more (37 poses 60 -> 29 us a call; 64 ids and their
    // places are 512 bytes of arguments). More are copied, both lists at once.
    const bool few = n_sel <= kOptFew;
    if (!few) {
        int rc = ensure_sel(const_cast<ud2_ligset*>(ls), 2 * int64_t(n_sel));
        if (rc) return rc;
        UD2_HIP(hipMemcpy(ls->d_sel_all, ids.data(), ids.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    OptArgs A{};
    A.L = ls->view();
    SceneDev empty{};
    A.S = sc ? sc->view() : empty;
    A.P = pose_view(P);
    A.mode = mode;
    A.max_steps = max_steps;
    A.v_cap = v_cap;
    A.slope = slope;
    A.out_e = out_e;
    A.out_g = out_g;
    A.dir = dir;
    A.alpha = alpha;
    A.op = op;
    for (int apl = 1; apl <= kMaxApl; apl++) {
        const int n = start[apl + 1] - start[apl];
        if (n == 0) continue;
        A.hdim_ld = odd_ld(dmax[apl]);
        A.lds_floats_per_wave = lds_round4(lds_head_floats(apl, A.hdim_ld) + dmax[apl] * A.hdim_ld);
        if (few) {
            std::copy_n(&ids[start[apl]], n, A.few);
            std::copy_n(&ids[n_sel + start[apl]], n, A.few_pos);
        } else {
            A.sel = ls->d_sel_all + start[apl];
            A.pos = ls->d_sel_all + n_sel + start[apl];
        }
        A.n_sel = n;
        UD2_HIP(launch_opt(A, apl, st));
    }
    return UD2_OK;
}

McArgs mc_args(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_mc_params* prm) {
    McArgs A;
    std::memset(&A, 0, sizeof(A));
    A.L = ls->view();
    A.S = sc->view();
    A.P = pose_view(P);
    A.mode = prm->mode;
    A.mc_steps = prm->mc_steps;
    A.opt_steps = prm->opt_steps;
    A.randomize = prm->randomize;
    A.seed = prm->seed;
    A.lig_index_base = prm->lig_index_base;
    A.stats = reinterpret_cast<unsigned long long*>(prm->stats_d);
    return A;
}

// Searches of few chains run each chain on a team of four waves (see Team in ud2_device.h), which ends a chain in
// about half the time and takes about twice one wave's time on the chip. A CU holds three to six teams, so what counts is
// the work in units of the costliest chain: the chains where all ligands are of one size, fewer where the small
// ones are done before the largest. Time of a plain grid search with teams over that with one wave per chain (256 CUs,
// 128 chains per ligand, 6 and 10 steps of 28 iterations), by units per CU:
//   ligands of one size, 9 to 120 atoms: 4 0.47-0.81, 6 0.64-0.97, 7 0.72-1.02, 7.5 0.76-1.02, 8 0.79-1.30, 12 1.10-1.58;
//   seven ranges of sizes in 10-80 atoms: up to 5 0.36-0.75, 5-7 0.54-0.97, 7-8 0.65-0.90, 8-9 0.80-1.20, above 0.89-1.22.
// In direct mode, by chains per CU: ligands of one size 2 0.48-0.71, 4 0.47-0.94, 6 0.54-0.92; 10-60 atoms 8 1.03, 12 1.04.
constexpr int kTeamMaxApl = 2;
constexpr double kTeamLoadPerCu = 8.0;                    // grid: fewer units of work than this,
constexpr int kTeamPerCuGrid = 12, kTeamPerCuDirect = 6;  // and at most so many chains

bool team_search(const ud2_ligset* ls, const McArgs& A, int nchain) {
    if (A.mc_steps <= 0 || A.opt_steps <= 0) return false;
    const int64_t chains = int64_t(ls->n_lig) * nchain, cus = n_cus();
    if (A.mode == kDirect) return chains <= kTeamPerCuDirect * cus;
    return chains <= kTeamPerCuGrid * cus && ls->load * nchain < kTeamLoadPerCu * double(cus);
}

// One persistent MC launch over n ligands of the work order at order (atoms-per-lane class apl, kernel
// variant, largest 6 + ntors dmax), its queue head at counter.
// team: the search runs its chains on teams (where the class has a build for it).
// shared: the launch runs beside the one-slot class of the same search. A wider class then takes one block
// per CU less than it could alone, so one-slot waves fit beside it (three two-slot waves of 168 VGPRs fill
// a SIMD's register file, and the one-slot launch would wait for the whole two-slot queue to drain).
int launch_mc_part(McArgs A, int apl, int variant, const int32_t* order, int n, int32_t* counter, int dmax,
                   int nchain, hipStream_t st, bool team, bool shared = false) {
    if (n <= 0) return UD2_OK;
    // in direct mode the sum over the receptor outweighs what two chains per wave share: whole waves only
    if (A.mode == kDirect) variant = kMcWhole;
    const int tw = mc_variant_tw(variant);
    const int cpw = kWave / tw;  // chains per wave
    A.order = order;
    A.n_order = n;
    A.counter = counter;
    A.hdim_ld = odd_ld(dmax);
    A.lds_floats_per_wave = cpw * lds_round4(lds_head_floats(apl, A.hdim_ld, tw) + dmax * A.hdim_ld);
    const int lds_bytes = A.lds_floats_per_wave * kWavesPerBlock * int(sizeof(float));
    if (lds_bytes > 160 * 1024) return fail(UD2_ERR_LIMIT, "per-block LDS exceeds 160 KB");
    const int64_t items = int64_t(n) * ((nchain + cpw - 1) / cpw);
    if (team && variant == kMcWhole && apl <= kTeamMaxApl &&
        lds_bytes + team_floats(apl) * int(sizeof(float)) <= 160 * 1024) {
        UD2_HIP(launch_mc_team(A, apl, int(items), st));
        return UD2_OK;
    }
    const int64_t need = (items + kWavesPerBlock - 1) / kWavesPerBlock;
    int bpc = mc_blocks_per_cu(apl, variant, A.mode, lds_bytes);
    if (shared && apl > 1) bpc = std::max(1, bpc - 1);
    const int64_t cap = int64_t(n_cus()) * bpc;
    const int nb = int(std::max<int64_t>(1, std::min(need, cap)));
    // the most waves per SIMD the launch keeps resident: a block of four waves per CU is one per SIMD
    const int64_t per_cu = (need + n_cus() - 1) / n_cus();
    const int waves = per_cu <= 2 ? 2 : per_cu <= 4 ? 4 : 6;
    UD2_HIP(launch_mc(A, apl, variant, nb, waves, st));
    return UD2_OK;
}

// Side streams of a device for the MC search's concurrent launches (default priority), created on the
// first search that may create them; with the fork / join events. kMcSide + 1 streams keep to the
// process's four hardware queues.
constexpr int kMcSide = 3;
struct SideStreams {
    hipStream_t s[kMcSide] = {};
    hipEvent_t fork = nullptr, join[kMcSide] = {};
    bool ready = false;
};
constexpr int kMaxDevices = 64;
std::mutex g_side_mu;
SideStreams g_side[kMaxDevices];

// The current device's side streams, or null when they do not exist and may not be created. Called
// with g_side_mu held.
SideStreams* side_streams(bool may_create) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    SideStreams& S = g_side[dev];
    if (S.ready || !may_create) return S.ready ? &S : nullptr;
    bool ok = hipEventCreateWithFlags(&S.fork, hipEventDisableTiming) == hipSuccess;
    for (int i = 0; i < kMcSide && ok; i++)
        ok = hipStreamCreateWithFlags(&S.s[i], hipStreamNonBlocking) == hipSuccess &&
             hipEventCreateWithFlags(&S.join[i], hipEventDisableTiming) == hipSuccess;
    S.ready = ok;
    return ok ? &S : nullptr;
}

// The MC search's persistent launches, one per atoms-per-lane class present in the set (widest
// first), each over its part of the set's work order, the one-atom-per-lane class in one launch per
// kernel variant its ligands are assigned. Queue heads at heads[0 .. kMcHeads): the variant parts at
// heads[variant], class apl >= 2 at heads[kMcVariants + apl - 2] (all set to zero on the stream
// first). With more than one launch they go to the stream and its device's side streams (forked
// from and joined back into the stream, the launches dealt round the streams), so each launch's tail
// overlaps the next one's start; where side streams do not exist and may_create is false, they run
// one after the other on the stream. The same poses either way. No allocation and no
// synchronisation; a host copy and a synchronisation only when the tile split is rebuilt.
int launch_mc_classes(const ud2_ligset* ls, const ud2_poses* P, McArgs A, int32_t* heads, hipStream_t st,
                      bool may_create) {
    static_assert(kMcVariants + kMaxApl - 2 < kMcHeads, "queue head of the widest class");
    int rc = refresh_split(ls, st);
    if (rc) return rc;
    struct Part {
        int apl, variant, n, dmax;
        const int32_t* order;
        int32_t* head;
    };
    std::vector<Part> parts;
    for (int apl = kMaxApl; apl >= 2; apl--)
        if (ls->cls_cnt[apl] > 0)
            parts.push_back({apl, kMcWhole, ls->cls_cnt[apl], ls->cls_dmax[apl], ls->d_order + ls->cls_pos[apl],
                             heads + kMcVariants + apl - 2});
    // the tuned table comes from launches that fill the chip, where a team has no place: a search of few chains keeps its
    // teams (2 ligands of 20 atoms at 128 chains, 6 steps: 2.1 ms, two chains per wave 7.1)
    const bool team = team_search(ls, A, P->nchain);
    for (int v = 0; v < kMcVariants; v++)
        if (ls->part_cnt[v] > 0)
            parts.push_back({1, team && !ls->split_forced ? int(kMcWhole) : v, ls->part_cnt[v], ls->part_dmax[v],
                             ls->d_split + ls->part_pos[v], heads + v});
    UD2_HIP(launch_fill_i32(heads, 0, kMcHeads, st));
    std::lock_guard<std::mutex> lock(g_side_mu);
    SideStreams* S = parts.size() > 1 ? side_streams(may_create) : nullptr;
    if (S) UD2_HIP(hipEventRecord(S->fork, st));
    bool used[kMcSide] = {};
    for (size_t i = 0; i < parts.size(); i++) {
        const Part& p = parts[i];
        hipStream_t s = st;
        const int k = int(i % (kMcSide + 1)) - 1;  // -1: the stream itself
        if (S && k >= 0) {
            s = S->s[k];
            if (!used[k]) UD2_HIP(hipStreamWaitEvent(s, S->fork, 0));
            used[k] = true;
        }
        rc = launch_mc_part(A, p.apl, p.variant, p.order, p.n, p.head, p.dmax, P->nchain, s,
                            team, S != nullptr && ls->cls_cnt[1] > 0);
        if (rc) return rc;
    }
    for (int k = 0; S && k < kMcSide; k++)
        if (used[k]) {
            UD2_HIP(hipEventRecord(S->join[k], S->s[k]));
            UD2_HIP(hipStreamWaitEvent(st, S->join[k], 0));
        }
    return UD2_OK;
}

}  // namespace

namespace ud2 {
// Validation and launches of ud2_mc, with the launches' queue heads at heads (kMcHeads int32 of
// device memory that the call zeroes on the stream).
int mc_search(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_mc_params* prm,
              int32_t* heads, hipStream_t st, bool may_create) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (!prm) return fail(UD2_ERR_ARG, "null parameters");
    rc = check_mode(sc, ls, prm->mode);
    if (rc) return rc;
    if (prm->mc_steps < 0 || prm->opt_steps < 0) return fail(UD2_ERR_ARG, "negative step count");
    if (int64_t(ls->n_lig) * P->nchain > (int64_t(1) << 30)) return fail(UD2_ERR_LIMIT, "too many chains");
    if (!heads) return fail(UD2_ERR_ARG, "null queue heads");
    return launch_mc_classes(ls, P, mc_args(sc, ls, P, prm), heads, st, may_create);
}
}  // namespace ud2

extern "C" {

const char* ud2_version(void) { return "ud2-mi355x 0.1.0 (gfx950)"; }

const char* ud2_last_error(void) { return g_err.c_str(); }

int ud2_device_count(int32_t* n_h) {
    if (!n_h) return fail(UD2_ERR_ARG, "null output");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) {
        *n_h = 0;
        return fail(UD2_ERR_NODEV, std::string("hipGetDeviceCount: ") + hipGetErrorString(e));
    }
    *n_h = n;
    return UD2_OK;
}

int ud2_set_device(int32_t id) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(UD2_ERR_NODEV, "no GPU device is visible");
    if (id < 0 || id >= n) return fail(UD2_ERR_NODEV, "device id out of range");
    UD2_HIP(hipSetDevice(id));
    return UD2_OK;
}

int ud2_synchronize(void) {
    UD2_HIP(hipDeviceSynchronize());
    return UD2_OK;
}

int ud2_device_memory(int64_t* free_h, int64_t* total_h) {
    size_t f = 0, t = 0;
    UD2_HIP(hipMemGetInfo(&f, &t));
    if (free_h) *free_h = int64_t(f);
    if (total_h) *total_h = int64_t(t);
    return UD2_OK;
}

// ------------------------------------------------------------------- scene
namespace {

// The scene's reach lists: cells of kReachEdge A over the box and kReachMargin A around it, where a receptor atom is
// within 8 A at all; coarser where that makes more than kReachCells cells or kReachEntries entries. A
// finer cell lists fewer atoms out of the cutoff (2 A: 1.65 listed per atom in reach, 3 A: 2.06) and
// the lists then take more memory (a 30 A box: 15,625 cells, 15 MB). The margin holds the atoms of most poses
// that the penalty is about to push back into the box. They are built with the scene, for every scene: 0.12 ms, a
// quarter of it waiting for their size. (Built at the first direct sum, a captured or allocation-free search could not
// have them.) With a copy of every cell's count to the host and its sum back, 0.24 ms.
constexpr double kReachEdge = 2.0, kReachMargin = 10.0, kReachDist = 8.02;
constexpr int64_t kReachCells = 1 << 14, kReachEntries = 1 << 23;

void drop_reach(ud2_scene* sc) {
    for (int d = 0; d < 3; d++) sc->rn[d] = 0;
    if (sc->d_reach) (void)hipFree(sc->d_reach);
    if (sc->d_reach_off) (void)hipFree(sc->d_reach_off);
    sc->d_reach = nullptr;
    sc->d_reach_off = nullptr;
    sc->reach_bytes = 0;
}

int build_reach(ud2_scene* sc, const std::vector<float4>& rec) {
    double lo[3], hi[3];
    for (int d = 0; d < 3; d++) {
        lo[d] = INFINITY;
        hi[d] = -INFINITY;
    }
    for (const float4& r : rec) {
        const float x[3] = {r.x, r.y, r.z};
        if (!std::isfinite(r.x) || !std::isfinite(r.y) || !std::isfinite(r.z)) continue;  // never in reach
        for (int d = 0; d < 3; d++) {
            lo[d] = std::min(lo[d], double(x[d]) - kReachDist);
            hi[d] = std::max(hi[d], double(x[d]) + kReachDist);
        }
    }
    bool any = true;
    for (int d = 0; d < 3; d++) {
        sc->rec_lo[d] = float(lo[d]);
        sc->rec_hi[d] = float(hi[d]);
        lo[d] = std::max(lo[d], double(sc->box_lo[d]) - kReachMargin);
        hi[d] = std::min(hi[d], double(sc->box_hi[d]) + kReachMargin);
        any = any && hi[d] > lo[d];
    }
    if (!any) return UD2_OK;
    ReachArgs A{};
    unsigned long long total = 0;
    for (double edge = kReachEdge;; edge *= 1.25) {
        int64_t cells = 1;
        for (int d = 0; d < 3; d++) {
            const double n = std::ceil((hi[d] - lo[d]) / edge);
            if (!(n <= double(kReachCells))) cells = kReachCells + 1;
            else {
                sc->rn[d] = std::max(1, int32_t(n));
                cells = std::min(cells * sc->rn[d], kReachCells + 1);
            }
        }
        if (cells > kReachCells) continue;
        sc->redge = float(edge);
        A.rec = sc->d_rec;
        A.nrec = sc->nrec;
        A.total = reinterpret_cast<unsigned long long*>(sc->d_rec + sc->nrec);
        for (int d = 0; d < 3; d++) {
            A.rn[d] = sc->rn[d];
            A.rorigin[d] = sc->rorigin[d] = float(lo[d]);
        }
        A.edge = sc->redge;
        if (!sc->d_reach_off)  // fewer cells in every further round
            UD2_HIP(hipMalloc(reinterpret_cast<void**>(&sc->d_reach_off), size_t(cells) * sizeof(int2)));
        A.off = sc->d_reach_off;
        if (total) UD2_HIP(launch_fill_i32(reinterpret_cast<int32_t*>(A.total), 0, 2, nullptr));
        UD2_HIP(launch_reach(A, false, nullptr));
        UD2_HIP(hipMemcpy(&total, A.total, sizeof(total), hipMemcpyDeviceToHost));
        if (total <= (unsigned long long)kReachEntries || cells == 1) break;
    }
    hipError_t e = hipErrorOutOfMemory;
    if (total <= (unsigned long long)kReachEntries)
        e = hipMalloc(reinterpret_cast<void**>(&sc->d_reach), std::max<size_t>(total, 1) * sizeof(float4));
    if (e == hipErrorOutOfMemory) {  // one cell and still too many, or no memory: the whole receptor, by scalar loads
        (void)hipGetLastError();
        drop_reach(sc);
        return UD2_OK;
    }
    UD2_HIP(e);
    A.reach = sc->d_reach;
    sc->reach_bytes = int64_t(total * sizeof(float4)) + int64_t(sc->rn[0]) * sc->rn[1] * sc->rn[2] * int64_t(sizeof(int2));
    UD2_HIP(launch_reach(A, true, nullptr));
    UD2_HIP(hipStreamSynchronize(nullptr));
    return UD2_OK;
}

}  // namespace

int ud2_scene_create(const float* rec_xyz_h, const int32_t* rec_types_h, int32_t n_rec, const float box_lo_h[3],
                     const float box_hi_h[3], ud2_scene** out) {
    if (!out) return fail(UD2_ERR_ARG, "null output");
    *out = nullptr;
    if (n_rec < 0 || (n_rec > 0 && (!rec_xyz_h || !rec_types_h)) || !box_lo_h || !box_hi_h)
        return fail(UD2_ERR_ARG, "bad receptor arguments");
    for (int d = 0; d < 3; d++)
        if (!(box_hi_h[d] > box_lo_h[d])) return fail(UD2_ERR_ARG, "box must have hi > lo on every axis");
    std::vector<float4> rec;
    rec.reserve(n_rec);
    for (int i = 0; i < n_rec; i++) {
        int t = rec_types_h[i];
        if (t < 0 || t >= kNumTypes) return fail(UD2_ERR_ARG, "receptor atom type out of range");
        if (t == 0) continue;  // hydrogens carry no Vina term
        float4 v;
        v.x = rec_xyz_h[3 * i];
        v.y = rec_xyz_h[3 * i + 1];
        v.z = rec_xyz_h[3 * i + 2];
        const uint32_t word = atom_word(float_bits(kVdwHost[t]), uint32_t(kFlagsHost[t]));
        std::memcpy(&v.w, &word, sizeof(word));
        rec.push_back(v);
    }
    ud2_scene* sc = new ud2_scene();
    hipGetDevice(&sc->device);
    for (int d = 0; d < 3; d++) {
        sc->box_lo[d] = box_lo_h[d];
        sc->box_hi[d] = box_hi_h[d];
    }
    for (int t = 0; t < kNumTypes; t++) sc->slot_of_type[t] = -1;
    sc->nrec = int32_t(rec.size());
    rec.push_back(make_float4(0.0f, 0.0f, 0.0f, 0.0f));  // where the entries of the reach lists are counted
    int rc = upload(&sc->d_rec, rec);
    rec.pop_back();
    if (!rc) rc = build_reach(sc, rec);
    if (rc) {
        ud2_scene_destroy(sc);
        return rc;
    }
    *out = sc;
    return UD2_OK;
}

namespace {

// A scene's maps: what is checked of a request for them before anything of the scene changes.
struct GridPlan {
    int32_t gn[3];
    float origin[3], spacing;
    std::vector<int32_t> probe_types;
    int32_t slot_of_type[kNumTypes];
    int64_t points = 1;
};

int plan_probes(GridPlan& g, const int32_t* probe_types_h, int32_t n_types) {
    if (n_types <= 0 || n_types > kNumTypes || !probe_types_h) return fail(UD2_ERR_ARG, "bad probe type list");
    for (int t = 0; t < kNumTypes; t++) g.slot_of_type[t] = -1;
    g.probe_types.assign(probe_types_h, probe_types_h + n_types);
    for (int k = 0; k < n_types; k++) {
        int t = probe_types_h[k];
        if (t <= 0 || t >= kNumTypes) return fail(UD2_ERR_ARG, "probe type out of range (hydrogen has no map)");
        if (g.slot_of_type[t] >= 0) return fail(UD2_ERR_ARG, "duplicate probe type");
        g.slot_of_type[t] = k;
    }
    return UD2_OK;
}

void drop_grids(ud2_scene* sc) {
    for (void* p : {(void*)sc->d_maps, (void*)sc->d_cells, (void*)sc->d_slot})
        if (p) (void)hipFree(p);
    sc->d_maps = nullptr;
    sc->d_cells = nullptr;
    sc->d_slot = nullptr;
    sc->probe_types.clear();
    for (int t = 0; t < kNumTypes; t++) sc->slot_of_type[t] = -1;
    for (int d = 0; d < 3; d++) sc->gn[d] = 0;
    sc->gspacing = 0.0f;
}

// The plan's maps in place of the scene's: filled by `fill`, then copied cell-major. Without maps where a step fails.
int make_grids(ud2_scene* sc, const GridPlan& g, const std::function<int()>& fill) {
    drop_grids(sc);
    for (int d = 0; d < 3; d++) {
        sc->gn[d] = g.gn[d];
        sc->gorigin[d] = g.origin[d];
    }
    sc->gspacing = g.spacing;
    sc->probe_types = g.probe_types;
    std::copy(g.slot_of_type, g.slot_of_type + kNumTypes, sc->slot_of_type);
    const auto make = [&]() -> int {
        int rc = upload(&sc->d_slot, std::vector<int32_t>(g.slot_of_type, g.slot_of_type + kNumTypes));
        if (rc) return rc;
        UD2_HIP(hipMalloc(reinterpret_cast<void**>(&sc->d_maps), size_t(g.points) * g.probe_types.size() * sizeof(float)));
        rc = fill();
        if (rc) return rc;
        const size_t ncell = size_t(g.gn[0] - 1) * (g.gn[1] - 1) * (g.gn[2] - 1) * g.probe_types.size();
        UD2_HIP(hipMalloc(reinterpret_cast<void**>(&sc->d_cells), ncell * 2 * sizeof(float4)));
        BrickArgs B;
        B.maps = sc->d_maps;
        B.cells = sc->d_cells;
        for (int d = 0; d < 3; d++) B.gn[d] = g.gn[d];
        B.nslot = int32_t(g.probe_types.size());
        UD2_HIP(launch_brick(B, nullptr));
        UD2_HIP(hipDeviceSynchronize());
        return UD2_OK;
    };
    const int rc = make();
    if (rc) drop_grids(sc);
    return rc;
}

}  // namespace

int ud2_scene_build_grids(ud2_scene* sc, float spacing, const int32_t* probe_types_h, int32_t n_types) {
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    if (!(spacing > 0.0f)) return fail(UD2_ERR_ARG, "spacing must be positive");
    GridPlan g;
    int rc = plan_probes(g, probe_types_h, n_types);
    if (rc) return rc;
    for (int d = 0; d < 3; d++) {
        float size = sc->box_hi[d] - sc->box_lo[d];
        g.gn[d] = int32_t(std::lround(double(size) / double(spacing))) + 1;
        if (g.gn[d] < 2) return fail(UD2_ERR_ARG, "box smaller than two grid points");
        g.origin[d] = sc->box_lo[d];
        g.points *= g.gn[d];
    }
    g.spacing = spacing;
    return make_grids(sc, g, [&]() -> int {
        GridArgs A{};
        A.S = sc->view();
        std::vector<int32_t> by_radius(n_types);
        std::iota(by_radius.begin(), by_radius.end(), 0);
        std::stable_sort(by_radius.begin(), by_radius.end(), [&](int a, int b) {
            return kVdwHost[g.probe_types[a]] < kVdwHost[g.probe_types[b]];
        });
        for (int k = 0; k < n_types; k++) {
            const int t = g.probe_types[by_radius[k]];
            A.radius[k] = kVdwHost[t];
            A.lut[k] = pair_lut_host(t);
            A.slot[k] = by_radius[k];
        }
        A.nslot = n_types;
        A.maps = sc->d_maps;
        UD2_HIP(launch_grid_build(A, nullptr));
        return UD2_OK;
    });
}

int ud2_scene_set_grids(ud2_scene* sc, const int32_t n_h[3], const float origin_h[3], float spacing,
                        const int32_t* probe_types_h, int32_t n_types, const float* maps_h) {
    if (!sc || !n_h || !origin_h || !maps_h) return fail(UD2_ERR_ARG, "null argument");
    if (!(spacing > 0.0f)) return fail(UD2_ERR_ARG, "spacing must be positive");
    GridPlan g;
    int rc = plan_probes(g, probe_types_h, n_types);
    if (rc) return rc;
    for (int d = 0; d < 3; d++) {
        if (n_h[d] < 2) return fail(UD2_ERR_ARG, "grid needs at least two points per axis");
        g.gn[d] = n_h[d];
        g.origin[d] = origin_h[d];
        g.points *= n_h[d];
    }
    g.spacing = spacing;
    return make_grids(sc, g, [&]() -> int {
        UD2_HIP(hipMemcpy(sc->d_maps, maps_h, size_t(g.points) * n_types * sizeof(float), hipMemcpyHostToDevice));
        return UD2_OK;
    });
}

int ud2_scene_grid_info(const ud2_scene* sc, int32_t n_h[3], float origin_h[3], float* spacing_h,
                        int32_t* n_types_h) {
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    for (int d = 0; d < 3; d++) {
        if (n_h) n_h[d] = sc->gn[d];
        if (origin_h) origin_h[d] = sc->gorigin[d];
    }
    if (spacing_h) *spacing_h = sc->gspacing;
    if (n_types_h) *n_types_h = int32_t(sc->probe_types.size());
    return UD2_OK;
}

int ud2_scene_download_maps(const ud2_scene* sc, float* maps_h) {
    if (!sc || !maps_h) return fail(UD2_ERR_ARG, "null argument");
    if (!sc->d_maps) return fail(UD2_ERR_STATE, "scene has no grid maps");
    size_t n = size_t(sc->gn[0]) * sc->gn[1] * sc->gn[2] * sc->probe_types.size();
    UD2_HIP(hipMemcpy(maps_h, sc->d_maps, n * sizeof(float), hipMemcpyDeviceToHost));
    return UD2_OK;
}

int ud2_scene_gather_probe(const ud2_scene* sc, int64_t n_gathers, int64_t span_cells, uint32_t seed, float* out_d,
                           void* stream) {
    if (!sc || !out_d || n_gathers <= 0) return fail(UD2_ERR_ARG, "bad arguments");
    if (!sc->d_cells) return fail(UD2_ERR_STATE, "the scene has no grid maps");
    const int64_t total = int64_t(sc->gn[0] - 1) * (sc->gn[1] - 1) * (sc->gn[2] - 1) * int64_t(sc->probe_types.size());
    const int64_t span = span_cells > 0 ? span_cells : total;
    if (span > total || span > int64_t(UINT32_MAX)) return fail(UD2_ERR_ARG, "span beyond the maps");
    const int64_t n_threads = (n_gathers + kProbePerThread - 1) / kProbePerThread;
    UD2_HIP(launch_gather_probe(sc->d_cells, uint32_t(span), seed, out_d, n_threads, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

int ud2_valu_probe(int64_t n_threads, int32_t iters, float* out_d, void* stream) {
    if (n_threads < 0 || iters < 0) return fail(UD2_ERR_ARG, "negative size");
    if (n_threads > 0 && !out_d) return fail(UD2_ERR_ARG, "null output");
    UD2_HIP(launch_valu_probe(out_d, iters, n_threads, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

int ud2_scene_reach(ud2_scene* sc, int32_t keep, int64_t* bytes_h) {
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    if (!keep) drop_reach(sc);
    if (bytes_h) *bytes_h = sc->reach_bytes;
    return UD2_OK;
}

int ud2_scene_destroy(ud2_scene* sc) {
    if (!sc) return UD2_OK;
    if (sc->d_rec) hipFree(sc->d_rec);
    drop_grids(sc);
    drop_reach(sc);
    delete sc;
    return UD2_OK;
}

// ------------------------------------------------------------------ ligands
int ud2_ligset_create(const ud2_ligand_batch* b, ud2_ligset** out) {
    if (!out) return fail(UD2_ERR_ARG, "null output");
    *out = nullptr;
    if (!b || b->n_lig <= 0) return fail(UD2_ERR_ARG, "empty ligand batch");
    if (!b->atom_off_h || !b->tors_off_h || !b->pair_off_h || !b->types_h || !b->xyz_h)
        return fail(UD2_ERR_ARG, "null ligand array");
    const int n = b->n_lig;
    const int nt_all = b->tors_off_h[n];
    if (nt_all > 0 && (!b->axis_h || !b->dihe0_h || !b->rot_off_h || !b->rot_atoms_h || !b->range_off_h || !b->ranges_h))
        return fail(UD2_ERR_ARG, "null torsion array");
    if (b->pair_off_h[n] > 0 && !b->pairs_h) return fail(UD2_ERR_ARG, "null pair array");
    if (b->atom_off_h[0] != 0 || b->tors_off_h[0] != 0 || b->pair_off_h[0] != 0)
        return fail(UD2_ERR_ARG, "CSR offsets must start at 0");

    std::vector<DevLig> ligs(n);
    std::vector<float4> x0(b->atom_off_h[n]);
    std::vector<int2> axis(nt_all), trange(nt_all);
    std::vector<float> dihe0(nt_all);
    std::vector<float2> ranges;
    std::vector<unsigned long long> mask(size_t(nt_all) * kMaxApl, 0ull);
    std::vector<uint2> pairs;
    std::vector<unsigned long long> fold;
    std::vector<uint4> pack;
    std::vector<uint8_t> has_type(kNumTypes, 0);
    for (int l = 0; l < n; l++) {
        const int a0 = b->atom_off_h[l], na = b->atom_off_h[l + 1] - a0;
        const int t0 = b->tors_off_h[l], nt = b->tors_off_h[l + 1] - t0;
        const int p0 = b->pair_off_h[l], np = b->pair_off_h[l + 1] - p0;
        const std::string tag = "ligand " + std::to_string(l) + ": ";
        if (na <= 0 || nt < 0 || np < 0) return fail(UD2_ERR_ARG, tag + "negative or empty sizes");
        if (na > kMaxAtoms) return fail(UD2_ERR_LIMIT, tag + "more than " + std::to_string(kMaxAtoms) + " atoms");
        if (nt > kMaxTors) return fail(UD2_ERR_LIMIT, tag + "more than " + std::to_string(kMaxTors) + " torsions");
        DevLig& d = ligs[l];
        d.natom = na;
        d.ntors = nt;
        d.atom_off = a0;
        d.tors_off = t0;
        d.pair_off = int32_t(pairs.size());
        d.apl = (na + kWave - 1) / kWave;
        d.nheavy = 0;
        for (int a = 0; a < na; a++) {
            int t = b->types_h[a0 + a];
            if (t < 0 || t >= kNumTypes) return fail(UD2_ERR_ARG, tag + "atom type out of range");
            float4 v;
            v.x = b->xyz_h[3 * (a0 + a)];
            v.y = b->xyz_h[3 * (a0 + a) + 1];
            v.z = b->xyz_h[3 * (a0 + a) + 2];
            if (!std::isfinite(v.x) || !std::isfinite(v.y) || !std::isfinite(v.z))
                return fail(UD2_ERR_ARG, tag + "non-finite input coordinate");
            std::memcpy(&v.w, &t, sizeof(int));
            x0[a0 + a] = v;
            if (t != 0) {
                d.nheavy++;
                has_type[t] = 1;
            }
        }
        for (int t = 0; t < nt; t++) {
            const int tg = t0 + t;
            int from = b->axis_h[2 * tg], to = b->axis_h[2 * tg + 1];
            if (from < 0 || from >= na || to < 0 || to >= na || from == to)
                return fail(UD2_ERR_ARG, tag + "torsion axis atom out of range");
            axis[tg] = make_int2(from, to);
            dihe0[tg] = b->dihe0_h[tg];
            const int r0 = b->rot_off_h[tg], r1 = b->rot_off_h[tg + 1];
            if (r1 < r0) return fail(UD2_ERR_ARG, tag + "bad rotated-atom offsets");
            for (int k = r0; k < r1; k++) {
                int a = b->rot_atoms_h[k];
                if (a < 0 || a >= na) return fail(UD2_ERR_ARG, tag + "rotated atom out of range");
                mask[size_t(tg) * kMaxApl + a / kWave] |= 1ull << (a % kWave);
            }
            const int q0 = b->range_off_h[tg], q1 = b->range_off_h[tg + 1];
            if (q1 <= q0) return fail(UD2_ERR_ARG, tag + "torsion without an allowed range");
            trange[tg] = make_int2(int(ranges.size()), q1 - q0);
            for (int k = q0; k < q1; k++) {
                float lo = b->ranges_h[2 * k], hi = b->ranges_h[2 * k + 1];
                if (!(lo <= hi)) return fail(UD2_ERR_ARG, tag + "torsion range with lo > hi");
                ranges.push_back(make_float2(lo, hi));
            }
        }
        // Leaf-first application order: a torsion that rotates another's pivot is its ancestor,
        // and deeper torsions go first. The order is valid when no torsion rotates the axis
        // atoms of one applied after it (a proper torsion tree); a pose update can then take
        // every pivot and axis from the coordinates before the update, as the result of the
        // reference's index-order application (bfgs.cuh:565-567) is the same in exact arithmetic.
        {
            auto rotates = [&](int tp, int atom) {
                return (mask[size_t(t0 + tp) * kMaxApl + atom / kWave] >> (atom % kWave)) & 1ull;
            };
            std::vector<int> depth(nt, 0), ord(nt);
            for (int t = 0; t < nt; t++)
                for (int tp = 0; tp < nt; tp++)
                    if (tp != t && rotates(tp, axis[t0 + t].y)) depth[t]++;
            std::iota(ord.begin(), ord.end(), 0);
            std::stable_sort(ord.begin(), ord.end(), [&](int a, int c) { return depth[a] > depth[c]; });
            bool ok = true;
            for (int i = 0; i < nt && ok; i++)
                for (int j = i + 1; j < nt; j++)
                    if (rotates(ord[i], axis[t0 + ord[j]].x) || rotates(ord[i], axis[t0 + ord[j]].y)) {
                        ok = false;
                        break;
                    }
            // entry k: .y holds the torsion applied k-th, .x the rank at which torsion k is applied
            for (int k = 0; k < nt; k++) {
                axis[t0 + k].y |= ord[k] << 16;
                axis[t0 + ord[k]].x |= k << 16;
            }
            d.leaf_first = ok ? 1 : 0;
        }
        // Heavy pairs as records for the final score (each pair once, i < j), in
        // diagonal order (j - i, i).
        std::vector<std::pair<int, int>> pl;
        for (int k = 0; k < np; k++) {
            int i = b->pairs_h[2 * (p0 + k)], j = b->pairs_h[2 * (p0 + k) + 1];
            if (i < 0 || i >= na || j < 0 || j >= na || i == j) return fail(UD2_ERR_ARG, tag + "pair atom out of range");
            if (i > j) std::swap(i, j);
            int ti = b->types_h[a0 + i], tj = b->types_h[a0 + j];
            if (ti == 0 || tj == 0) continue;  // eval_ef is zero for hydrogen pairs (vina.h:223-225)
            pl.emplace_back(i, j);
        }
        std::stable_sort(pl.begin(), pl.end(), [](const std::pair<int, int>& a, const std::pair<int, int>& c) {
            const int da = a.second - a.first, dc = c.second - c.first;
            return da != dc ? da < dc : a.first < c.first;
        });
        for (auto& ij : pl) {
            const int i = ij.first, j = ij.second;
            const int ti = b->types_h[a0 + i], tj = b->types_h[a0 + j];
            uint2 rec;
            rec.x = uint32_t(i) | (uint32_t(j) << 8) | (uint32_t(pair_flags_host(ti, tj)) << 16);
            float rs = kVdwHost[ti] + kVdwHost[tj];
            std::memcpy(&rec.y, &rs, sizeof(float));
            pairs.push_back(rec);
        }
        d.npair = int32_t(pairs.size()) - d.pair_off;
        // The same pairs as folded diagonals for one-slot ligands: on diagonal d lane l scores
        // {l, (l + d) mod na}; diagonals 1 .. na / 2 visit every unordered pair once (on the
        // last diagonal of an even na only lanes below na / 2).
        // Per diagonal, one 64-bit word per atom slot (atom a in bit a % 64 of word a / 64).
        d.fold_off = int32_t(fold.size());
        d.nfold = na / 2;
        {
            const int apl = (na + kWave - 1) / kWave;
            std::vector<uint8_t> scored(size_t(na) * na, 0);
            for (auto& ij : pl) scored[size_t(ij.first) * na + ij.second] = scored[size_t(ij.second) * na + ij.first] = 1;
            size_t seen = 0;
            for (int dd = 1; dd <= d.nfold; dd++) {
                std::vector<unsigned long long> m(apl, 0ull);
                const int lanes = (2 * dd == na) ? na / 2 : na;
                for (int l = 0; l < lanes; l++)
                    if (scored[size_t(l) * na + (l + dd) % na]) {
                        m[l / kWave] |= 1ull << (l % kWave);
                        seen++;
                    }
                fold.insert(fold.end(), m.begin(), m.end());
            }
            if (seen != pl.size()) return fail(UD2_ERR_STATE, tag + "pair diagonals do not cover the pairs");
        }
        d.pack_off = int32_t(pack.size() / kWave);
        d.npack = 0;
        if (na > kWave / 2 && na <= kWave && !pl.empty()) {
            const int n_steps = pack_pairs(na, pl, b->types_h + a0, pack);
            if (n_steps < 0) return fail(UD2_ERR_STATE, tag + "packed pair steps do not cover the pairs");
            d.npack = n_steps;
        }
        if (na <= kWave / 2 && !pl.empty()) d.npack = (d.nfold + 1) / 2;
    }
    // the tables of the ligands of up to 32 atoms follow, written on the GPU from their diagonals, and one step more: the
    // kernels load one step ahead
    int64_t steps = int64_t(pack.size() / kWave);
    bool diagonals = false;
    for (DevLig& d : ligs)
        if (d.natom <= kWave / 2 && d.npack > 0) {
            d.pack_off = int32_t(steps);
            steps += d.npack;
            diagonals = true;
        }
    ud2_ligset* ls = new ud2_ligset();
    hipGetDevice(&ls->device);
    ls->n_lig = n;
    ls->h_ligs = ligs;
    ls->has_slot_type = has_type;
    ls->h_order.resize(n);
    std::iota(ls->h_order.begin(), ls->h_order.end(), 0);
    {
        // Weight of one chain, in units that mean nothing by themselves (only ratios are used): energy evaluations, growing
        // with the atoms, times a fixed part, the pair loop (per atom up to 32 atoms, per packed step up to 64,
        // per atom and slot beyond) and the torsions. Against the time of a chain on a full GPU (12-200 atoms, 0-20 torsions,
        // 28 iterations a step) the weights of flexible ligands of up to 64 atoms agree within 15 %, and those of
        // 65-200 atoms among themselves within 30 %, a quarter low beside the smaller ones; rigid ligands take half of theirs.
        auto cost = [&](int l) {
            const DevLig& d = ligs[l];
            const double pairs = d.natom <= kWave / 2 ? 23.5 * d.natom
                                 : d.apl == 1         ? 95.0 * d.npack
                                                      : 41.5 * double(d.apl) * d.natom;
            return (2800.0 + 36.0 * d.natom) * (1500.0 + pairs + 64.0 * d.ntors);
        };
        std::stable_sort(ls->h_order.begin(), ls->h_order.end(), [&](int a, int c) {
            if (ligs[a].apl != ligs[c].apl) return ligs[a].apl > ligs[c].apl;
            return cost(a) > cost(c);
        });
        double sum = 0.0, most = 0.0;
        for (int k = 0; k < n; k++) {
            sum += cost(k);
            most = std::max(most, cost(k));
        }
        ls->load = sum / most;
        for (int k = 0; k < n; k++) {
            const DevLig& d = ligs[ls->h_order[k]];
            if (ls->cls_cnt[d.apl]++ == 0) ls->cls_pos[d.apl] = k;
            ls->cls_dmax[d.apl] = std::max<int32_t>(ls->cls_dmax[d.apl], 6 + d.ntors);
        }
    }
    int rc = UD2_OK;
    if (!rc) rc = upload(&ls->d_ligs, ligs);
    if (!rc) rc = upload(&ls->d_x0, x0);
    if (!rc) rc = upload(&ls->d_axis, axis);
    if (!rc) rc = upload(&ls->d_dihe0, dihe0);
    if (!rc) rc = upload(&ls->d_trange, trange);
    if (!rc) rc = upload(&ls->d_ranges, ranges);
    if (!rc) rc = upload(&ls->d_mask, mask);
    if (!rc) rc = upload(&ls->d_pairs, pairs);
    if (!rc) rc = upload(&ls->d_fold, fold);
    const auto tables = [&]() {
        UD2_HIP(hipMalloc(reinterpret_cast<void**>(&ls->d_pack), size_t(steps + 1) * kWave * sizeof(uint4)));
        if (!pack.empty())
            UD2_HIP(hipMemcpy(ls->d_pack, pack.data(), pack.size() * sizeof(uint4), hipMemcpyHostToDevice));
        if (diagonals) UD2_HIP(launch_pack_diagonals(ls->view(), n, ls->d_pack, nullptr));
        return int(UD2_OK);
    };
    if (!rc) rc = tables();
    if (!rc) rc = upload(&ls->d_counter, std::vector<int32_t>(std::max(kMcHeads, kMaxApl + 1), 0));
    if (!rc) rc = upload(&ls->d_order, ls->h_order);
    if (!rc) rc = upload(&ls->d_split, std::vector<int32_t>(std::max(ls->cls_cnt[1], 1), 0));
    if (!rc) rc = refresh_split(ls, nullptr);
    if (rc) {
        ud2_ligset_destroy(ls);
        return rc;
    }
    *out = ls;
    return UD2_OK;
}

int ud2_ligset_destroy(ud2_ligset* ls) {
    if (!ls) return UD2_OK;
    void* ptrs[] = {ls->d_ligs,   ls->d_x0,      ls->d_axis,    ls->d_dihe0,       ls->d_trange,
                    ls->d_ranges, ls->d_mask,    ls->d_pairs,   ls->d_fold,        ls->d_pack,     ls->d_counter,  ls->d_order,
                    ls->d_sel_all, ls->d_bias_start, ls->d_bias_site, ls->d_bias_r2, ls->d_split};
    for (void* p : ptrs)
        if (p) hipFree(p);
    delete ls;
    return UD2_OK;
}

int ud2_ligset_set_bias(ud2_ligset* ls, int32_t bias_type, float bias_k, const int32_t* bias_off_h,
                        const float* bias_h) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    if (bias_type < UD2_BIAS_NO || bias_type > UD2_BIAS_ALIGN)
        return fail(UD2_ERR_ARG, "bias_type must be 0 (no), 1 (pos) or 2 (align)");
    if (!std::isfinite(bias_k)) return fail(UD2_ERR_ARG, "non-finite bias_k");
    const int natoms = ls->h_ligs.back().atom_off + ls->h_ligs.back().natom;
    std::vector<int32_t> start;
    std::vector<float4> site;
    std::vector<float> r2;
    if (bias_off_h) {
        if (bias_off_h[0] != 0) return fail(UD2_ERR_ARG, "bias offsets must start at 0");
        for (int a = 0; a < natoms; a++)
            if (bias_off_h[a + 1] < bias_off_h[a]) return fail(UD2_ERR_ARG, "bias offsets must not decrease");
        const int nsite = bias_off_h[natoms];
        if (nsite > 0 && !bias_h) return fail(UD2_ERR_ARG, "null bias array");
        for (int j = 0; j < nsite; j++) {
            const float* b = bias_h + 5 * j;
            for (int k = 0; k < 5; k++)
                if (!std::isfinite(b[k])) return fail(UD2_ERR_ARG, "non-finite bias parameter at site " + std::to_string(j));
            if (bias_type == UD2_BIAS_POS && !(b[4] > 0.0f))
                return fail(UD2_ERR_ARG, "pos bias site " + std::to_string(j) + " needs r2 > 0");
            site.push_back(make_float4(b[0], b[1], b[2], b[3]));
            r2.push_back(b[4]);
        }
        if (nsite > 0) start.assign(bias_off_h, bias_off_h + natoms + 1);
    }
    void* old[] = {ls->d_bias_start, ls->d_bias_site, ls->d_bias_r2};
    for (void* p : old)
        if (p) UD2_HIP(hipFree(p));
    ls->d_bias_start = nullptr;
    ls->d_bias_site = nullptr;
    ls->d_bias_r2 = nullptr;
    if (!start.empty()) {
        int rc = upload(&ls->d_bias_start, start);
        if (!rc) rc = upload(&ls->d_bias_site, site);
        if (!rc) rc = upload(&ls->d_bias_r2, r2);
        if (rc) return rc;
    }
    ls->bias_type = bias_type;
    ls->bias_k = bias_k;
    return UD2_OK;
}

int ud2_ligset_sizes(const ud2_ligset* ls, int32_t* n_lig_h, int32_t* natom_h, int32_t* ntors_h) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    if (n_lig_h) *n_lig_h = ls->n_lig;
    for (int l = 0; l < ls->n_lig; l++) {
        if (natom_h) natom_h[l] = ls->h_ligs[l].natom;
        if (ntors_h) ntors_h[l] = ls->h_ligs[l].ntors;
    }
    return UD2_OK;
}

int ud2_ligset_set_constraint(ud2_ligset* ls, int32_t constraint) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    ls->constraint = constraint ? 1 : 0;
    return UD2_OK;
}

int ud2_ligset_pose_layout(const ud2_ligset* ls, int32_t nchain, int64_t* x_floats_h, int64_t* dihe_floats_h,
                           int64_t* n_pose_h) {
    if (!ls || nchain <= 0) return fail(UD2_ERR_ARG, "bad arguments");
    int64_t na = 0, nt = 0;
    for (auto& l : ls->h_ligs) {
        na += l.natom;
        nt += l.ntors;
    }
    if (x_floats_h) *x_floats_h = na * nchain * 3;
    if (dihe_floats_h) *dihe_floats_h = nt * nchain;
    if (n_pose_h) *n_pose_h = int64_t(ls->n_lig) * nchain;
    return UD2_OK;
}

int ud2_init_poses(const ud2_ligset* ls, const ud2_poses* P, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    const int64_t npose = int64_t(ls->n_lig) * P->nchain;
    if (npose > (int64_t(1) << 30)) return fail(UD2_ERR_LIMIT, "too many poses");
    std::vector<int32_t> ids(npose);
    std::iota(ids.begin(), ids.end(), 0);
    int32_t* d_ids = nullptr;
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(&d_ids), ids.size() * sizeof(int32_t)));
    hipError_t e = hipMemcpy(d_ids, ids.data(), ids.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess)
        rc = run_opt(nullptr, ls, P, d_ids, int32_t(npose), UD2_MODE_DIRECT, 4, 0, 0.0f, 0.0f, nullptr, nullptr,
                     nullptr, 0.0f, static_cast<hipStream_t>(stream));
    hipStreamSynchronize(static_cast<hipStream_t>(stream));
    hipFree(d_ids);
    if (e != hipSuccess) return fail(UD2_ERR_HIP, std::string("hipMemcpy: ") + hipGetErrorString(e));
    return rc;
}

// ------------------------------------------------------------------ hot path
int ud2_score_posevecs(const ud2_scene* sc, const ud2_ligset* ls, int32_t lig, int64_t n, const float* pv_d,
                       float* e_d, float* g_d, int32_t mode, float v_cap, float slope, void* stream) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    int rc = check_mode(sc, ls, mode);
    if (rc) return rc;
    if (lig < 0 || lig >= ls->n_lig) return fail(UD2_ERR_ARG, "ligand index out of range");
    if (n < 0) return fail(UD2_ERR_ARG, "negative pose count");
    if (n == 0) return UD2_OK;
    if (!pv_d || !e_d || !g_d) return fail(UD2_ERR_ARG, "null buffer");
    const DevLig& d = ls->h_ligs[lig];
    PoseVecArgs A;
    A.L = ls->view();
    A.S = sc->view();
    A.lig = lig;
    A.n = n;
    A.pv = pv_d;
    A.e = e_d;
    A.g = g_d;
    A.v_cap = v_cap;
    A.slope = slope;
    A.mode = mode;
    A.hdim_ld = odd_ld(6 + d.ntors);
    A.lds_floats_per_wave = lds_round4(lds_head_floats(d.apl, A.hdim_ld));
    const int lds_bytes = A.lds_floats_per_wave * kWavesPerBlock * int(sizeof(float));
    const int64_t need = (n + kWavesPerBlock - 1) / kWavesPerBlock;
    const int64_t cap = int64_t(n_cus()) * posevec_blocks_per_cu(d.apl, mode, lds_bytes);
    const int nb = int(std::max<int64_t>(1, std::min(need, cap)));
    UD2_HIP(launch_posevec(A, d.apl, nb, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

int ud2_energy_grad(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, int32_t mode, float v_cap, float slope, float* e_d, float* g_d, void* stream) {
    int rc = check_poses(ls, P);
    if (!rc) rc = check_mode(sc, ls, mode);
    if (rc) return rc;
    return run_opt(sc, ls, P, sel_d, n_sel, mode, 1, 0, v_cap, slope, e_d, g_d, nullptr, 0.0f,
                   static_cast<hipStream_t>(stream));
}

int ud2_pose_update(const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel, const float* dir_d,
                    float alpha, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (n_sel > 0 && !dir_d) return fail(UD2_ERR_ARG, "null direction buffer");
    return run_opt(nullptr, ls, P, sel_d, n_sel, UD2_MODE_DIRECT, 2, 0, 0.0f, 0.0f, nullptr, nullptr, dir_d, alpha,
                   static_cast<hipStream_t>(stream));
}

int ud2_line_search(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, int32_t mode, float v_cap, float slope, float* alpha_d, float* g_d, void* stream) {
    int rc = check_poses(ls, P);
    if (!rc) rc = check_mode(sc, ls, mode);
    if (rc) return rc;
    return run_opt(sc, ls, P, sel_d, n_sel, mode, 3, 0, v_cap, slope, alpha_d, g_d, nullptr, 0.0f,
                   static_cast<hipStream_t>(stream));
}

int ud2_optimize(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                 int32_t n_sel, int32_t mode, int32_t max_steps, float v_cap, float slope, float* e_d, void* stream) {
    int rc = check_poses(ls, P);
    if (!rc) rc = check_mode(sc, ls, mode);
    if (rc) return rc;
    if (max_steps < 0) return fail(UD2_ERR_ARG, "negative max_steps");
    return run_opt(sc, ls, P, sel_d, n_sel, mode, 0, max_steps, v_cap, slope, e_d, nullptr, nullptr, 0.0f,
                   static_cast<hipStream_t>(stream));
}

int ud2_mc(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_mc_params* prm, void* stream) {
    return mc_search(sc, ls, P, prm, ls ? ls->d_counter : nullptr, static_cast<hipStream_t>(stream), true);
}

int ud2_set_tile_policy(int32_t policy, int32_t variant) {
    if (policy < UD2_TILE_AUTO || policy > UD2_TILE_ALWAYS)
        return fail(UD2_ERR_ARG, "tile policy must be 0 (auto), 1 (never) or 2 (always)");
    if (variant == 0) variant = kMcHalf4;
    if (variant < kMcHalf4 || variant >= kMcVariants) return fail(UD2_ERR_ARG, "variant must name a half-wave kernel");
    std::lock_guard<std::mutex> lock(g_tune.mu);
    if (g_tune.policy != policy || g_tune.forced != variant) {
        g_tune.policy = policy;
        g_tune.forced = variant;
        g_tune.version++;
    }
    return UD2_OK;
}

int ud2_tune_info(int32_t* policy_h, int32_t* variant_h, float* ms_h, int32_t* range_h) {
    std::lock_guard<std::mutex> lock(g_tune.mu);
    if (policy_h) *policy_h = g_tune.policy;
    for (int b = 0; b < kTuneBuckets; b++) {
        if (variant_h) variant_h[b] = g_tune.variant[b];
        if (ms_h)
            for (int v = 0; v < kMcVariants; v++) ms_h[kMcVariants * b + v] = g_tune.ms[b][v];
        if (range_h) {
            const int ia = b / kTuneTorsBuckets, it = b % kTuneTorsBuckets;
            range_h[4 * b] = 8 * ia + 1;
            range_h[4 * b + 1] = 8 * ia + 8;
            range_h[4 * b + 2] = 4 * it;
            range_h[4 * b + 3] = it == kTuneTorsBuckets - 1 ? kTileNarrowTors : 4 * it + 3;
        }
    }
    return UD2_OK;
}

int ud2_autotune(const ud2_scene* sc, const ud2_ligset* ls, const ud2_mc_params* prm, int32_t nchain,
                 const char* cache_path, void* stream) {
    if (!ls) return fail(UD2_ERR_ARG, "null ligand set");
    if (!prm) return fail(UD2_ERR_ARG, "null parameters");
    int rc = check_mode(sc, ls, prm->mode);
    if (rc) return rc;
    if (prm->mc_steps < 0 || prm->opt_steps < 0) return fail(UD2_ERR_ARG, "negative step count");
    if (nchain <= 0) nchain = 8;
    if (nchain > 1024) return fail(UD2_ERR_ARG, "nchain above 1024");
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0;
    UD2_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    UD2_HIP(hipGetDeviceProperties(&prop, dev));
    const std::string key = std::string("ud2-mc-tune 3 ") + prop.gcnArchName + " cus " + std::to_string(n_cus()) +
                            " mode " + std::to_string(prm->mode);
    bool have[kTuneBuckets] = {};
    int8_t choice[kTuneBuckets] = {};
    float ms[kTuneBuckets][kMcVariants];
    if (cache_path && *cache_path) {
        // one line per bucket: bucket, variant, then the probe time of each variant
        std::ifstream f(cache_path);
        std::string line;
        if (f && std::getline(f, line) && line == key) {
            while (std::getline(f, line)) {
                std::istringstream in(line);
                int b = -1, v = -1;
                float m[kMcVariants];
                in >> b >> v;
                for (int k = 0; k < kMcVariants; k++) in >> m[k];
                if (!in || b < 0 || b >= kTuneBuckets || v < 0 || v >= kMcVariants) continue;
                have[b] = true;
                choice[b] = int8_t(v);
                for (int k = 0; k < kMcVariants; k++) ms[b][k] = m[k];
            }
        }
    }
    std::vector<std::vector<int32_t>> members(kTuneBuckets);
    bool any = false;
    for (int l = 0; l < ls->n_lig; l++) {
        const DevLig& d = ls->h_ligs[l];
        const int b = d.apl == 1 ? tune_bucket(d.natom, d.ntors) : -1;
        if (b >= 0 && !have[b]) {
            members[b].push_back(l);
            any = true;
        }
    }
    if (any) {
        // probe searches with the caller's parameters: each bucket's ligands, repeated until the launch
        // holds two rounds of the chip's resident whole-wave chains, searched with every variant (each
        // variant run once untimed first); a half-wave variant replaces whole waves only when it is at
        // least 2% faster (in direct mode every variant runs whole waves). Repeated ligands write the same
        // pose slots (the probe's poses are discarded).
        const DevLig& last = ls->h_ligs.back();
        const int64_t n_atoms = int64_t(last.atom_off) + last.natom, n_tors = int64_t(last.tors_off) + last.ntors;
        float *x = nullptr, *c = nullptr, *rv = nullptr, *dh = nullptr, *e = nullptr;
        int32_t* ord = nullptr;
        hipEvent_t ev0 = nullptr, ev1 = nullptr;
        const int lds1 = kWavesPerBlock * int(sizeof(float)) *
                         lds_round4(lds_head_floats(1, odd_ld(kTileNarrow), kWave) + kTileNarrow * odd_ld(kTileNarrow));
        const int64_t slots = int64_t(n_cus()) * mc_blocks_per_cu(1, kMcWhole, prm->mode, lds1) * kWavesPerBlock;
        const int reps = int(std::max<int64_t>(1, (2 * slots + nchain - 1) / nchain));
        auto run = [&]() -> int {
            UD2_HIP(hipMalloc(&x, size_t(n_atoms) * nchain * 3 * sizeof(float)));
            UD2_HIP(hipMalloc(&c, size_t(ls->n_lig) * nchain * 3 * sizeof(float)));
            UD2_HIP(hipMalloc(&rv, size_t(ls->n_lig) * nchain * 3 * sizeof(float)));
            UD2_HIP(hipMalloc(&dh, size_t(std::max<int64_t>(n_tors, 1)) * nchain * sizeof(float)));
            UD2_HIP(hipMalloc(&e, size_t(ls->n_lig) * nchain * sizeof(float)));
            UD2_HIP(hipMalloc(&ord, size_t(reps) * sizeof(int32_t) + sizeof(int32_t)));
            UD2_HIP(hipEventCreate(&ev0));
            UD2_HIP(hipEventCreate(&ev1));
            ud2_poses P{x, c, rv, dh, e, nchain};
            ud2_mc_params pp = *prm;
            pp.stats_d = nullptr;
            const McArgs A = mc_args(sc, ls, &P, &pp);
            int32_t* head = ord + reps;
            std::vector<int32_t> h(reps);
            bool warm = false;
            for (int b = 0; b < kTuneBuckets; b++) {
                if (members[b].empty()) continue;
                int dmax = 6;
                for (int k = 0; k < reps; k++) {
                    h[k] = members[b][k % members[b].size()];
                    dmax = std::max(dmax, 6 + int(ls->h_ligs[h[k]].ntors));
                }
                UD2_HIP(hipMemcpyAsync(ord, h.data(), size_t(reps) * sizeof(int32_t), hipMemcpyHostToDevice, st));
                float best[kMcVariants];
                for (int v = 0; v < kMcVariants; v++) best[v] = 1e30f;
                for (int pass = warm ? 1 : 0; pass < 2; pass++)
                    for (int v = 0; v < kMcVariants; v++) {
                        UD2_HIP(launch_fill_i32(head, 0, 1, st));
                        UD2_HIP(hipEventRecord(ev0, st));
                        const int r = launch_mc_part(A, 1, v, ord, reps, head, dmax, nchain, st, false);
                        if (r) return r;
                        UD2_HIP(hipEventRecord(ev1, st));
                        UD2_HIP(hipEventSynchronize(ev1));
                        float t = 0;
                        UD2_HIP(hipEventElapsedTime(&t, ev0, ev1));
                        best[v] = std::min(best[v], t);
                    }
                warm = true;
                have[b] = true;
                int fast = kMcHalf4;
                for (int v = 0; v < kMcVariants; v++) {
                    ms[b][v] = best[v];
                    if (v != kMcWhole && best[v] < best[fast]) fast = v;
                }
                choice[b] = int8_t(prm->mode != kDirect && best[fast] < 0.98f * best[kMcWhole] ? fast : kMcWhole);
            }
            return UD2_OK;
        };
        rc = run();
        for (void* p : {(void*)x, (void*)c, (void*)rv, (void*)dh, (void*)e, (void*)ord})
            if (p) hipFree(p);
        if (ev0) hipEventDestroy(ev0);
        if (ev1) hipEventDestroy(ev1);
        if (rc) return rc;
    }
    {
        std::lock_guard<std::mutex> lock(g_tune.mu);
        for (int b = 0; b < kTuneBuckets; b++)
            if (have[b]) {
                g_tune.variant[b] = choice[b];
                for (int v = 0; v < kMcVariants; v++) g_tune.ms[b][v] = ms[b][v];
            }
        g_tune.version++;
    }
    if (any && cache_path && *cache_path) {
        std::ostringstream o;
        o << key << "\n";
        for (int b = 0; b < kTuneBuckets; b++)
            if (have[b]) {
                o << b << " " << int(choice[b]);
                for (int v = 0; v < kMcVariants; v++) o << " " << ms[b][v];
                o << "\n";
            }
        std::ofstream f(cache_path, std::ios::trunc);
        if (!f || !(f << o.str())) return fail(UD2_ERR_ARG, std::string("cannot write the tuning cache ") + cache_path);
    }
    return UD2_OK;
}

int ud2_cluster(const ud2_ligset* ls, const ud2_poses* P, float rmsd_limit, int32_t* leaders_d, int32_t* nleaders_d,
                void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (!leaders_d || !nleaders_d) return fail(UD2_ERR_ARG, "null output");
    if (P->nchain > kClusterMaxPoses) return fail(UD2_ERR_LIMIT, "nchain too large for clustering");
    ClusterArgs A;
    A.L = ls->view();
    A.x = P->x_d;
    A.e = P->e_d;
    A.nchain = P->nchain;
    A.n_lig = ls->n_lig;
    A.limit = rmsd_limit;
    A.leaders = leaders_d;
    A.nleaders = nleaders_d;
    UD2_HIP(launch_cluster(A, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

namespace {

int run_score(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel,
              float* out4_d, float* decomp_d, int32_t decomp_stride, void* stream) {
    std::vector<int32_t> h(n_sel);
    UD2_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    UD2_HIP(hipMemcpy(h.data(), sel_d, size_t(n_sel) * sizeof(int32_t), hipMemcpyDeviceToHost));
    int apl_max = 1;
    const int64_t npose = int64_t(ls->n_lig) * P->nchain;
    for (int32_t p : h) {
        if (p < 0 || p >= npose) return fail(UD2_ERR_ARG, "pose id out of range: " + std::to_string(p));
        const DevLig& d = ls->h_ligs[p / P->nchain];
        if (decomp_d && d.natom > decomp_stride)
            return fail(UD2_ERR_ARG, "atom_stride " + std::to_string(decomp_stride) + " is below the " +
                                         std::to_string(d.natom) + " atoms of pose " + std::to_string(p));
        apl_max = std::max(apl_max, int(d.apl));
    }
    ScoreArgs A;
    A.L = ls->view();
    A.S = sc->view();
    A.x = P->x_d;
    A.nchain = P->nchain;
    A.sel = sel_d;
    A.n_sel = n_sel;
    A.out4 = out4_d;
    A.decomp = decomp_d;
    A.decomp_stride = decomp_stride;
    // one launch at the widest class: narrower ligands run with idle register slots
    UD2_HIP(launch_final_score(A, apl_max, decomp_d != nullptr, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

}  // namespace

int ud2_final_score(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                    int32_t n_sel, float* out4_d, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    if (n_sel <= 0) return UD2_OK;
    if (!sel_d || !out4_d) return fail(UD2_ERR_ARG, "null buffer");
    return run_score(sc, ls, P, sel_d, n_sel, out4_d, nullptr, 0, stream);
}

int ud2_score_decomp(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d,
                     int32_t n_sel, int32_t atom_stride, float* decomp_d, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (!sc) return fail(UD2_ERR_ARG, "null scene");
    if (n_sel <= 0) return UD2_OK;
    if (!sel_d || !decomp_d) return fail(UD2_ERR_ARG, "null buffer");
    if (atom_stride <= 0) return fail(UD2_ERR_ARG, "atom_stride must be positive");
    return run_score(sc, ls, P, sel_d, n_sel, nullptr, decomp_d, atom_stride, stream);
}

}  // extern "C"

// ------------------------------------------------------- learned proposal
struct ud2_mlp {
    int device = 0;
    float* d_params = nullptr;  // canonical FP32 parameters, then mu and inv_sigma
    float* d_m = nullptr;       // Adam moments
    float* d_v = nullptr;
    uint16_t* d_w1 = nullptr;
    uint16_t* d_w1s = nullptr;
    uint16_t* d_w2t = nullptr;
    uint16_t* d_w2s = nullptr;
    uint16_t* d_w2 = nullptr;
    float* d_w3r = nullptr;
    int32_t step = 0;
    // training scratch, sized for cap_groups groups
    int32_t cap_groups = 0;
    uint16_t* d_fm = nullptr;   // xn, a1, dz1, dz2 (MlpTrain)
    float* d_part = nullptr;
    float* d_gpart = nullptr;   // split-K partials of the weight-gradient GEMMs

    MlpPack pack() const { return MlpPack{d_w1, d_w1s, d_w2t, d_w2s, d_w2, d_w3r}; }

    MlpDev view() const {
        MlpDev w;
        w.w1 = d_w1;
        w.w1s = d_w1s;
        w.w2t = d_w2t;
        w.w2s = d_w2s;
        w.w2 = d_w2;
        w.b1 = d_params + kOffB1;
        w.b2 = d_params + kOffB2;
        w.w3 = d_w3r;
        w.b3 = d_params + kOffB3;
        w.mu = d_params + kMlpNParam;
        w.inv_sigma = d_params + kMlpNParam + kFeat;
        return w;
    }
};

namespace {

// Ranges of the weight-gradient GEMMs' rows: 16 ranges of 40 tiles are 640 waves.
constexpr int kGemmSplits = 16;

void free_train(ud2_mlp* m) {
    for (void* p : {(void*)m->d_fm, (void*)m->d_part, (void*)m->d_gpart})
        if (p) (void)hipFree(p);
    m->d_part = m->d_gpart = nullptr;
    m->d_fm = nullptr;
    m->cap_groups = 0;
}

int ensure_train(ud2_mlp* m, int32_t n_groups) {
    if (n_groups <= m->cap_groups) return UD2_OK;
    free_train(m);
    const size_t rows = size_t(n_groups) * kGroup;
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(&m->d_fm), rows * size_t(kFeat + 3 * kHidden) * sizeof(uint16_t)));
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(&m->d_part), size_t(n_groups) * kPartStride * sizeof(float)));
    UD2_HIP(hipMalloc(reinterpret_cast<void**>(&m->d_gpart), size_t(kGemmSplits) * kGradW * sizeof(float)));
    m->cap_groups = n_groups;
    return UD2_OK;
}

int check_mlp_inputs(const uint16_t* x_d, int32_t n_groups) {
    if (n_groups <= 0) return fail(UD2_ERR_ARG, "n_groups must be positive");
    if (!x_d) return fail(UD2_ERR_ARG, "null feature buffer");
    if (reinterpret_cast<uintptr_t>(x_d) % 8) return fail(UD2_ERR_ARG, "feature buffer must be 8-byte aligned");
    return UD2_OK;
}

// The minibatch's partial sums (dy null: of the loss to label_d; else for the given d loss / d y_hat), then the
// gradient into grad, or the Adam step O where grad is null.
int mlp_step(ud2_mlp* m, const uint16_t* x_d, const float* label_d, const int32_t* groups_d, int32_t n_groups,
             const float* dy, float* grad, const MlpAdam& O, hipStream_t st) {
    int rc = ensure_train(m, n_groups);
    if (rc) return rc;
    const size_t rows = size_t(n_groups) * kGroup;
    MlpTrain T;
    T.x = x_d;
    T.groups = groups_d;
    T.n_groups = n_groups;
    T.label = label_d;
    T.dy = dy;
    T.xn = m->d_fm;
    T.a1 = T.xn + rows * kFeat;
    T.dz1 = T.a1 + rows * kHidden;
    T.dz2 = T.dz1 + rows * kHidden;
    T.part = m->d_part;
    int splits = kGemmSplits;
    while (splits > 1 && n_groups % splits) splits >>= 1;
    UD2_HIP(launch_mlp_train(m->view(), T, splits, m->d_gpart, st));
    UD2_HIP(launch_mlp_update(m->d_gpart, splits, m->d_part, n_groups, grad, O, m->pack(), st));
    return UD2_OK;
}

}  // namespace

int ud2_mlp_create(const float* params_h, ud2_mlp** out) {
    if (!out) return fail(UD2_ERR_ARG, "null output");
    *out = nullptr;
    if (!params_h) return fail(UD2_ERR_ARG, "null parameters");
    ud2_mlp* m = new ud2_mlp();
    hipGetDevice(&m->device);
    const size_t np = kMlpNParam;
    int rc = UD2_OK;
    auto al = [&](void** p, size_t bytes) {
        if (rc == UD2_OK && hipMalloc(p, bytes) != hipSuccess) rc = fail(UD2_ERR_HIP, "hipMalloc failed");
    };
    al(reinterpret_cast<void**>(&m->d_params), (np + kMlpNNorm) * sizeof(float));
    al(reinterpret_cast<void**>(&m->d_m), np * sizeof(float));
    al(reinterpret_cast<void**>(&m->d_v), np * sizeof(float));
    al(reinterpret_cast<void**>(&m->d_w1), size_t(kFeat) * kHidden * sizeof(uint16_t));
    al(reinterpret_cast<void**>(&m->d_w1s), size_t(kW1sSize) * sizeof(uint16_t));
    al(reinterpret_cast<void**>(&m->d_w2t), size_t(kHidden) * kHidden * sizeof(uint16_t));
    al(reinterpret_cast<void**>(&m->d_w2s), size_t(kHidden) * kHidden * sizeof(uint16_t));
    al(reinterpret_cast<void**>(&m->d_w2), size_t(kHidden) * kHidden * sizeof(uint16_t));
    al(reinterpret_cast<void**>(&m->d_w3r), size_t(kHidden) * sizeof(float));
    if (rc == UD2_OK) rc = ud2_mlp_set_params(m, params_h);
    if (rc != UD2_OK) {
        std::string keep = g_err;
        ud2_mlp_destroy(m);
        g_err = keep;
        return rc;
    }
    *out = m;
    return UD2_OK;
}

int ud2_mlp_set_params(ud2_mlp* m, const float* params_h) {
    if (!m || !params_h) return fail(UD2_ERR_ARG, "null argument");
    for (int i = 0; i < kMlpNParam + kMlpNNorm; i++)
        if (!std::isfinite(params_h[i])) return fail(UD2_ERR_ARG, "non-finite network parameter " + std::to_string(i));
    UD2_HIP(hipMemcpy(m->d_params, params_h, size_t(kMlpNParam + kMlpNNorm) * sizeof(float), hipMemcpyHostToDevice));
    UD2_HIP(hipMemset(m->d_m, 0, size_t(kMlpNParam) * sizeof(float)));
    UD2_HIP(hipMemset(m->d_v, 0, size_t(kMlpNParam) * sizeof(float)));
    m->step = 0;
    UD2_HIP(hipMemset(m->d_w1s, 0, size_t(kW1sSize) * sizeof(uint16_t)));  // the features past 79 of the last K block
    UD2_HIP(launch_mlp_pack(m->d_params, m->pack(), nullptr));
    UD2_HIP(hipDeviceSynchronize());
    return UD2_OK;
}

int ud2_mlp_get_params(const ud2_mlp* m, float* params_h) {
    if (!m || !params_h) return fail(UD2_ERR_ARG, "null argument");
    UD2_HIP(hipDeviceSynchronize());
    UD2_HIP(hipMemcpy(params_h, m->d_params, size_t(kMlpNParam + kMlpNNorm) * sizeof(float), hipMemcpyDeviceToHost));
    return UD2_OK;
}

int ud2_mlp_destroy(ud2_mlp* m) {
    if (!m) return UD2_OK;
    free_train(m);
    for (void* p : {(void*)m->d_params, (void*)m->d_m, (void*)m->d_v, (void*)m->d_w1, (void*)m->d_w1s,
                    (void*)m->d_w2t, (void*)m->d_w2s, (void*)m->d_w2, (void*)m->d_w3r})
        if (p) (void)hipFree(p);
    delete m;
    return UD2_OK;
}

int ud2_mlp_forward(const ud2_mlp* m, const uint16_t* x_d, const int32_t* groups_d, int32_t n_groups, float* y_d,
                    void* stream) {
    if (!m || !y_d) return fail(UD2_ERR_ARG, "null argument");
    int rc = check_mlp_inputs(x_d, n_groups);
    if (rc) return rc;
    UD2_HIP(launch_mlp_forward(m->view(), x_d, groups_d, n_groups, y_d, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

int ud2_mlp_backward(ud2_mlp* m, const uint16_t* x_d, const int32_t* groups_d, int32_t n_groups, const float* dy_d,
                     float* grad_d, void* stream) {
    if (!m || !dy_d || !grad_d) return fail(UD2_ERR_ARG, "null argument");
    int rc = check_mlp_inputs(x_d, n_groups);
    if (rc) return rc;
    return mlp_step(m, x_d, nullptr, groups_d, n_groups, dy_d, grad_d, MlpAdam{}, static_cast<hipStream_t>(stream));
}

int ud2_mlp_train_step(ud2_mlp* m, const uint16_t* x_d, const float* label_d, const int32_t* groups_d,
                       int32_t n_groups, const ud2_adam* opt, float* loss_d, void* stream) {
    if (!m || !label_d || !opt) return fail(UD2_ERR_ARG, "null argument");
    int rc = check_mlp_inputs(x_d, n_groups);
    if (rc) return rc;
    if (!(opt->lr > 0.0f) || !(opt->beta1 >= 0.0f && opt->beta1 < 1.0f) || !(opt->beta2 >= 0.0f && opt->beta2 < 1.0f) ||
        !(opt->eps > 0.0f))
        return fail(UD2_ERR_ARG, "invalid Adam settings");
    const int32_t step = m->step + 1;
    MlpAdam O;
    O.p = m->d_params;
    O.m = m->d_m;
    O.v = m->d_v;
    O.lr = opt->lr;
    O.beta1 = opt->beta1;
    O.beta2 = opt->beta2;
    O.eps = opt->eps;
    O.c1 = 1.0f - std::pow(opt->beta1, float(step));
    O.c2 = 1.0f - std::pow(opt->beta2, float(step));
    O.loss = loss_d;
    O.loss_scale = 1.0f / (float(n_groups) * kGroup);
    rc = mlp_step(m, x_d, label_d, groups_d, n_groups, nullptr, nullptr, O, static_cast<hipStream_t>(stream));
    if (rc == UD2_OK) m->step = step;
    return rc;
}

int ud2_features(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const int32_t* sel_d, int32_t n_sel,
                 uint16_t* x_d, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    rc = check_mode(sc, ls, UD2_MODE_GRID);
    if (rc) return rc;
    if (n_sel <= 0) return UD2_OK;
    if (!sel_d || !x_d) return fail(UD2_ERR_ARG, "null buffer");
    std::vector<int32_t> h(n_sel);
    UD2_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    UD2_HIP(hipMemcpy(h.data(), sel_d, size_t(n_sel) * sizeof(int32_t), hipMemcpyDeviceToHost));
    const int64_t npose = int64_t(ls->n_lig) * P->nchain;
    int apl = 1, dmax = 6;
    for (int32_t p : h) {
        if (p < 0 || p >= npose) return fail(UD2_ERR_ARG, "pose id out of range: " + std::to_string(p));
        apl = std::max(apl, int(ls->h_ligs[p / P->nchain].apl));
        dmax = std::max(dmax, 6 + int(ls->h_ligs[p / P->nchain].ntors));
    }
    FeatArgs A;
    A.L = ls->view();
    A.S = sc->view();
    A.P = pose_view(P);
    A.sel = sel_d;
    A.n_sel = n_sel;
    A.x = x_d;
    A.hdim_ld = odd_ld(dmax);
    A.lds_floats_per_wave = lds_round4(lds_prop_floats(apl, A.hdim_ld));
    UD2_HIP(launch_features(A, apl, static_cast<hipStream_t>(stream)));
    return UD2_OK;
}

// Learned-proposal MC: one persistent launch per atoms-per-lane class over a
// size-sorted queue, as ud2_mc; the chains keep their state on chip.
int ud2_lmc(const ud2_scene* sc, const ud2_ligset* ls, const ud2_poses* P, const ud2_lmc_params* prm,
            const ud2_mlp* mlp, void* stream) {
    int rc = check_poses(ls, P);
    if (rc) return rc;
    if (!prm) return fail(UD2_ERR_ARG, "null parameters");
    const ud2_mc_params& mc = prm->mc;
    rc = check_mode(sc, ls, mc.mode);
    if (rc) return rc;
    if (mc.mc_steps < 1 || mc.opt_steps < 0) return fail(UD2_ERR_ARG, "mc_steps must be >= 1, opt_steps >= 0");
    const int policy = prm->policy;
    if (policy < UD2_POLICY_PLAIN || policy > UD2_POLICY_COLLECT) return fail(UD2_ERR_ARG, "unknown policy");
    const int n_cand = policy == UD2_POLICY_PLAIN ? 1 : prm->n_cand;
    if (n_cand < 1 || n_cand > kMaxCand) return fail(UD2_ERR_ARG, "n_cand must be in 1..16");
    if (policy == UD2_POLICY_LEARNED && !(prm->sel_temp > 0.0f) && (prm->top_k < 1 || prm->top_k > n_cand))
        return fail(UD2_ERR_ARG, "top_k must be in 1..n_cand");
    if (!(prm->sel_temp >= 0.0f) || !std::isfinite(prm->sel_temp)) return fail(UD2_ERR_ARG, "sel_temp must be >= 0");
    if (prm->n_start > kMaxCand) return fail(UD2_ERR_ARG, "n_start must be <= 16");
    if (prm->n_start > 1 && policy == UD2_POLICY_COLLECT) return fail(UD2_ERR_ARG, "collect policy with n_start > 1");
    if (policy == UD2_POLICY_LEARNED && !mlp) return fail(UD2_ERR_ARG, "learned policy without a network");
    const bool feats = policy == UD2_POLICY_LEARNED || policy == UD2_POLICY_COLLECT;
    if (feats) {
        rc = check_mode(sc, ls, UD2_MODE_GRID);  // the features read the grid maps
        if (rc) return rc;
    }
    if (policy == UD2_POLICY_COLLECT && (!prm->collect_x_d || !prm->collect_y_d))
        return fail(UD2_ERR_ARG, "collect policy without output buffers");
    const int64_t npose = int64_t(ls->n_lig) * P->nchain;
    if (npose > (int64_t(1) << 30)) return fail(UD2_ERR_LIMIT, "too many chains");
    hipStream_t st = static_cast<hipStream_t>(stream);
    LmcArgs A;
    std::memset(&A, 0, sizeof(A));
    A.L = ls->view();
    A.S = sc->view();
    A.P = pose_view(P);
    A.mode = mc.mode;
    A.mc_steps = mc.mc_steps;
    A.opt_steps = mc.opt_steps;
    A.randomize = mc.randomize;
    A.seed = mc.seed;
    A.lig_index_base = mc.lig_index_base;
    A.policy = policy;
    A.n_cand = n_cand;
    A.top_k = prm->top_k;
    A.sel_temp = prm->sel_temp;
    A.n_start = prm->n_start < 1 ? 1 : prm->n_start;
    // hidden rows the network stages: the candidates (or starts) of one group, in halves of the MFMA tile
    A.a1_rows = std::max(A.n_cand, A.n_start) <= kGroup / 2 ? kGroup / 2 : kGroup;
    if (mlp) A.W = mlp->view();
    A.n_pose = npose;
    A.collect_x = prm->collect_x_d;
    A.collect_y = prm->collect_y_d;
    A.collect_e0 = prm->collect_e0_d;
    A.stats = reinterpret_cast<unsigned long long*>(mc.stats_d);
    UD2_HIP(launch_fill_i32(ls->d_counter, 0, kMaxApl + 1, st));
    const int cus = n_cus();
    for (int apl = kMaxApl; apl >= 1; apl--) {
        const int cnt = ls->cls_cnt[apl], dmax = ls->cls_dmax[apl];
        if (cnt == 0) continue;
        A.order = ls->d_order + ls->cls_pos[apl];
        A.n_order = cnt;
        A.counter = ls->d_counter + apl;
        A.hdim_ld = odd_ld(dmax);
        // While candidates are scored the energy's LDS is idle: the 16 bf16
        // candidate rows (640 floats) take the coordinate / force / BFGS-start
        // area at the slice start, the feature scratch (8 floats per atom) and
        // the hidden layer (a1_rows x 264 bf16) the Hessian's. The torsion table
        // between them stays in use. With 8 hidden rows one-atom-per-lane ligands
        // fit six blocks (24 waves) per CU.
        const int head = lds_head_floats(apl, A.hdim_ld);
        // hidden-layer rows: those that fit below the accepted pose's parking slot (coordinate and
        // force tiles and the BFGS-start slot, idle while the network runs; the first rows overlay
        // the candidate rows, which the network reads into registers first) go at the slice start,
        // the others after the head
        const int row_floats = kA1Stride / 2;
        const int idle_floats = 7 * kWave * apl + (kWave * (3 * apl + 1) + 8);
        A.a1_split = std::min(A.a1_rows, idle_floats / row_floats);
        const int a1_floats = (A.a1_rows - A.a1_split) * row_floats;
        const int shared = feats ? std::max(dmax * A.hdim_ld, std::max(8 * kWave * apl, a1_floats)) : dmax * A.hdim_ld;
        static_assert(kGroup * kFeat / 2 <= 7 * kWave + kWave * 4 + 8, "candidate rows exceed the idle LDS");
        A.lfeat = 0;
        A.lscr = head;
        A.la1 = 0;
        A.la1b = head;
        A.lds_floats_per_wave = lds_round4(head + shared);
        const int lds_bytes = A.lds_floats_per_wave * kWavesPerBlock * int(sizeof(float));
        if (lds_bytes > 160 * 1024) return fail(UD2_ERR_LIMIT, "per-block LDS exceeds 160 KB");
        const int64_t items = int64_t(cnt) * P->nchain;
        const int64_t need = (items + kWavesPerBlock - 1) / kWavesPerBlock;
        const int64_t cap = int64_t(cus) * lmc_blocks_per_cu(apl, A.policy, A.mode, lds_bytes);
        const int nb = int(std::max<int64_t>(1, std::min(need, cap)));
        UD2_HIP(launch_lmc(A, apl, nb, st));
    }
    return UD2_OK;
}
