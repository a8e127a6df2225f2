// engine.hip — host engine and C ABI (include/lima.h) of the gfx950 LIMA_MD step.
//
// Replaces the reference's Engine (Engine.cuh:109-208; Engine.cu:9-132,
// 400-451): the engine owns all device memory (hipMalloc, no managed memory),
// runs the whole step — forces, integration, PBC, thermostat and the scheduled
// neighbour-list rebuild — on one HIP stream, and replays each rebuild cycle as
// a captured hipGraph.  Errors are status codes plus a device error word read
// once per lima_step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/lima.h"
#include "adjoint.h"
#include "device_buffer.h"
#include "kernels.h"

using namespace lima;

// Staging of lima_step_observed_noalloc (an energy series, [records][systems][kEnergyTerms]
// doubles then [records][systems] floats of lambda): a file-scope device array, one copy per
// device, held until the process ends, so that the entry point calls no allocator.  In host
// code `scratch` only names the symbol; its device address comes from hipGetSymbolAddress,
// looked up once per device at engine creation (scratch_address).  Every call on a device
// shares its copy: calls that overlap on one device race.
constexpr size_t kObservedScratchBytes = (size_t)4 << 20;
static __device__ __align__(256) unsigned char scratch[kObservedScratchBytes];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kScratchDevices] = {};

// the device address of `scratch` on the current device `device`; null past kScratchDevices
unsigned char* scratch_address(int device) {
    if (device < 0 || device >= kScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        const hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (rc != hipSuccess || !ptr)
            throw LimaError(LIMA_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(rc));
        g_scratch_ptr[device] = static_cast<unsigned char*>(ptr);
    }
    return g_scratch_ptr[device];
}

struct LaunchConfig {
    int spt = 1;                  // solvents per lane of the all-pairs role: 1 (a field of saved tunings, and reported)
    int chunk_particles = 0;      // target chain particles per solvent<-chain work item (0: by each system's size)
    int listed_grid = 0;          // wavefront pairs of the listed compound role (0: by the number of items)
    int use_graph = 1;
    int listed_lanes = 4;         // lanes per solvent of the listed solvent role: 4 (saved tunings may say 1: reported, the same role)
    int listed_packed = -1;       // compounds of <= 64 particles: the packed listed role (1), the plain one (0), or
                                  // (FP32) the plain one with small compounds' rows split (2); -1: by the number of compounds
    int fused_thermostat = 0;     // 0: the thermostat as its own kernel; 1: in the integrate launch's last blocks (saved tunings
                                  // may say 2, a second form when the integrators were two launches: reported, the same)
};

// Device buffers of lima_adjoint_run / lima_record_frames, grown on demand and
// kept with the engine.  N = chain + solvent particles, chain first.
struct AdjBufs {
    DBuf<float4> ck;          // [segments][2N]: chain pos, chain prev, solvent pos, solvent prev
    DBuf<int> ck_cc;          // [segments][NC + NC*cap_cc]: compound lists before the segment's rebuild
    DBuf<int> lists;          // [slots][list words]: slot 0 the entry lists, then a segment's periods
    DBuf<float4> X, Rs;       // [segment frames][N]: positions, 2 beta (F - F*)
    DBuf<float> Tc, Ts;       // [K][n][3] force targets of the call
    DBuf<double4> adj;        // [3][N] a_k, a_{k+1}, a_{k+2} in rotation (FP64)
    DBuf<float4> w;           // [N]
    DBuf<float4> gxc, gxs;    // position-gradient parts
    DBuf<float4> gpart;       // [work item][128] listed-term parts of the compound side
    DBuf<float> cfac, gE;     // [N] dt^2/m, [K][R] energy weights
    DBuf<int> prep;           // [N] system of each particle
    DBuf<double> beta, loss, gpar, efr, lacc;
    DBuf<uint32_t> mask;
    DBuf<int> mask_off, comp_of;
    int n_cchunks = 1, n_sslices = 1, comp_chunk = 1, comp_split = 1, solv_slice = kAdjRows;
    bool ready = false;
};

}  // namespace

struct lima_engine {
    // ---- configuration ----
    lima_run_params params{};
    LaunchConfig cfg;
    int R = 0;
    std::vector<ReplicaInfo> reps_h;
    int NC = 0, NCH = 0, NS = 0, NB = 0;
    int n_types = 1;              // atom types in use, counted from type 0
    int max_cn = 0, max_cb = 0, max_ca = 0, max_cd = 0;   // most particles, bonds, angles, dihedrals of a compound
    std::vector<int> sys_chain_begin, sys_solv_begin, sys_comp_begin;  // per system, into the concatenation
    int n_cells = 0, n_stiles = 0;
    int kmax = 0;                 // max solvent<-chain chunks in any replica
    int chunk_cap = kRowPad;      // rows of the largest chunk (LDS tile of the all-pairs kernel)
    size_t max_slots = 0;
    bool listed_split_all = false;   // every system's listed items are summed in parts
    size_t max_items = 0;         // most work items of the listed compound role that the systems can have
    std::vector<SCWork> scwork_h;
    std::vector<int> comp_off_h, comp_row_h;
    int device = 0;
    // host copies behind lima_get/set_parameters
    std::vector<lima_forcefield> ff_h;
    std::vector<BondD> bonds_h, brb_h;
    std::vector<AngleD> angles_h, bra_h;
    std::vector<int> bond_off_h, angle_off_h, brb_off_h, bra_off_h, br_rep_h;

    // ---- device buffers ----
    DBuf<ReplicaInfo> reps;
    DBuf<float4> cpos[2], cprev, cforce, fbridge;
    DBuf<uint32_t> intra_mask;
    DBuf<int> xoff;
    DBuf<int2> xent;
    DBuf<int> comp_off, comp_rep, comp_key;
    DBuf<int> comp_row, row_src;  // rows of the all-pairs kernel's tiles
    DBuf<float> comp_sphere;
    DBuf<int> bond_off, angle_off, dih_off, inc_off;
    DBuf<BondD> bonds;
    DBuf<AngleD> angles;
    DBuf<DihD> dihs;
    DBuf<uint32_t> inc;
    DBuf<int> br_off, br_glob, br_rep, brb_off, bra_off, brd_off;
    DBuf<BondD> brb;
    DBuf<AngleD> bra;
    DBuf<DihD> brd;
    DBuf<float4> spos[2], sprev, sforce;
    DBuf<int> solv_rep;
    DBuf<int4> stiles;
    DBuf<float> mass;
    DBuf<float4> tab_sc, tab_cs, tab_inter, tab_intra, tab_ss;
    DBuf<int> cc_cnt, cc_ids, cs_cnt, cs_ids, ss_cnt, ss_ids, seg_cnt;
    int max_segs = 1;
    DBuf<int> cw_off, cw_total;
    DBuf<int> item_comp;          // [max_slots] compound of each work item
    DBuf<int> run_off, run_cs_off, run_total, run_comp;   // runs of the packed listed kernel (compounds of <= 64 particles)
    DBuf<float2> tab_inter_ab, tab_intra_ab;   // [R*1024] lj_ab of tab_inter, tab_intra
    DBuf<float4> partC, partS, cloc;
    DBuf<I3> partC_fx, partS_fx, cloc_fx;
    DBuf<SCWork> scwork;
    DBuf<float> lambda, lambda_applied;
    DBuf<double> ke_comp, ke_stile, temperature, energy;
    DBuf<long long> step_count;   // per replica: steps done (the reference cadence thermostat reads it)
    DBuf<int> thermo_cnt, thermo_total;   // the thermostat in the integrators' last blocks
    bool thermo_ok = false;       // every system has integrator blocks for it
    int thermo_form() const { return thermo_ok ? cfg.fused_thermostat : 0; }
    bool thermo_fused() const { return thermo_form() != 0; }
    // While a graph of several steps is captured: the step being enqueued starts with the thermostat
    // of the one before, and leaves its own to the next.  Not where a force role reads or writes what
    // it does (the logs' step counter, the kernel clock).
    bool thermo_pending = false, thermo_deferred = false;
    bool can_defer() const { return !thermo_fused() && log_rep < 0 && !kclock_on; }
    // per-step logs (lima_step_logged): replica, slots per compound, ring length and rings
    int log_rep = -1, log_slots = 0, log_ring = 1;
    bool log_train = false;
    DBuf<float> log_data, train_data;
    // in-step timing of the all-pairs kernel (lima_set_kernel_clock)
    bool kclock_on = false;
    bool kclock_step = false;     // the step being enqueued is one the clock samples
    DBuf<unsigned long long> kclock;
    DBuf<uint32_t> err;
    DBuf<int> cell_cnt, cell_start, cell_cursor, cell_ids, solv_cell, cell_rep;
    DBuf<float4> ss_part, ss_img;
    DBuf<float> comp_cs_bound;
    AdjBufs adjb;
    // triples of the state or forces on their way (io_get, io_set): of four arrays, allocated with the
    // engine, so that its state can be read whatever has become of the device's memory since
    DBuf<float> io_dev;
    float* io_pinned = nullptr;
    uint32_t* err_pinned = nullptr;   // the error words as of the last fetch_errors

    // a step is two launches on this stream (force roles, then the integrators), the thermostat's
    // kernel unless it is fused, and the rebuild's launches where one follows
    hipStream_t stream = nullptr;
    hipEvent_t ev_t0 = nullptr, ev_t1 = nullptr;   // lima_step's device timer
    // Captured launch graphs: one whole rebuild cycle (replayed from its start), and one step
    // of each kind [parity][rebuild follows][clocked] for steps that do not start a cycle.
    // Both are captured together on the first stepping call after any change of shape.
    hipGraphExec_t graph_exec = nullptr;
    static constexpr int kStrip = 8;           // steps of a strip graph: without a rebuild, from either parity
    hipGraphExec_t strip_graph[2] = {};
    hipGraphExec_t step_graph[2][2][2] = {};
    bool graphs_ready = false;
    int graph_steps = 0;
    long long dev_step = -1;      // the device step counters' value after the queued work (-1: unknown)
    bool async_open = false;      // ev_t0 marks the start of steps queued by lima_step_async
    unsigned char* scratch_d = nullptr;   // this device's copy of `scratch` (no-alloc staging)

    // ---- run state ----
    int cur = 0;                  // ping-pong parity of the current state
    long long step = 0;
    long long since_rebuild = 0;
    double t_device_us = 0, t_rebuild_us = 0, t_host_us = 0;
    long long n_rebuilds = 0;
    std::string last_error;

    ~lima_engine() {
        drop_graphs();
        for (hipEvent_t e : {ev_t0, ev_t1})
            if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
        for (void* p : {(void*)io_pinned, (void*)err_pinned})
            if (p) (void)hipHostFree(p);
    }

    void create_streams() {
        HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        HIP_TRY(hipEventCreate(&ev_t0));
        HIP_TRY(hipEventCreate(&ev_t1));
    }

    // every captured graph holds the launch shape, buffers and logging switches of its capture
    void drop_graphs() {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        graph_exec = nullptr;
        for (hipGraphExec_t& g : strip_graph) {
            if (g) (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
        for (auto& a : step_graph)
            for (auto& b : a)
                for (hipGraphExec_t& g : b) {
                    if (g) (void)hipGraphExecDestroy(g);
                    g = nullptr;
                }
        graphs_ready = false;
    }

    StepArgs step_args(int parity) {
        StepArgs a{};
        a.reps = reps.p;
        a.n_replicas = R;
        a.cpos = cpos[parity].p;
        a.cpos_next = cpos[parity ^ 1].p;
        a.cprev = cprev.p;
        a.cforce = cforce.p;
        a.fbridge = fbridge.p;
        a.intra_mask = intra_mask.p;
        a.xoff = xoff.p;
        a.xent = xent.p;
        a.n_comp = NC;
        a.comp_off = comp_off.p;
        a.comp_rep = comp_rep.p;
        a.comp_key = comp_key.p;
        a.comp_sphere = comp_sphere.p;
        a.bond_off = bond_off.p; a.bonds = bonds.p;
        a.angle_off = angle_off.p; a.angles = angles.p;
        a.dih_off = dih_off.p; a.dihs = dihs.p;
        a.inc_off = inc_off.p; a.inc = inc.p;
        a.n_bridges = NB;
        a.br_off = br_off.p; a.br_glob = br_glob.p; a.br_rep = br_rep.p;
        a.brb_off = brb_off.p; a.brb = brb.p;
        a.bra_off = bra_off.p; a.bra = bra.p;
        a.brd_off = brd_off.p; a.brd = brd.p;
        a.n_solv = NS;
        a.spos = spos[parity].p;
        a.spos_next = spos[parity ^ 1].p;
        a.sprev = sprev.p;
        a.sforce = sforce.p;
        a.solv_rep = solv_rep.p;
        a.stiles = stiles.p;
        a.mass = mass.p;
        a.tab_sc = tab_sc.p; a.tab_cs = tab_cs.p; a.tab_inter = tab_inter.p; a.tab_intra = tab_intra.p; a.tab_ss = tab_ss.p;
        a.tab_inter_ab = tab_inter_ab.p;
        a.tab_intra_ab = tab_intra_ab.p;
        a.cap_cc = params.max_compound_neighbors;
        a.cap_cs = params.max_compound_solvents;
        a.cap_ss = params.max_solvent_neighbors;
        a.cc_cnt = cc_cnt.p; a.cc_ids = cc_ids.p;
        a.cs_cnt = cs_cnt.p; a.cs_ids = cs_ids.p;
        a.ss_cnt = ss_cnt.p; a.ss_ids = ss_ids.p; a.ss_ld = ss_ld();
        a.ss_part = ss_part.p; a.ss_img = ss_img.p;
        a.cw_off = cw_off.p; a.cw_total = cw_total.p; a.item_comp = item_comp.p;
        a.run_off = run_off.p; a.run_cs_off = run_cs_off.p; a.run_total = run_total.p; a.run_comp = run_comp.p;
        a.partC = partC.p; a.partC_fx = partC_fx.p;
        a.cloc = cloc.p; a.cloc_fx = cloc_fx.p;
        a.partS = partS.p; a.partS_fx = partS_fx.p;
        a.scwork = scwork.p; a.n_scwork = (int)scwork_h.size();
        a.chunk_cap = chunk_cap;
        a.comp_row = comp_row.p;
        a.row_src = row_src.p;
        a.lambda = lambda.p;
        a.ke_comp = ke_comp.p;
        a.ke_stile = ke_stile.p;
        a.ke_ref = params.thermostat == LIMA_THERMOSTAT_REFERENCE ? 1 : 0;
        a.log_rep = log_rep;
        a.log_slots = log_slots;
        a.log_ring = log_ring;
        a.step_count = step_count.p;
        a.thermo_cnt = thermo_fused() ? thermo_cnt.p : nullptr;
        a.thermo_total = thermo_total.p;
        a.lambda_next = lambda.p;
        a.lambda_applied = lambda_applied.p;
        a.temperature = temperature.p;
        a.step_count_w = step_count.p;
        a.thermo_mode = params.thermostat;
        a.kclock = kclock_on && kclock_step ? kclock.p : nullptr;
        a.log_data = log_data.p;
        a.train_data = log_rep >= 0 && log_train ? train_data.p : nullptr;
        a.energy = energy.p;
        a.err = err.p;
        a.enable_solvents = params.enable_solvents;
        a.enable_dihedrals = params.enable_dihedrals;
        a.loc_nb = max_cb; a.loc_na = max_ca; a.loc_nd = max_cd;
        a.n_types = n_types;
        a.local_stage = (int)local_lds_bytes<64>(max_cb, max_ca, max_cd);
        a.listed_split = listed_form() == 2 ? 1 : 0;
        return a;
    }

    NlistArgs nlist_args(int parity) {
        NlistArgs a{};
        a.reps = reps.p;
        a.cpos = cpos[parity].p;
        a.spos = spos[parity].p;
        a.n_comp = NC;
        a.n_solv = NS;
        a.comp_off = comp_off.p; a.comp_rep = comp_rep.p; a.comp_key = comp_key.p; a.comp_sphere = comp_sphere.p;
        a.solv_rep = solv_rep.p;
        a.cutoff = params.cutoff;
        a.cap_cc = params.max_compound_neighbors;
        a.cap_cs = params.max_compound_solvents;
        a.cap_ss = params.max_solvent_neighbors;
        a.cc_cnt = cc_cnt.p; a.cc_ids = cc_ids.p;
        a.seg_cnt = seg_cnt.p; a.max_segs = max_segs;
        a.cs_cnt = cs_cnt.p; a.cs_ids = cs_ids.p;
        a.ss_cnt = ss_cnt.p; a.ss_ids = ss_ids.p; a.ss_ld = ss_ld();
        a.n_cells = n_cells;
        a.cell_cnt = cell_cnt.p; a.cell_start = cell_start.p; a.cell_cursor = cell_cursor.p;
        a.cell_ids = cell_ids.p; a.solv_cell = solv_cell.p;
        a.cell_rep = cell_rep.p;
        a.comp_cs_bound = comp_cs_bound.p;
        a.cw_off = cw_off.p; a.cw_total = cw_total.p; a.item_comp = item_comp.p;
        a.run_len = pack_ppl() ? cc_run(pack_ppl()) : 0;
        a.run_off = run_off.p; a.run_cs_off = run_cs_off.p; a.run_total = run_total.p; a.run_comp = run_comp.p;
        a.err = err.p;
        a.enable_solvents = params.enable_solvents;
        return a;
    }

    // solvent list row stride: capacity rounded up to the 16 ids that a quad reads at a time
    int ss_ld() const { return (params.max_solvent_neighbors + kListChunk - 1) / kListChunk * kListChunk; }

    // ---- launches ----
    // Target rows of a system's all-pairs chunks.  The sums of a chunk are added to the next one's,
    // so the choice depends on the system alone and not on what is batched with it: 1024 rows where
    // that leaves about one block a wavefront slot (1000 of 256 threads), else 512 or 256.  Alone, us,
    // at 1024, 512 and 256 rows: 46 tiles x 2,700 particles 46.7, 24.6, 17.2; the demo 49.8, 26.2, 14.6;
    // production (1,235 blocks at 1024) 121, 116, 110, where its step is the shortest at 1024; the
    // 18 nm box 2,552, 2,575, 2,675 (the rows' staging).  128 rows gained small systems 2-3% and cost
    // batches as much.
    int chunk_target(const ReplicaInfo& ri) const {
        if (cfg.chunk_particles > 0) return std::min(cfg.chunk_particles, kChunkParticles);
        const int tiles = (ri.solv_end - ri.solv_begin + kStepThreads - 1) / kStepThreads;
        const int rows = comp_row_h[ri.comp_end] - comp_row_h[ri.comp_begin];
        int target = 1024;
        while (target > 256 && (long long)tiles * ((rows + target - 1) / target) < 1000) target /= 2;
        return target;
    }

    // Work list of the all-pairs role: per replica, solvent tiles of 256 x chunks of consecutive
    // compounds; heaviest items first.  Sizes the partial buffer and the LDS tile.  If there is no
    // memory for it, the engine keeps the list that it had.
    void build_scwork() {
        const int tile_sz = kStepThreads;
        std::vector<SCWork> work;
        std::vector<int> counts(R);
        int most = 0, cap = kRowPad;
        for (int r = 0; r < R; r++) {
            const ReplicaInfo& ri = reps_h[r];
            const int target = chunk_target(ri);
            std::vector<std::pair<int, int>> chunks;
            int c = ri.comp_begin;
            while (c < ri.comp_end) {
                int c1 = c, np = 0;
                while (c1 < ri.comp_end && (c1 - c) < kChunkCompounds) {
                    const int n = comp_row_h[c1 + 1] - comp_row_h[c1];
                    if (np > 0 && np + n > target) break;
                    np += n;
                    c1++;
                }
                cap = std::max(cap, np);
                chunks.push_back({c, c1});
                c = c1;
            }
            if (ri.solv_end == ri.solv_begin) chunks.clear();
            counts[r] = (int)chunks.size();
            most = std::max(most, counts[r]);
            for (int t0 = ri.solv_begin; t0 < ri.solv_end; t0 += tile_sz)
                for (int k = 0; k < (int)chunks.size(); k++)
                    work.push_back(SCWork{r, t0, std::min(t0 + tile_sz, ri.solv_end), chunks[k].first, chunks[k].second, k, 0, 0});
        }
        std::stable_sort(work.begin(), work.end(), [&](const SCWork& x, const SCWork& y) {
            const long long wx = (long long)(x.solv_end - x.solv_begin) * (comp_off_h[x.comp_end] - comp_off_h[x.comp_begin]);
            const long long wy = (long long)(y.solv_end - y.solv_begin) * (comp_off_h[y.comp_end] - comp_off_h[y.comp_begin]);
            return wx > wy;
        });
        const size_t need = std::max<size_t>(1, (size_t)most * std::max(NS, 1));
        const bool fixed = params.accumulation == LIMA_ACCUM_FIXED64;
        drop_graphs();   // captured launches name the buffers' addresses
        partS_fx.grow(fixed ? need : 1);
        partS.grow(fixed ? 1 : need);
        scwork.grow(std::max<size_t>(work.size(), 1));
        if (!work.empty()) HIP_TRY(hipMemcpy(scwork.p, work.data(), work.size() * sizeof(SCWork), hipMemcpyHostToDevice));
        scwork_h.swap(work);
        kmax = most;
        chunk_cap = cap;
        for (int r = 0; r < R; r++) reps_h[r].chunk_count = counts[r];
    }

    // a failed growth that could not even give the former buffers back
    void check_work_list() const {
        const size_t partials = params.accumulation == LIMA_ACCUM_FIXED64 ? partS_fx.n : partS.n;
        if (partials < (size_t)kmax * NS || scwork.n < scwork_h.size())
            throw LimaError(LIMA_E_HIP, "the all-pairs work list has no device memory");
    }

    // particles per lane of the packed listed role (compounds of at most 16, 32, 64 particles), 0: plain only
    int pack_ppl() const { return max_cn <= 16 ? 1 : max_cn <= 32 ? 2 : max_cn <= 64 ? 4 : 0; }

    // The listed compound role's form.  Packed and plain give the same sums; the packed one works on
    // 16 lanes a compound and wins once there are enough compounds to fill the device with it (256
    // replicas, 5,000 compounds: 350 us against 1,117; the demo, 36 compounds: 49 against 24).
    int listed_form() const {
        if (!pack_ppl()) return 0;
        if (cfg.listed_packed >= 0) return cfg.listed_packed == 2 && params.accumulation == LIMA_ACCUM_FIXED64 ? 0 : cfg.listed_packed;
        return NC >= 512 ? 1 : 0;
    }
    // A block per item of the plain listed compound role for at most kListedWideItems of them, which
    // a wavefront each would leave most of the device idle (alone, us, a wavefront and a block an
    // item: 2 compounds of 128 and 3,000 solvents 22.1 and 9.3, the demo 15.5 and 12.4, 36 compounds
    // of 75 and 11,800 solvents 30 and 23), where every system's items are split.
    static constexpr size_t kListedWideItems = 4096;
    static constexpr size_t kListedNeighbors = 256, kListedSolvents = 16384;   // the capacities that callers start from (RunParams)
    bool listed_wide() const { return listed_form() == 0 && listed_split_all && max_items <= kListedWideItems; }
    // blocks of the listed compound role: a wavefront per item up to 16,384 wavefronts, which then take several
    int listed_blocks() const {
        if (listed_wide()) return (int)max_items;
        if (cfg.listed_grid > 0) return std::max(1, cfg.listed_grid / 2);
        return (int)std::min<size_t>(4096, (max_items + 3) / 4);
    }

    enum Role { kRoleListedSolvents = 1, kRoleLocal = 2, kRoleBridges = 4, kRoleAllPairs = 8, kRoleListed = 16, kRoleEvery = 31 };

    ForceBlocks force_blocks(int roles) const {
        const bool solv = params.enable_solvents && NS > 0;
        ForceBlocks f{};
        // a block per 64 solvents, or (65,536 and up, where that leaves the list blocks as many as the
        // others and no room to spread them) per tile of 256
        f.solvent_rounds = NS > 65536 ? 4 : 1;
        f.solvent_items = n_stiles * (256 / kQuadSolvents / f.solvent_rounds);
        f.local_waves = max_cn <= 64 && 4 * local_lds_bytes<64>(max_cb, max_ca, max_cd) <= 40960 ? 1 : 0;
        if (solv && (roles & kRoleListedSolvents)) f.listed_solvents = xcd_grid(f.solvent_items);
        if (roles & kRoleLocal) f.local = f.local_waves ? (NC + 3) / 4 : NC;
        if (roles & kRoleBridges) f.bridges = (NB + 3) / 4;
        if (solv && (roles & kRoleAllPairs)) f.all_pairs = (int)scwork_h.size();
        f.listed_wide = listed_wide() ? 1 : 0;
        if (NC > 0 && (roles & kRoleListed)) f.listed = listed_blocks();
        // The packed form's blocks, bound by LDS and the gathers of their rows, go among the all-pairs
        // blocks, and the solvent-list groups among everything but the last 2,048 blocks.  Periods are
        // odd: the dispatcher deals blocks out to 8 XCDs of 32 CUs in turn, so an even period puts one
        // role on every second CU (256 replicas, us a step: 1065 with the list blocks first, 1332 and
        // 1643 at periods 2 and 4, 1012 and 977 at 3 and 5).
        auto even = [](int v) { return v - v % 2; };
        f.mix = f.listed > 0 && listed_form() == 1 ? even(f.all_pairs / f.listed) : 0;
        f.thermostat = thermo_pending && roles == kRoleEvery ? (R + 3) / 4 : 0;
        const int others = (f.local + f.bridges + f.all_pairs + f.listed) / kXcds, lists = f.listed_solvents / kXcds;
        f.spread = lists > 0 ? even(std::max(0, others - 256) / lists) : 0;
        return f;
    }

    // LDS of the force launch: the most that any of its roles takes
    size_t force_lds(const ForceBlocks& f, int ppl) const {
        size_t n = 16;
        if (f.local) n = std::max(n, f.local_waves ? 4 * local_lds_bytes<64>(max_cb, max_ca, max_cd)
                                                   : local_lds_bytes<kStepThreads>(max_cb, max_ca, max_cd));
        if (f.bridges) n = std::max(n, 4 * sizeof(BridgeStage));
        if (f.all_pairs) n = std::max(n, all_pairs_lds_bytes(chunk_cap));
        if (f.listed)
            n = std::max(n, ppl == 0 ? kListedLds
                                     : 4 * (ppl == 1 ? sizeof(PackedStage<1>) : ppl == 2 ? sizeof(PackedStage<2>) : sizeof(PackedStage<4>)) +
                                           (size_t)n_types * n_types * sizeof(float2));
        return n;
    }

    template <bool FIXED, bool ENERGY> void launch_roles(const StepArgs& a, int roles) {
        ForceBlocks f = force_blocks(roles);
        const int n = f.listed_solvents + xcd_grid(f.thermostat + f.local + f.bridges + f.all_pairs + f.listed);
        if (n == 0) return;
        if (f.all_pairs) check_work_list();
        const int ppl = listed_form() == 1 ? pack_ppl() : 0;
        const size_t lds = force_lds(f, ppl);
        const dim3 grid = grid_of(n);
        f.width = (int)grid.x;
        switch (ppl) {
            case 1: step_forces_kernel<FIXED, ENERGY, 1><<<grid, kStepThreads, lds, stream>>>(a, f); break;
            case 2: step_forces_kernel<FIXED, ENERGY, 2><<<grid, kStepThreads, lds, stream>>>(a, f); break;
            case 4: step_forces_kernel<FIXED, ENERGY, 4><<<grid, kStepThreads, lds, stream>>>(a, f); break;
            default: step_forces_kernel<FIXED, ENERGY, 0><<<grid, kStepThreads, lds, stream>>>(a, f);
        }
    }
    template <bool ADVANCE, bool FIXED, bool ENERGY> void launch_integrate(const StepArgs& a, bool compounds, bool solvents) {
        const int cb = compounds ? (NC + 1) / 2 : 0, tiles = solvents && params.enable_solvents && NS > 0 ? n_stiles : 0;
        if (cb + tiles == 0) return;
        // 40 steps of the demo (36 compounds) 1,000 -> 982 us with 16 partials in flight, 20 of 256
        // replicas (7,000) 21.16 -> 21.36 ms
        if (!FIXED && NC <= 1024) step_integrate_kernel<ADVANCE, FIXED, ENERGY, 16><<<cb + tiles, kStepThreads, 0, stream>>>(a, cb);
        else step_integrate_kernel<ADVANCE, FIXED, ENERGY, 8><<<cb + tiles, kStepThreads, 0, stream>>>(a, cb);
    }

    // one force pass (and integration when ADVANCE)
    template <bool ADVANCE, bool FIXED, bool ENERGY> void launch_forces(int parity) {
        const StepArgs a = step_args(parity);
        launch_roles<FIXED, ENERGY>(a, kRoleEvery);
        launch_integrate<ADVANCE, FIXED, ENERGY>(a, true, true);
    }

    // one step; with `energy` the force pass also accumulates the FP64 energy
    // terms (the caller clears the energy buffer first)
    void launch_step(int parity, bool energy = false) {
        const bool fx = params.accumulation == LIMA_ACCUM_FIXED64;
        if (energy) {
            if (fx) launch_forces<true, true, true>(parity);
            else launch_forces<true, false, true>(parity);
        } else {
            if (fx) launch_forces<true, true, false>(parity);
            else launch_forces<true, false, false>(parity);
        }
        // with solvents disabled the solvent state is carried across the ping-pong unchanged
        if (!params.enable_solvents && NS > 0)
            HIP_TRY(hipMemcpyAsync(spos[parity ^ 1].p, spos[parity].p, NS * sizeof(float4), hipMemcpyDeviceToDevice, stream));
        if (!thermo_fused() && !thermo_deferred)
            thermostat_kernel<<<R, 64, 0, stream>>>(reps.p, R, ke_comp.p, ke_stile.p, lambda.p, lambda_applied.p,
                                                temperature.p, step_count.p, params.thermostat,
                                                kclock_on && kclock_step ? kclock.p : nullptr);
        if (dev_step >= 0) dev_step++;   // the thermostat kernel advances the device step counters
    }

    // compound lists, then the solvent cell pipeline and its lists, then the work list
    void launch_rebuild(int parity) {
        NlistArgs a = nlist_args(parity);
        const bool solv = params.enable_solvents && NS > 0;
        if (NC > 0) nl_compound_compound_kernel<<<NC, 64, 0, stream>>>(a);
        if (solv) {
            const dim3 blocks = grid_of((long long)NC * max_segs + (NS + 255) / 256);
            nl_count_kernel<<<blocks, 256, 0, stream>>>(a);
            nl_cell_scan_kernel<<<1, 1024, 0, stream>>>(a);
            nl_write_kernel<<<blocks, 256, 0, stream>>>(a);
            nl_cell_sort_kernel<<<grid_of(n_cells), 256, 0, stream>>>(a);
            nl_solvent_solvent_kernel<<<grid_of(xcd_grid(n_cells)), kSolventListThreads, 0, stream>>>(a);
        }
        launch_work_list(a, stream);
    }

    // the listed work items of the current lists: per-compound offsets, then each item's compound
    void launch_work_list(const NlistArgs& a, hipStream_t st) {
        if (NC <= 0) return;
        nl_work_kernel<<<1, 1024, 0, st>>>(a);
        if (NC > kWorkItemsInPlace) nl_item_kernel<<<NC, 64, 0, st>>>(a);
    }

    // lj_ab of the inter- and intra-compound tables (after any change of them)
    void fill_ab_tables() {
        const int n = R * kMaxTypes * kMaxTypes;
        ab_table_kernel<<<(n + 255) / 256, 256, 0, stream>>>(tab_inter.p, tab_inter_ab.p, n);
        ab_table_kernel<<<(n + 255) / 256, 256, 0, stream>>>(tab_intra.p, tab_intra_ab.p, n);
        HIP_TRY(hipStreamSynchronize(stream));
    }

    int cycle_steps() const {
        const int iv = params.nlist_interval > 0 ? params.nlist_interval : 1;
        return (iv % 2 == 0) ? iv : 2 * iv;
    }

    // What distinguishes one step's launches from another's: the state parity, whether the
    // scheduled rebuild (Engine::hostMaster, Engine.cu:49-75) follows it, and whether the kernel
    // clock samples it (one step per list period: the second, clear of the rebuild's tail).
    struct StepKind {
        int parity;
        bool rebuild;
        bool clocked;
    };
    StepKind next_kind() const {
        const int iv = params.nlist_interval;
        const int pick = iv > 1 ? 1 : 0;
        StepKind k;
        k.parity = cur;
        k.rebuild = iv > 0 && since_rebuild + 1 >= iv;
        k.clocked = kclock_on && (iv > 0 ? since_rebuild == pick : step % 8 == 0);
        return k;
    }
    void enqueue_kind(const StepKind& k) {
        kclock_step = k.clocked;
        launch_step(k.parity);
        kclock_step = false;   // steps launched directly (observed, adjoint) are never clocked
        if (k.rebuild) launch_rebuild(k.parity ^ 1);
    }
    void advance(const StepKind& k) {
        cur ^= 1;
        step++;
        since_rebuild++;
        if (k.rebuild) {
            since_rebuild = 0;
            n_rebuilds++;
        }
    }
    // one step plus the rebuild it schedules
    void enqueue_one() {
        const StepKind k = next_kind();
        enqueue_kind(k);
        advance(k);
    }

    void enqueue_many(int n) {
        struct Reset {
            lima_engine* E;
            ~Reset() { E->thermo_pending = E->thermo_deferred = false; }
        } reset{this};
        for (int i = 0; i < n; i++) {
            thermo_pending = can_defer() && i > 0;
            thermo_deferred = can_defer() && i + 1 < n;
            enqueue_one();
        }
    }

    template <typename F> hipGraphExec_t capture(F&& enqueue) {
        hipGraph_t g;
        HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        enqueue();
        HIP_TRY(hipStreamEndCapture(stream, &g));
        hipGraphExec_t ex = nullptr;
        HIP_TRY(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
        HIP_TRY(hipGraphDestroy(g));
        // the one-time upload of the executable graph here, not inside its first replay
        HIP_TRY(hipGraphUpload(ex, stream));
        return ex;
    }

    // Captures the cycle graph and every step kind that can occur, so that no later stepping
    // call captures: replays of either kind can follow each other in any order.
    void ensure_graphs() {
        if (graphs_ready) return;
        drop_graphs();
        check_work_list();   // not inside a capture
        const int save_cur = cur;
        const long long save_step = step, save_since = since_rebuild, save_nr = n_rebuilds, save_dev = dev_step;
        const int iv = params.nlist_interval;
        if (iv > 0) {
            // the whole cycle, from parity 0 and a fresh rebuild cycle
            const int n = cycle_steps();
            cur = 0;
            since_rebuild = 0;
            graph_exec = capture([&] { enqueue_many(n); });
            graph_steps = n;
        }
        // strips of a longer list period (or of none), for runs that the cycle does not fit
        for (int p = 0; p < 2 && can_defer() && (iv <= 0 || iv > kStrip); p++) {
            cur = p;
            since_rebuild = 0;
            strip_graph[p] = capture([&] { enqueue_many(kStrip); });
        }
        for (int p = 0; p < 2; p++)
            for (int rb = 0; rb < (iv > 0 ? 2 : 1); rb++)
                for (int ck = 0; ck < (kclock_on ? 2 : 1); ck++) {
                    const StepKind k{p, rb != 0, ck != 0};
                    step_graph[p][rb][ck] = capture([&] { enqueue_kind(k); });
                }
        cur = save_cur;
        step = save_step;
        since_rebuild = save_since;
        n_rebuilds = save_nr;
        dev_step = save_dev;
        graphs_ready = true;
    }

    // the device step counters follow the host's count (set before any stepping call enqueues)
    void sync_step_count() {
        set_step_count_kernel<<<(R + 63) / 64, 64, 0, stream>>>(step_count.p, R, step);
        dev_step = step;
    }

    // allow_capture false: replays only graphs already built, else launches directly
    void enqueue_steps(int n, bool allow_capture = true) {
        if (n <= 0) return;
        if (dev_step != step) sync_step_count();
        const bool graphs = cfg.use_graph != 0 && (allow_capture || graphs_ready);
        if (graphs) ensure_graphs();
        const int cyc = cycle_steps();
        while (n > 0) {
            if (graphs && graph_exec && cur == 0 && since_rebuild == 0 && n >= cyc) {
                HIP_TRY(hipGraphLaunch(graph_exec, stream));
                step += cyc;
                dev_step += cyc;
                n_rebuilds += cyc / params.nlist_interval;
                n -= cyc;
                continue;
            }
            if (graphs && strip_graph[cur] && n >= kStrip &&
                (params.nlist_interval <= 0 || since_rebuild + kStrip < params.nlist_interval)) {
                HIP_TRY(hipGraphLaunch(strip_graph[cur], stream));
                step += kStrip;
                dev_step += kStrip;
                since_rebuild += kStrip;
                n -= kStrip;
                continue;
            }
            const StepKind k = next_kind();
            if (graphs) {
                HIP_TRY(hipGraphLaunch(step_graph[k.parity][k.rebuild ? 1 : 0][k.clocked ? 1 : 0], stream));
                dev_step++;
            } else {
                enqueue_kind(k);
            }
            advance(k);
            n--;
        }
    }

    // the error words' copy, in stream order behind the work that may set them
    void fetch_errors() {
        if (!err_pinned) HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&err_pinned), 4 * sizeof(uint32_t), 0));
        HIP_TRY(hipMemcpyAsync(err_pinned, err.p, 4 * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    }
    int check_errors() {
        fetch_errors();
        HIP_TRY(hipStreamSynchronize(stream));
        return fetched_errors();
    }
    int fetched_errors() {
        const uint32_t* e = err_pinned;
        if (e[0] == 0) return LIMA_OK;
        HIP_TRY(hipMemset(err.p, 0, 4 * sizeof(uint32_t)));
        char buf[256];
        if (e[0] & kErrCapacity) {
            snprintf(buf, sizeof(buf), "neighbour list capacity exceeded (needed: compound-compound %u, compound-solvent %u, solvent %u)",
                     e[1], e[2], e[3]);
            last_error = buf;
            return LIMA_E_CAPACITY;
        }
        if (e[0] & kErrCriticalForce) { last_error = "critical force |F| > 2e12 on a chain particle"; return LIMA_E_CRITICAL_FORCE; }
        if (e[0] & kErrNaN) { last_error = "NaN solvent position"; return LIMA_E_NAN; }
        last_error = "unknown device error";
        return LIMA_E_HIP;
    }
};

namespace {

// Smallest non-negative float x with sqrtf(x) >= t.  sqrtf is correctly rounded
// (here and on the device) and monotone, so  sqrtf(d2) < t  <=>  d2 < sqrt_bound(t):
// the neighbour tests compare squared distances with the exact same outcome.
float sqrt_bound(float t) {
    uint32_t lo = 0, hi = 0x7f800000u;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        float x;
        std::memcpy(&x, &mid, 4);
        if (std::sqrt(x) >= t) hi = mid;
        else lo = mid + 1;
    }
    float r;
    std::memcpy(&r, &lo, 4);
    return r;
}

// LJ parameters of one call site: sigma^2 and 24*eps rounded as the reference
// rounds sigma*sigma and 24.f*epsilon (Engine.cu:488-490), -2*(24 eps), and the
// mixed sigma itself (d sigma^2 / d sigma_type = sigma for the arithmetic sigma rule).
float4 pair_params(float sigma, float eps) {
    const float e24 = 24.f * eps;
    return make_float4(sigma * sigma, e24, -2.0f * e24, sigma);
}

// type tables of one system (mixing per call site, Engine.cu:643-646, 668-670,
// 689-691, 711-713, 724-727): [32] masses, [32] solvent <- type, [32] type <-
// solvent, [32*32] inter-compound, [32*32] intra-compound, [1] solvent-solvent
void fill_tables(const lima_particle_params* pp, float* mass, float4* tsc, float4* tcs, float4* tinter, float4* tintra,
                 float4* tss) {
    for (int t = 0; t < kMaxTypes; t++) {
        mass[t] = pp[t].mass;
        float sg = (pp[0].sigma + pp[t].sigma) * 0.5f;
        float ep = (pp[0].epsilon + pp[t].epsilon) * 0.5f;
        tsc[t] = pair_params(sg, ep);
        float epg = sqrtf(pp[t].epsilon * pp[0].epsilon);
        tcs[t] = pair_params(sg, epg);
        for (int u = 0; u < kMaxTypes; u++) {
            float su = (pp[t].sigma + pp[u].sigma) * 0.5f;
            float ea = (pp[t].epsilon + pp[u].epsilon) * 0.5f;
            float eg = sqrtf(pp[t].epsilon * pp[u].epsilon);
            tinter[t * 32 + u] = pair_params(su, ea);
            tintra[t * 32 + u] = pair_params(su, eg);
        }
    }
    *tss = pair_params(pp[0].sigma, pp[0].epsilon);
}

void validate_and_build(lima_engine* E, const lima_system* sys, int nsys) {
    const lima_run_params& P = E->params;
    std::vector<float> cs_bound;
    std::vector<int> cell_rep_h;
    if (nsys <= 0) throw LimaError(LIMA_E_ARG, "n_systems must be >= 1");
    if (!(P.cutoff > 0)) throw LimaError(LIMA_E_ARG, "cutoff must be > 0");
    if (P.thermostat < LIMA_THERMOSTAT_NONE || P.thermostat > LIMA_THERMOSTAT_REFERENCE)
        throw LimaError(LIMA_E_ARG, "unknown thermostat");
    if (P.max_compound_neighbors <= 0 || P.max_compound_solvents <= 0 || P.max_solvent_neighbors <= 0)
        throw LimaError(LIMA_E_ARG, "capacities must be > 0");
    std::vector<float4> cpos, cprev, spos, sprev;
    std::vector<uint32_t> imask;
    std::vector<int> xoff{0};
    std::vector<int2> xent;
    std::vector<int> comp_off{0}, comp_rep, comp_key;
    std::vector<float> comp_sphere;
    std::vector<int> bond_off{0}, angle_off{0}, dih_off{0}, inc_off{0};
    std::vector<BondD> bonds;
    std::vector<AngleD> angles;
    std::vector<DihD> dihs;
    std::vector<uint32_t> inc;
    std::vector<int> br_off{0}, br_glob, br_rep, brb_off{0}, bra_off{0}, brd_off{0};
    std::vector<BondD> brb;
    std::vector<AngleD> bra;
    std::vector<DihD> brd;
    std::vector<int> solv_rep;
    std::vector<float> mass(nsys * kMaxTypes);
    std::vector<float4> tsc(nsys * kMaxTypes), tcs(nsys * kMaxTypes), tinter(nsys * 1024), tintra(nsys * 1024), tss(nsys);
    E->reps_h.clear();
    E->ff_h.clear();
    E->sys_chain_begin.clear(); E->sys_solv_begin.clear(); E->sys_comp_begin.clear();
    std::vector<int> bridge_owner;

    for (int r = 0; r < nsys; r++) {
        const lima_system& s = sys[r];
        if (!(s.box_len > 0) || !(s.dt > 0)) throw LimaError(LIMA_E_ARG, "box_len and dt must be > 0");
        if (s.n_compounds < 0 || s.n_solvents < 0 || s.n_bridges < 0) throw LimaError(LIMA_E_ARG, "negative counts");
        ReplicaInfo ri{};
        ri.L = s.box_len;
        ri.half = s.box_len * 0.5f;
        ri.dt = s.dt;
        ri.tau = P.thermostat_tau > 0 ? P.thermostat_tau : 1.0;
        ri.T0 = s.thermostat_target;
        const int cb = (int)comp_rep.size();
        const int chb = (int)cpos.size();
        const int sb = (int)spos.size();
        E->sys_comp_begin.push_back(cb);
        E->sys_chain_begin.push_back(chb);
        E->sys_solv_begin.push_back(sb);
        ri.comp_begin = cb; ri.comp_end = cb + s.n_compounds;
        const int nchain = s.n_compounds > 0 ? s.compound_offset[s.n_compounds] : 0;
        ri.chain_begin = chb; ri.chain_end = chb + nchain;
        ri.solv_begin = sb; ri.solv_end = sb + s.n_solvents;
        fill_tables(s.forcefield.particle_parameters, &mass[r * kMaxTypes], &tsc[r * kMaxTypes], &tcs[r * kMaxTypes],
                    &tinter[r * 1024], &tintra[r * 1024], &tss[r]);
        E->ff_h.push_back(s.forcefield);
        // compounds
        for (int c = 0; c < s.n_compounds; c++) {
            const int o0 = s.compound_offset[c], o1 = s.compound_offset[c + 1];
            const int n = o1 - o0;
            if (n <= 0 || n > kCompoundBlock) throw LimaError(LIMA_E_CAPACITY, "compound size must be 1..128 particles");
            if (s.key_particle_index[c] < 0 || s.key_particle_index[c] >= n) throw LimaError(LIMA_E_ARG, "key_particle_index out of range");
            comp_off.push_back(comp_off.back() + n);
            comp_rep.push_back(r);
            comp_key.push_back(s.key_particle_index[c]);
            comp_sphere.push_back(s.confining_particle_sphere[c]);
            // threshold of the compound-solvent test, C + (r + C) (Engine.cu:182, 231)
            cs_bound.push_back(sqrt_bound(P.cutoff + (s.confining_particle_sphere[c] + P.cutoff)));
            const int gbase = chb + o0;
            const int nbd = s.bond_offset[c + 1] - s.bond_offset[c];
            const int nan = s.angle_offset[c + 1] - s.angle_offset[c];
            const int ndh = s.dihedral_offset[c + 1] - s.dihedral_offset[c];
            if (nbd > kMaxBondsPerCompound || nan > kMaxAnglesPerCompound || ndh > kMaxDihedralsPerCompound)
                throw LimaError(LIMA_E_CAPACITY, "too many bonded terms in a compound");
            E->max_cn = std::max(E->max_cn, n);
            E->max_cb = std::max(E->max_cb, nbd);
            E->max_ca = std::max(E->max_ca, nan);
            E->max_cd = std::max(E->max_cd, ndh);
            std::vector<std::vector<uint32_t>> pinc(n);
            for (int t = 0; t < nbd; t++) {
                const lima_pair_bond& b = s.bonds[s.bond_offset[c] + t];
                for (int k = 0; k < 2; k++) if ((int)b.atom_indexes[k] >= n) throw LimaError(LIMA_E_ARG, "bond index out of range");
                bonds.push_back(BondD{b.b0, b.kb, (int)b.atom_indexes[0], (int)b.atom_indexes[1]});
                for (int k = 0; k < 2; k++) pinc[b.atom_indexes[k]].push_back((0u << 30) | ((uint32_t)t << 2) | (uint32_t)k);
            }
            for (int t = 0; t < nan; t++) {
                const lima_angle_bond& b = s.angles[s.angle_offset[c] + t];
                for (int k = 0; k < 3; k++) if ((int)b.atom_indexes[k] >= n) throw LimaError(LIMA_E_ARG, "angle index out of range");
                angles.push_back(AngleD{b.theta_0, b.k_theta, (int)b.atom_indexes[0], (int)b.atom_indexes[1], (int)b.atom_indexes[2], 0});
                for (int k = 0; k < 3; k++) pinc[b.atom_indexes[k]].push_back((1u << 30) | ((uint32_t)t << 2) | (uint32_t)k);
            }
            for (int t = 0; t < ndh; t++) {
                const lima_dihedral_bond& b = s.dihedrals[s.dihedral_offset[c] + t];
                for (int k = 0; k < 4; k++) if ((int)b.atom_indexes[k] >= n) throw LimaError(LIMA_E_ARG, "dihedral index out of range");
                dihs.push_back(DihD{b.phi_0, b.k_phi, (int)b.n, (int)b.atom_indexes[0], (int)b.atom_indexes[1],
                                    (int)b.atom_indexes[2], (int)b.atom_indexes[3], 0});
                for (int k = 0; k < 4; k++) pinc[b.atom_indexes[k]].push_back((2u << 30) | ((uint32_t)t << 2) | (uint32_t)k);
            }
            bond_off.push_back((int)bonds.size());
            angle_off.push_back((int)angles.size());
            dih_off.push_back((int)dihs.size());
            for (int p = 0; p < n; p++) {
                for (uint32_t v : pinc[p]) inc.push_back(v);
                inc_off.push_back((int)inc.size());
            }
            for (int p = 0; p < n; p++) {
                const int li = o0 + p;
                const float* x = s.chain_positions + 3 * li;
                const float* xm = s.chain_prev_positions + 3 * li;
                const int t = s.chain_atom_types[li];
                if (t >= kMaxTypes) throw LimaError(LIMA_E_ARG, "atom type >= 32");
                float w;
                std::memcpy(&w, &t, 4);
                cpos.push_back(make_float4(x[0], x[1], x[2], w));
                cprev.push_back(make_float4(xm[0], xm[1], xm[2], 0.f));
                uint32_t m[4] = {0, 0, 0, 0};
                for (int e = s.ignore_offset[li]; e < s.ignore_offset[li + 1]; e++) {
                    const int oc = s.ignore_compound[e], ol = s.ignore_local[e];
                    if (oc < 0 || oc >= s.n_compounds) throw LimaError(LIMA_E_ARG, "ignore compound id out of range");
                    if (ol < 0 || ol >= kCompoundBlock) throw LimaError(LIMA_E_ARG, "ignore local id out of range");
                    if (oc == c) m[ol >> 5] |= 1u << (ol & 31);
                    else xent.push_back(make_int2(cb + oc, ol));
                }
                for (int k = 0; k < 4; k++) imask.push_back(m[k]);
                xoff.push_back((int)xent.size());
            }
            (void)gbase;
        }
        // bridges
        for (int b = 0; b < s.n_bridges; b++) {
            const int q0 = s.bridge_particle_offset[b], q1 = s.bridge_particle_offset[b + 1];
            if (q1 - q0 > 32 || q1 - q0 <= 0) throw LimaError(LIMA_E_CAPACITY, "bridge must have 1..32 particles");
            for (int k = q0; k < q1; k++) {
                const int cc = s.bridge_particle_compound[k], ll = s.bridge_particle_local[k];
                if (cc < 0 || cc >= s.n_compounds || ll < 0 || ll >= s.compound_offset[cc + 1] - s.compound_offset[cc])
                    throw LimaError(LIMA_E_ARG, "bridge particle reference out of range");
                br_glob.push_back(chb + s.compound_offset[cc] + ll);
            }
            br_off.push_back((int)br_glob.size());
            br_rep.push_back(r);
            const int np = q1 - q0;
            for (int t = s.bridge_bond_offset[b]; t < s.bridge_bond_offset[b + 1]; t++) {
                const lima_pair_bond& x = s.bridge_bonds[t];
                for (int k = 0; k < 2; k++) if ((int)x.atom_indexes[k] >= np) throw LimaError(LIMA_E_ARG, "bridge bond index out of range");
                brb.push_back(BondD{x.b0, x.kb, (int)x.atom_indexes[0], (int)x.atom_indexes[1]});
            }
            for (int t = s.bridge_angle_offset[b]; t < s.bridge_angle_offset[b + 1]; t++) {
                const lima_angle_bond& x = s.bridge_angles[t];
                for (int k = 0; k < 3; k++) if ((int)x.atom_indexes[k] >= np) throw LimaError(LIMA_E_ARG, "bridge angle index out of range");
                bra.push_back(AngleD{x.theta_0, x.k_theta, (int)x.atom_indexes[0], (int)x.atom_indexes[1], (int)x.atom_indexes[2], 0});
            }
            for (int t = s.bridge_dihedral_offset[b]; t < s.bridge_dihedral_offset[b + 1]; t++) {
                const lima_dihedral_bond& x = s.bridge_dihedrals[t];
                for (int k = 0; k < 4; k++) if ((int)x.atom_indexes[k] >= np) throw LimaError(LIMA_E_ARG, "bridge dihedral index out of range");
                brd.push_back(DihD{x.phi_0, x.k_phi, (int)x.n, (int)x.atom_indexes[0], (int)x.atom_indexes[1],
                                   (int)x.atom_indexes[2], (int)x.atom_indexes[3], 0});
            }
            brb_off.push_back((int)brb.size());
            bra_off.push_back((int)bra.size());
            brd_off.push_back((int)brd.size());
        }
        for (int k = 0; k < s.n_solvents; k++) {
            const float* x = s.solvent_positions + 3 * k;
            const float* xm = s.solvent_prev_positions + 3 * k;
            spos.push_back(solvent_pos(x[0], x[1], x[2], s.box_len));
            sprev.push_back(make_float4(xm[0], xm[1], xm[2], 0.f));
            solv_rep.push_back(r);
        }
        E->reps_h.push_back(ri);
    }
    // a chain particle may belong to at most one bridge (the bridge force is a store)
    {
        std::vector<char> seen(cpos.size(), 0);
        for (int g : br_glob) {
            if (seen[g]) throw LimaError(LIMA_E_ARG, "a particle belongs to more than one bridge");
            seen[g] = 1;
        }
    }
    E->R = nsys;
    E->NC = (int)comp_rep.size();
    E->NCH = (int)cpos.size();
    E->NS = (int)spos.size();
    E->NB = (int)br_rep.size();

    for (const float4& p : cpos) {
        int t;
        std::memcpy(&t, &p.w, 4);
        E->n_types = std::max(E->n_types, t + 1);
    }

    // ---- solvent tiles, cell grids (the solvent<-chain work list: build_scwork) ----
    E->comp_off_h = comp_off;
    {
        std::vector<int> row_src;
        E->comp_row_h.assign(1, 0);
        for (int c = 0; c < E->NC; c++) {
            for (int i = comp_off[c]; i < comp_off[c + 1]; i++) row_src.push_back(i);
            while (row_src.size() % kRowPad) row_src.push_back(-1);
            E->comp_row_h.push_back((int)row_src.size());
        }
        E->comp_row.upload(E->comp_row_h);
        E->row_src.upload(row_src);
    }
    std::vector<int4> stl;
    int cell_begin = 0;
    for (int r = 0; r < nsys; r++) {
        ReplicaInfo& ri = E->reps_h[r];
        ri.stile_begin = (int)stl.size();
        for (int t0 = ri.solv_begin; t0 < ri.solv_end; t0 += 256)
            stl.push_back(make_int4(r, t0, std::min(t0 + 256, ri.solv_end), (int)stl.size()));
        ri.stile_end = (int)stl.size();
        const float thr = P.cutoff + P.cutoff;   // Engine.cu:198, 264
        ri.ss_bound = sqrt_bound(thr);
        int ncell = (int)std::floor(ri.L / (thr * (1.0f + 1e-5f)));
        ncell = std::max(1, std::min(ncell, 256));
        ri.ncell = ncell;
        ri.cell_inv = (float)ncell / ri.L;
        ri.cell_begin = cell_begin;
        cell_begin += ncell * ncell * ncell;
        cell_rep_h.insert(cell_rep_h.end(), (size_t)ncell * ncell * ncell, r);
    }
    E->build_scwork();
    E->n_cells = std::max(cell_begin, 1);
    E->n_stiles = (int)stl.size();

    E->max_items = 0;
    E->listed_split_all = true;
    for (ReplicaInfo& ri : E->reps_h) {
        const size_t nc = ri.comp_end - ri.comp_begin, nsr = P.enable_solvents ? ri.solv_end - ri.solv_begin : 0;
        // the most items that lists of these capacities can hold
        auto items = [&](size_t neighbors, size_t solvents) -> size_t {
            return nc == 0 ? 0 : nc * (std::min(neighbors, nc - 1) + (std::min(solvents, nsr) + kSolventChunk - 1) / kSolventChunk);
        };
        int largest = 0;
        for (int c = ri.comp_begin; c < ri.comp_end; c++) largest = std::max(largest, E->comp_off_h[c + 1] - E->comp_off_h[c]);
        // The parts group FP32 sums, so whether a system has them follows from the system alone: its items
        // are counted at the default capacities, and other capacities change no bit of a trajectory.
        ri.listed_split = items(lima_engine::kListedNeighbors, lima_engine::kListedSolvents) <= lima_engine::kListedWideItems && largest > 32 ? 1 : 0;
        E->listed_split_all = E->listed_split_all && (nc == 0 || ri.listed_split);
        E->max_items += items(P.max_compound_neighbors, P.max_compound_solvents);
    }

    // ---- upload ----
    E->reps.upload(E->reps_h);
    for (int k = 0; k < 2; k++) E->cpos[k].upload(cpos);
    E->cprev.upload(cprev);
    E->cforce.alloc(std::max(E->NCH, 1)); E->cforce.zero();
    E->fbridge.alloc(std::max(E->NCH, 1)); E->fbridge.zero();
    E->intra_mask.upload(imask);
    E->xoff.upload(xoff);
    E->xent.upload(xent);
    E->comp_off.upload(comp_off);
    E->comp_rep.upload(comp_rep);
    E->comp_key.upload(comp_key);
    E->comp_sphere.upload(comp_sphere);
    E->bond_off.upload(bond_off); E->bonds.upload(bonds);
    E->angle_off.upload(angle_off); E->angles.upload(angles);
    E->dih_off.upload(dih_off); E->dihs.upload(dihs);
    E->inc_off.upload(inc_off); E->inc.upload(inc);
    E->br_off.upload(br_off); E->br_glob.upload(br_glob); E->br_rep.upload(br_rep);
    E->brb_off.upload(brb_off); E->brb.upload(brb);
    E->bra_off.upload(bra_off); E->bra.upload(bra);
    E->brd_off.upload(brd_off); E->brd.upload(brd);
    E->bonds_h = bonds; E->angles_h = angles; E->brb_h = brb; E->bra_h = bra;
    E->bond_off_h = bond_off; E->angle_off_h = angle_off; E->brb_off_h = brb_off; E->bra_off_h = bra_off;
    E->br_rep_h = br_rep;
    for (int k = 0; k < 2; k++) E->spos[k].upload(spos);
    E->sprev.upload(sprev);
    E->sforce.alloc(std::max(E->NS, 1)); E->sforce.zero();
    E->solv_rep.upload(solv_rep);
    E->stiles.upload(stl);
    E->mass.upload(mass);
    E->tab_sc.upload(tsc); E->tab_cs.upload(tcs); E->tab_inter.upload(tinter); E->tab_intra.upload(tintra); E->tab_ss.upload(tss);
    E->tab_inter_ab.alloc(tinter.size());
    E->tab_intra_ab.alloc(tintra.size());
    const size_t NCx = std::max(E->NC, 1), NSx = std::max(E->NS, 1), NCHx = std::max(E->NCH, 1);
    E->cc_cnt.alloc(NCx); E->cc_cnt.zero();
    E->cc_ids.alloc(NCx * P.max_compound_neighbors);
    E->cs_cnt.alloc(NCx); E->cs_cnt.zero();
    E->max_segs = 1;
    for (const ReplicaInfo& ri : E->reps_h)
        E->max_segs = std::max(E->max_segs, (ri.solv_end - ri.solv_begin + kSegSolvents - 1) / kSegSolvents);
    E->seg_cnt.alloc(NCx * E->max_segs); E->seg_cnt.zero();
    E->cs_ids.alloc(NCx * P.max_compound_solvents);
    E->ss_cnt.alloc(NSx); E->ss_cnt.zero();
    if ((NSx + 256) * (size_t)E->ss_ld() >= (size_t(1) << 32))
        throw LimaError(LIMA_E_ARG, "solvent lists exceed 2^32 entries (n_solvents x max_solvent_neighbors)");
    E->ss_ids.alloc(NSx * E->ss_ld());
    E->cw_off.alloc(NCx + 1); E->cw_off.zero();
    E->cw_total.alloc(1); E->cw_total.zero();
    E->max_slots = NCx * (size_t)(P.max_compound_neighbors + (P.max_compound_solvents + kSolventChunk - 1) / kSolventChunk);
    E->item_comp.alloc(std::max<size_t>(E->max_slots, 1)); E->item_comp.zero();
    E->run_off.alloc(NCx + 1); E->run_off.zero();
    E->run_cs_off.alloc(NCx + 1); E->run_cs_off.zero();
    E->run_total.alloc(2); E->run_total.zero();
    E->run_comp.alloc(std::max<size_t>(E->max_slots, 1)); E->run_comp.zero();
    if (P.accumulation == LIMA_ACCUM_FIXED64) {
        E->partC_fx.alloc(E->max_slots * kCompoundBlock);
        E->partC.alloc(1);
        E->cloc_fx.alloc(NCHx);
        E->cloc.alloc(1);
    } else {
        E->partC.alloc(E->max_slots * kCompoundBlock);
        E->partC_fx.alloc(1);
        E->cloc.alloc(NCHx);
        E->cloc_fx.alloc(1);
    }
    std::vector<float> ones(nsys, 1.0f);
    E->lambda.upload(ones);
    E->lambda_applied.upload(ones);
    E->ke_comp.alloc(NCx); E->ke_comp.zero();
    E->ke_stile.alloc(std::max(E->n_stiles, 1)); E->ke_stile.zero();
    E->temperature.alloc(nsys); E->temperature.zero();
    E->step_count.alloc(nsys); E->step_count.zero();
    {
        // the thermostat can run in a system's last integrator block where every system has one
        const bool solv = E->params.enable_solvents && E->NS > 0;
        std::vector<int> total(nsys);
        E->thermo_ok = true;
        for (int r = 0; r < nsys; r++) {
            const ReplicaInfo& ri = E->reps_h[r];
            total[r] = ri.comp_end - ri.comp_begin + (solv ? ri.stile_end - ri.stile_begin : 0);
            E->thermo_ok = E->thermo_ok && total[r] > 0;
        }
        E->thermo_total.upload(total);
        E->thermo_cnt.alloc(nsys); E->thermo_cnt.zero();
    }
    E->energy.alloc((size_t)nsys * kEnergyTerms); E->energy.zero();
    E->err.alloc(4); E->err.zero();
    E->cell_cnt.alloc(E->n_cells); E->cell_cnt.zero(); E->cell_start.alloc(E->n_cells + 1); E->cell_cursor.alloc(E->n_cells);
    E->cell_ids.alloc(NSx); E->solv_cell.alloc(NSx);
    E->cell_rep.upload(cell_rep_h);
    E->comp_cs_bound.upload(cs_bound);
    E->io_dev.alloc((size_t)6 * std::max(E->NCH + E->NS, 1));
    E->ss_part.alloc(NSx); E->ss_part.zero();
    E->ss_img.alloc(NSx); E->ss_img.zero();
}

// ---- reverse mode ------------------------------------------------------------
// Frames k = 0..K-1 start at the current state.  A forward pass stores a state
// checkpoint at the start of every segment (segments begin on list rebuilds,
// every `checkpoint_interval` frames or more) together with the compound lists
// the segment's first rebuild reads (its hysteresis input), and evaluates the
// loss.  The backward pass visits the segments last to first: it restores the
// checkpoint, rebuilds the segment's first lists from the stored compound lists
// (the same kernels on the same input give the same lists), recomputes the
// segment's frames keeping positions and force residuals (and a full copy of
// the lists before each rebuild inside the segment), then runs the adjoint
// recurrence over the segment's frames in reverse, restoring each period's lists.

size_t list_words(const lima_engine* E) {
    const lima_run_params& P = E->params;
    return (size_t)E->NC * (2 + P.max_compound_neighbors + P.max_compound_solvents) +
           (size_t)E->NS * (1 + E->ss_ld());
}

void d2d(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes) HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, st));
}

// full lists <-> one slot of words
void save_lists(lima_engine* E, int* dst) {
    const lima_run_params& P = E->params;
    const size_t nc = E->NC, ns = E->NS;
    hipStream_t st = E->stream;
    d2d(dst, E->cc_cnt.p, nc * 4, st); dst += nc;
    d2d(dst, E->cc_ids.p, nc * P.max_compound_neighbors * 4, st); dst += nc * P.max_compound_neighbors;
    d2d(dst, E->cs_cnt.p, nc * 4, st); dst += nc;
    d2d(dst, E->cs_ids.p, nc * P.max_compound_solvents * 4, st); dst += nc * P.max_compound_solvents;
    d2d(dst, E->ss_cnt.p, ns * 4, st); dst += ns;
    d2d(dst, E->ss_ids.p, ns * E->ss_ld() * 4, st);
}
void load_lists(lima_engine* E, const int* src) {
    const lima_run_params& P = E->params;
    const size_t nc = E->NC, ns = E->NS;
    hipStream_t st = E->stream;
    d2d(E->cc_cnt.p, src, nc * 4, st); src += nc;
    d2d(E->cc_ids.p, src, nc * P.max_compound_neighbors * 4, st); src += nc * P.max_compound_neighbors;
    d2d(E->cs_cnt.p, src, nc * 4, st); src += nc;
    d2d(E->cs_ids.p, src, nc * P.max_compound_solvents * 4, st); src += nc * P.max_compound_solvents;
    d2d(E->ss_cnt.p, src, ns * 4, st); src += ns;
    d2d(E->ss_ids.p, src, ns * E->ss_ld() * 4, st);
    E->launch_work_list(E->nlist_args(E->cur), st);   // listed work list of these lists
}
size_t cc_words(const lima_engine* E) { return (size_t)E->NC * (1 + E->params.max_compound_neighbors); }
void save_cc(lima_engine* E, int* dst) {
    d2d(dst, E->cc_cnt.p, (size_t)E->NC * 4, E->stream);
    d2d(dst + E->NC, E->cc_ids.p, (size_t)E->NC * E->params.max_compound_neighbors * 4, E->stream);
}
void load_cc(lima_engine* E, const int* src) {
    d2d(E->cc_cnt.p, src, (size_t)E->NC * 4, E->stream);
    d2d(E->cc_ids.p, src + E->NC, (size_t)E->NC * E->params.max_compound_neighbors * 4, E->stream);
}
// state (positions of the current parity and the previous positions) <-> a checkpoint
void save_state(lima_engine* E, float4* dst) {
    const size_t nch = E->NCH, ns = E->NS;
    d2d(dst, E->cpos[E->cur].p, nch * 16, E->stream);
    d2d(dst + nch, E->cprev.p, nch * 16, E->stream);
    d2d(dst + 2 * nch, E->spos[E->cur].p, ns * 16, E->stream);
    d2d(dst + 2 * nch + ns, E->sprev.p, ns * 16, E->stream);
}
void load_state(lima_engine* E, const float4* src) {
    const size_t nch = E->NCH, ns = E->NS;
    d2d(E->cpos[E->cur].p, src, nch * 16, E->stream);
    d2d(E->cprev.p, src + nch, nch * 16, E->stream);
    d2d(E->spos[E->cur].p, src + 2 * nch, ns * 16, E->stream);
    d2d(E->sprev.p, src + 2 * nch + ns, ns * 16, E->stream);
}

template <typename T> void ensure(DBuf<T>& b, size_t n) { b.grow(n); }

// per-particle constants of the adjoint (once per engine)
void adj_setup(lima_engine* E) {
    AdjBufs& B = E->adjb;
    if (B.ready) return;
    const int N = E->NCH + E->NS;
    std::vector<float> cfac(std::max(N, 1));
    std::vector<int> prep(std::max(N, 1));
    std::vector<float> mass_h((size_t)E->R * kMaxTypes);
    HIP_TRY(hipMemcpy(mass_h.data(), E->mass.p, mass_h.size() * 4, hipMemcpyDeviceToHost));
    std::vector<float4> cpos_h(std::max(E->NCH, 1));
    if (E->NCH) HIP_TRY(hipMemcpy(cpos_h.data(), E->cpos[E->cur].p, (size_t)E->NCH * 16, hipMemcpyDeviceToHost));
    int maxc = 1, maxs = 1, maxn = 1;
    std::vector<int> comp_of(std::max(E->NCH, 1));
    for (int c = 0; c < E->NC; c++)
        for (int i = E->comp_off_h[c]; i < E->comp_off_h[c + 1]; i++) comp_of[i] = c;
    std::vector<int> mask_off(std::max(E->NC, 1), 0);
    int words = 0;
    for (int r = 0; r < E->R; r++) {
        const ReplicaInfo& ri = E->reps_h[r];
        const double dt = ri.dt;
        for (int i = ri.chain_begin; i < ri.chain_end; i++) {
            int t;
            std::memcpy(&t, &cpos_h[i].w, 4);
            cfac[i] = (float)(dt / (double)mass_h[r * kMaxTypes + t] * dt);
            prep[i] = r;
        }
        for (int s = ri.solv_begin; s < ri.solv_end; s++) {
            cfac[E->NCH + s] = (float)(dt / (double)mass_h[r * kMaxTypes] * dt);
            prep[E->NCH + s] = r;
        }
        maxc = std::max(maxc, ri.comp_end - ri.comp_begin);
        maxs = std::max(maxs, ri.solv_end - ri.solv_begin);
        const int wr = (ri.solv_end - ri.solv_begin + 31) / 32;
        for (int c = ri.comp_begin; c < ri.comp_end; c++) {
            mask_off[c] = words;
            words += wr;
        }
    }
    // The solvent-side role: solvent tiles x chunks of compounds of at most kAdjRows particles, or
    // (where that leaves under about 1,024 blocks, four a CU) parts of a compound down to 32
    // particles.  The chain-side role: compounds x slices of solvents, to as many blocks, of 64 or
    // more.
    maxn = std::max(E->max_cn, 1);
    const int want = 1024, tiles = std::max(E->n_stiles, 1), comps = std::max(E->NC, 1);
    B.comp_chunk = std::max(1, std::min(kAdjRows / maxn, (int)((long long)tiles * maxc / want)));
    const int chunks = (maxc + B.comp_chunk - 1) / B.comp_chunk;
    B.comp_split = B.comp_chunk > 1 ? 1 : std::max(1, std::min((maxn + 31) / 32, want / (tiles * chunks)));
    B.n_cchunks = chunks * B.comp_split;
    const int nsl = std::max(1, want / comps);
    B.solv_slice = std::max(64, ((maxs + nsl - 1) / nsl + 63) / 64 * 64);
    B.n_sslices = (maxs + B.solv_slice - 1) / B.solv_slice;
    B.gpart.alloc(std::max<size_t>(E->max_slots, 1) * kCompoundBlock);
    B.cfac.upload(cfac);
    B.prep.upload(prep);
    B.mask_off.upload(mask_off);
    B.comp_of.upload(comp_of);
    B.mask.alloc(std::max(words, 1));
    B.adj.alloc((size_t)3 * std::max(N, 1));
    B.w.alloc(std::max(N, 1));
    B.gxc.alloc((size_t)(kAdjChainSlots + B.n_sslices) * std::max(E->NCH, 1));
    HIP_TRY(hipMemsetAsync(B.gxc.p, 0, B.gxc.n * sizeof(float4), E->stream));   // the bridges' slot outside any bridge
    B.gxs.alloc((size_t)(B.n_cchunks + 1) * std::max(E->NS, 1));
    B.beta.alloc(E->R);
    B.loss.alloc(E->R);
    B.lacc.alloc(std::max(N, 1));
    B.gpar.alloc((size_t)E->R * kAdjStride);
    B.ready = true;
}

void adj_build_mask(lima_engine* E) {
    AdjBufs& B = E->adjb;
    if (E->NC == 0 || E->NS == 0) return;
    adj_mask_zero_kernel<<<(int)((B.mask.n + 255) / 256), 256, 0, E->stream>>>(B.mask.p, (int)B.mask.n);
    adj_mask_set_kernel<<<E->NC, 256, 0, E->stream>>>(E->step_args(E->cur), B.mask.p, B.mask_off.p);
}

// the residuals 2 beta (F - F*) of the frame just stepped into Rs (and the loss and the frame's
// energies when given); targets are the frame's rows of the uploaded chain / solvent target arrays, or none
void adj_residuals(lima_engine* E, float4* rs, const float* tc, const float* ts, bool with_loss, bool solv, double* energies) {
    AdjBufs& B = E->adjb;
    const int n_energy = energies ? E->R * kEnergyTerms : 0, n = std::max(E->NCH + E->NS, n_energy);
    if (n > 0)
        adj_residual_kernel<<<(n + 255) / 256, 256, 0, E->stream>>>(E->cforce.p, solv ? E->sforce.p : nullptr, tc, ts, B.prep.p,
                                                                   B.beta.p, rs, with_loss ? B.lacc.p : nullptr, E->energy.p,
                                                                   energies, E->NCH, E->NS, n_energy);
}

// all K frames of the targets, once per call, as given (x, y, z per particle)
void adj_upload_targets(lima_engine* E, const lima_adjoint_spec& sp) {
    AdjBufs& B = E->adjb;
    const size_t K = sp.n_frames;
    if (sp.chain_force_target && E->NCH) {
        ensure(B.Tc, K * E->NCH * 3);
        HIP_TRY(hipMemcpy(B.Tc.p, sp.chain_force_target, K * E->NCH * 3 * sizeof(float), hipMemcpyHostToDevice));
    }
    if (sp.solvent_force_target && E->NS) {
        ensure(B.Ts, K * E->NS * 3);
        HIP_TRY(hipMemcpy(B.Ts.p, sp.solvent_force_target, K * E->NS * 3 * sizeof(float), hipMemcpyHostToDevice));
    }
}

// one step of the trajectory (the engine's step, optionally with FP64 energies), its positions kept in X if given
void adj_step(lima_engine* E, bool energy, float4* X = nullptr) {
    const int n_energy = energy ? (int)E->energy.n : 0, n = std::max(X ? E->NCH + E->NS : 0, n_energy);
    if (n > 0)
        adj_begin_kernel<<<(n + 255) / 256, 256, 0, E->stream>>>(E->cpos[E->cur].p, E->spos[E->cur].p, X, E->energy.p, E->NCH, E->NS,
                                                                 n_energy);
    E->launch_step(E->cur, energy);
    E->cur ^= 1;
    E->step++;
    E->since_rebuild++;
}

// one frame of the adjoint recurrence: positions X and energy weights gE, the weights w of the
// frame already formed; with rs_prev (the residual of the frame before) forms that one's
void adj_frame(lima_engine* E, int j, const float4* X, const float4* rs_prev, const float* gE, bool solv) {
    AdjBufs& B = E->adjb;
    const int nch = E->NCH, ns = E->NS, N = nch + ns;
    double4* a_out = B.adj.p + (size_t)(j % 3) * N;
    const double4* a1 = B.adj.p + (size_t)((j + 1) % 3) * N;
    const double4* a2 = B.adj.p + (size_t)((j + 2) % 3) * N;
    AdjArgs A{};
    A.s = E->step_args(E->cur);
    A.s.cpos = X;
    A.s.spos = X + nch;
    A.wc = B.w.p;
    A.ws = B.w.p + nch;
    A.gE = gE;
    A.gxc = B.gxc.p;
    A.gxs = B.gxs.p;
    A.gpar = B.gpar.p;
    A.cs_mask = B.mask.p;
    A.mask_off = B.mask_off.p;
    A.comp_of = B.comp_of.p;
    A.n_chain = nch;
    A.gpart = B.gpart.p;
    A.comp_chunk = B.comp_chunk;
    A.comp_split = B.comp_split;
    A.n_cchunks = B.n_cchunks;
    A.solv_slice = B.solv_slice;
    A.n_sslices = B.n_sslices;
    A.nb = E->max_cb;
    A.na = E->max_ca;
    const bool sv = solv && ns > 0;
    AdjBlocks f{};
    if (nch > 0) {
        f.bonded = f.intra = E->NC;
        f.bridges = (E->NB + 3) / 4;
        f.listed = (int)std::min<size_t>(4096, E->max_items);
        if (sv) f.chain = E->NC * B.n_sslices;
    }
    if (sv) {
        f.pairs = E->n_stiles * (256 * kAdjPairLanes / kAdjThreads);
        f.solvent = E->n_stiles * B.n_cchunks;
    }
    const size_t lds = kAdjHead + std::max({6 * kAdjThreads * sizeof(double), kAdjRows * (2 * sizeof(float4) + sizeof(float2)),
                                            sizeof(AdjPairStage), 4 * sizeof(AdjBridgeStage),
                                            adj_bonded_lds(E->max_cb, E->max_ca, E->max_cd)});
    const int blocks = f.bonded + f.bridges + f.intra + f.listed + f.chain + f.pairs + f.solvent;
    const dim3 grid = grid_of(blocks);
    f.width = (int)grid.x;
    if (blocks > 0) adj_frame_kernel<<<grid, kAdjThreads, lds, E->stream>>>(A, f);
    adj_update_kernel<<<(N + 255) / 256, 256, 0, E->stream>>>(A, kAdjChainSlots + (sv ? B.n_sslices : 0), sv ? B.n_cchunks + 1 : 0,
                                                              a1, a2, a_out, rs_prev, B.cfac.p, B.w.p);
}

struct SavedRun {
    int cur;
    long long step, since, nreb;
};

int adjoint_run(lima_engine* E, const lima_adjoint_spec& sp, double* loss_out, double* grad_out) {
    const lima_run_params& P = E->params;
    if (P.thermostat != LIMA_THERMOSTAT_NONE)
        throw LimaError(LIMA_E_UNSUPPORTED, "the adjoint differentiates the plain Verlet step: use LIMA_THERMOSTAT_NONE");
    const int K = sp.n_frames;
    if (K < 1) throw LimaError(LIMA_E_ARG, "n_frames must be >= 1");
    if (!loss_out) throw LimaError(LIMA_E_ARG, "null loss output");
    const int R = E->R, NCH = E->NCH, NS = E->NS, N = NCH + NS, NC = E->NC;
    const bool solv = P.enable_solvents && NS > 0;
    const int iv = P.nlist_interval;
    if (sp.checkpoint_interval < 0) throw LimaError(LIMA_E_ARG, "checkpoint_interval must be >= 0");
    HIP_TRY(hipSetDevice(E->device));
    HIP_TRY(hipStreamSynchronize(E->stream));
    adj_setup(E);
    AdjBufs& B = E->adjb;
    const long long since0 = E->since_rebuild;
    auto rebuild_after = [&](int j) { return iv > 0 && (since0 + j + 1) % iv == 0; };
    const size_t LW = std::max<size_t>(list_words(E), 1), CW = std::max<size_t>(cc_words(E), 1);
    // checkpoint_interval 0: one segment (nothing recomputed) when its frames, residuals and lists
    // take at most half of the free device memory, else segments of 20 frames
    int cpi = sp.checkpoint_interval;
    if (cpi == 0) {
        int rebuilds = 0;
        for (int j = 0; j + 1 < K; j++) rebuilds += rebuild_after(j) ? 1 : 0;
        const size_t need = (size_t)K * std::max(N, 1) * 2 * sizeof(float4) + (size_t)(1 + rebuilds) * LW * sizeof(int);
        const size_t held = B.X.n * sizeof(float4) + B.Rs.n * sizeof(float4) + B.lists.n * sizeof(int);
        size_t free_b = 0, total_b = 0;
        HIP_TRY(hipMemGetInfo(&free_b, &total_b));
        cpi = need <= held + free_b / 2 ? K : 20;
    }

    // the symmetric-pair terms need symmetric compound lists (the engine builds them so)
    if (NC > 0) {
        std::vector<int> cnt(NC), ids((size_t)NC * P.max_compound_neighbors);
        HIP_TRY(hipMemcpy(cnt.data(), E->cc_cnt.p, NC * 4, hipMemcpyDeviceToHost));
        HIP_TRY(hipMemcpy(ids.data(), E->cc_ids.p, ids.size() * 4, hipMemcpyDeviceToHost));
        std::vector<std::vector<int>> sets(NC);
        for (int c = 0; c < NC; c++) sets[c].assign(&ids[(size_t)c * P.max_compound_neighbors], &ids[(size_t)c * P.max_compound_neighbors] + cnt[c]);
        for (int c = 0; c < NC; c++)
            for (int nb : sets[c])
                if (nb < 0 || nb >= NC || std::find(sets[nb].begin(), sets[nb].end(), c) == sets[nb].end())
                    throw LimaError(LIMA_E_ARG, "the adjoint needs symmetric compound neighbour lists");
    }

    const SavedRun saved{E->cur, E->step, E->since_rebuild, E->n_rebuilds};
    // segment starts
    std::vector<int> starts{0};
    for (int j = 0; j + 1 < K; j++) {
        const bool boundary = iv > 0 ? rebuild_after(j) : true;
        if (boundary && j + 1 - starts.back() >= cpi) starts.push_back(j + 1);
    }
    const int nseg = (int)starts.size();
    int max_len = 0, max_inner = 0;
    for (int s = 0; s < nseg; s++) {
        const int k0 = starts[s], k1 = s + 1 < nseg ? starts[s + 1] : K;
        max_len = std::max(max_len, k1 - k0);
        int inner = 0;
        for (int j = k0; j + 1 < k1; j++) inner += rebuild_after(j) ? 1 : 0;
        max_inner = std::max(max_inner, inner);
    }
    ensure(B.ck, (size_t)nseg * 2 * std::max(N, 1));
    ensure(B.ck_cc, (size_t)nseg * CW);
    ensure(B.lists, (size_t)(1 + max_inner) * LW);
    ensure(B.X, (size_t)max_len * std::max(N, 1));
    ensure(B.Rs, (size_t)max_len * std::max(N, 1));
    ensure(B.efr, (size_t)K * R * kEnergyTerms);
    ensure(B.gE, (size_t)K * R);

    std::vector<double> beta(R, 0.0), alpha(R, 0.0);
    for (int r = 0; r < R; r++) {
        if (sp.force_weight) beta[r] = sp.force_weight[r];
        if (sp.energy_weight) alpha[r] = sp.energy_weight[r];
    }
    HIP_TRY(hipMemcpy(B.beta.p, beta.data(), R * 8, hipMemcpyHostToDevice));
    HIP_TRY(hipMemsetAsync(B.lacc.p, 0, (size_t)N * 8, E->stream));
    adj_upload_targets(E, sp);
    auto tgt_c = [&](int j) -> const float* {
        return sp.chain_force_target && NCH ? B.Tc.p + (size_t)j * NCH * 3 : nullptr;
    };
    auto tgt_s = [&](int j) -> const float* {
        return sp.solvent_force_target && NS ? B.Ts.p + (size_t)j * NS * 3 : nullptr;
    };

    // ---- forward pass: checkpoints, energies, force loss ----
    // The last segment is the first one reversed: when a gradient is wanted, its frames,
    // residuals and interior lists are kept here instead of being recomputed.
    std::vector<int> kept_period_end;
    save_lists(E, B.lists.p);
    for (int s = 0; s < nseg; s++) {
        const int k0 = starts[s], k1 = s + 1 < nseg ? starts[s + 1] : K;
        const bool keep = grad_out && s == nseg - 1;
        save_state(E, B.ck.p + (size_t)s * 2 * N);
        for (int j = k0; j < k1; j++) {
            adj_step(E, true, keep ? B.X.p + (size_t)(j - k0) * N : nullptr);
            adj_residuals(E, keep ? B.Rs.p + (size_t)(j - k0) * N : B.Rs.p, tgt_c(j), tgt_s(j), true, solv,
                          B.efr.p + (size_t)j * R * kEnergyTerms);
            if (j + 1 < K && rebuild_after(j)) {
                if (s + 1 < nseg && starts[s + 1] == j + 1) save_cc(E, B.ck_cc.p + (size_t)(s + 1) * CW);
                if (keep) {
                    save_lists(E, B.lists.p + (size_t)(1 + kept_period_end.size()) * LW);
                    kept_period_end.push_back(j);
                }
                E->launch_rebuild(E->cur);
                E->since_rebuild = 0;
            }
        }
    }
    adj_loss_reduce_kernel<<<R, 256, 0, E->stream>>>(E->reps.p, B.lacc.p, NCH, B.loss.p);
    HIP_TRY(hipStreamSynchronize(E->stream));
    int st = E->check_errors();
    std::vector<double> efr((size_t)K * R * kEnergyTerms), floss(R);
    HIP_TRY(hipMemcpy(efr.data(), B.efr.p, efr.size() * 8, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(floss.data(), B.loss.p, R * 8, hipMemcpyDeviceToHost));
    std::vector<float> gE((size_t)K * R);
    for (int r = 0; r < R; r++) loss_out[r] = floss[r];
    for (int k = 0; k < K; k++)
        for (int r = 0; r < R; r++) {
            const double* v = &efr[((size_t)k * R + r) * kEnergyTerms];
            const double pot = v[kE_bond] + v[kE_angle] + v[kE_dih] +
                               0.5 * (v[kE_intra] + v[kE_inter] + v[kE_cs] + v[kE_sc] + v[kE_ss]);
            const double tgt = sp.energy_target ? sp.energy_target[(size_t)k * R + r] : 0.0;
            loss_out[r] += alpha[r] * (pot - tgt) * (pot - tgt);
            gE[(size_t)k * R + r] = (float)(2.0 * alpha[r] * (pot - tgt));
        }

    // ---- backward pass ----
    if (st == LIMA_OK && grad_out) {
        HIP_TRY(hipMemcpy(B.gE.p, gE.data(), gE.size() * 4, hipMemcpyHostToDevice));
        HIP_TRY(hipMemsetAsync(B.adj.p, 0, (size_t)3 * N * sizeof(double4), E->stream));
        HIP_TRY(hipMemsetAsync(B.gpar.p, 0, (size_t)R * kAdjStride * 8, E->stream));
        for (int s = nseg - 1; s >= 0; s--) {
            const int k0 = starts[s], k1 = s + 1 < nseg ? starts[s + 1] : K;
            std::vector<int> period_end;
            if (s == nseg - 1) {
                // kept by the forward pass; the device holds the segment's last lists
                period_end = kept_period_end;
            } else {
                load_state(E, B.ck.p + (size_t)s * 2 * N);
                if (k0 == 0 || iv <= 0) {
                    load_lists(E, B.lists.p);
                    E->since_rebuild = iv > 0 ? (since0 + k0) % iv : 0;
                } else {
                    load_cc(E, B.ck_cc.p + (size_t)s * CW);
                    E->launch_rebuild(E->cur);
                    E->since_rebuild = 0;
                }
            }
            // recompute the segment
            for (int j = k0; j < k1 && s != nseg - 1; j++) {
                adj_step(E, false, B.X.p + (size_t)(j - k0) * N);
                adj_residuals(E, B.Rs.p + (size_t)(j - k0) * N, tgt_c(j), tgt_s(j), false, solv, nullptr);
                if (j + 1 < k1 && rebuild_after(j)) {
                    save_lists(E, B.lists.p + (size_t)(1 + period_end.size()) * LW);
                    period_end.push_back(j);
                    E->launch_rebuild(E->cur);
                    E->since_rebuild = 0;
                }
            }
            // reverse over the segment's frames
            int q = (int)period_end.size();
            bool mask_dirty = true;
            adj_weight_kernel<<<(N + 255) / 256, 256, 0, E->stream>>>(B.Rs.p + (size_t)(k1 - 1 - k0) * N,
                                                                      B.adj.p + (size_t)(k1 % 3) * N, B.cfac.p, B.w.p, N);
            for (int j = k1 - 1; j >= k0; j--) {
                if (q > 0 && j == period_end[q - 1]) {
                    load_lists(E, B.lists.p + (size_t)q * LW);
                    q--;
                    mask_dirty = true;
                }
                if (mask_dirty) {
                    adj_build_mask(E);
                    mask_dirty = false;
                }
                adj_frame(E, j, B.X.p + (size_t)(j - k0) * N, j > k0 ? B.Rs.p + (size_t)(j - 1 - k0) * N : nullptr,
                          B.gE.p + (size_t)j * R, solv);
            }
        }
        HIP_TRY(hipStreamSynchronize(E->stream));
        st = E->check_errors();
        std::vector<double> gp((size_t)R * kAdjStride);
        HIP_TRY(hipMemcpy(gp.data(), B.gpar.p, gp.size() * 8, hipMemcpyDeviceToHost));
        for (int r = 0; r < R; r++) {
            const double* g = &gp[(size_t)r * kAdjStride];
            double* o = grad_out + (size_t)r * LIMA_N_PARAMETERS;
            const lima_particle_params* pp = E->ff_h[r].particle_parameters;
            for (int t = 0; t < kMaxTypes; t++) {
                o[t] = g[t];
                const double eps = pp[t].epsilon;
                o[kMaxTypes + t] = 12.0 * g[kMaxTypes + t] + (eps > 0 ? g[2 * kMaxTypes + t] / (2.0 * eps) : 0.0);
            }
            for (int k = 0; k < 4; k++) o[2 * kMaxTypes + k] = g[kAdjTypeBins + k];
        }
    }

    // ---- leave the engine as it was ----
    E->cur = saved.cur;
    load_state(E, B.ck.p);
    load_lists(E, B.lists.p);
    HIP_TRY(hipStreamSynchronize(E->stream));
    E->step = saved.step;
    E->since_rebuild = saved.since;
    E->n_rebuilds = saved.nreb;
    return st;
}

// forces and potential energies of frames 0..K-1 from the current state
int record_frames(lima_engine* E, int K, float* cf, float* sf, double* pot) {
    if (K < 1) throw LimaError(LIMA_E_ARG, "n_frames must be >= 1");
    const int R = E->R, NCH = E->NCH, NS = E->NS, N = NCH + NS;
    const int iv = E->params.nlist_interval;
    HIP_TRY(hipSetDevice(E->device));
    HIP_TRY(hipStreamSynchronize(E->stream));
    AdjBufs& B = E->adjb;
    ensure(B.ck, (size_t)2 * std::max(N, 1));
    ensure(B.lists, std::max<size_t>(list_words(E), 1));
    const SavedRun saved{E->cur, E->step, E->since_rebuild, E->n_rebuilds};
    save_state(E, B.ck.p);
    save_lists(E, B.lists.p);
    // the thermostat scalars are part of the state handed back
    std::vector<float> lam(R), lam_applied(R);
    HIP_TRY(hipMemcpy(lam.data(), E->lambda.p, R * sizeof(float), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(lam_applied.data(), E->lambda_applied.p, R * sizeof(float), hipMemcpyDeviceToHost));
    E->sync_step_count();
    std::vector<float4> hc(std::max(NCH, 1)), hs(std::max(NS, 1));
    std::vector<double> e((size_t)R * kEnergyTerms);
    int st = LIMA_OK;
    for (int j = 0; j < K && st == LIMA_OK; j++) {
        adj_step(E, true);
        HIP_TRY(hipStreamSynchronize(E->stream));
        st = E->check_errors();
        if (cf && NCH) {
            HIP_TRY(hipMemcpy(hc.data(), E->cforce.p, (size_t)NCH * 16, hipMemcpyDeviceToHost));
            for (int i = 0; i < NCH; i++) {
                float* o = cf + ((size_t)j * NCH + i) * 3;
                o[0] = hc[i].x; o[1] = hc[i].y; o[2] = hc[i].z;
            }
        }
        if (sf && NS) {
            const bool solv = E->params.enable_solvents;
            if (solv) HIP_TRY(hipMemcpy(hs.data(), E->sforce.p, (size_t)NS * 16, hipMemcpyDeviceToHost));
            for (int i = 0; i < NS; i++) {
                float* o = sf + ((size_t)j * NS + i) * 3;
                o[0] = solv ? hs[i].x : 0.f; o[1] = solv ? hs[i].y : 0.f; o[2] = solv ? hs[i].z : 0.f;
            }
        }
        if (pot) {
            HIP_TRY(hipMemcpy(e.data(), E->energy.p, e.size() * 8, hipMemcpyDeviceToHost));
            for (int r = 0; r < R; r++) {
                const double* v = &e[(size_t)r * kEnergyTerms];
                pot[(size_t)j * R + r] = v[kE_bond] + v[kE_angle] + v[kE_dih] +
                                         0.5 * (v[kE_intra] + v[kE_inter] + v[kE_cs] + v[kE_sc] + v[kE_ss]);
            }
        }
        if (iv > 0 && E->since_rebuild >= iv) {
            E->launch_rebuild(E->cur);
            E->since_rebuild = 0;
        }
    }
    E->cur = saved.cur;
    load_state(E, B.ck.p);
    load_lists(E, B.lists.p);
    HIP_TRY(hipStreamSynchronize(E->stream));
    HIP_TRY(hipMemcpy(E->lambda.p, lam.data(), R * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(E->lambda_applied.p, lam_applied.data(), R * sizeof(float), hipMemcpyHostToDevice));
    E->step = saved.step;
    E->since_rebuild = saved.since;
    E->n_rebuilds = saved.nreb;
    return st;
}

// parameter vector of one system <-> force field and shared bonded constants
void get_parameters(lima_engine* E, int r, double* o) {
    const lima_particle_params* pp = E->ff_h[r].particle_parameters;
    for (int t = 0; t < kMaxTypes; t++) {
        o[t] = pp[t].sigma;
        o[kMaxTypes + t] = pp[t].epsilon;
    }
    const ReplicaInfo& ri = E->reps_h[r];
    const int b0 = E->bond_off_h[ri.comp_begin], b1 = E->bond_off_h[ri.comp_end];
    const int a0 = E->angle_off_h[ri.comp_begin], a1 = E->angle_off_h[ri.comp_end];
    o[64] = o[65] = o[66] = o[67] = 0.0;
    const BondD* bd = b1 > b0 ? &E->bonds_h[b0] : nullptr;
    const AngleD* ad = a1 > a0 ? &E->angles_h[a0] : nullptr;
    for (int b = 0; b < E->NB && (!bd || !ad); b++) {
        if (E->br_rep_h[b] != r) continue;
        if (!bd && E->brb_off_h[b + 1] > E->brb_off_h[b]) bd = &E->brb_h[E->brb_off_h[b]];
        if (!ad && E->bra_off_h[b + 1] > E->bra_off_h[b]) ad = &E->bra_h[E->bra_off_h[b]];
    }
    if (bd) { o[64] = bd->kb; o[65] = bd->b0; }
    if (ad) { o[66] = ad->k; o[67] = ad->t0; }
}

// Calls f(kb, b0) for every pair bond of system r (kind 0), or f(k_theta, theta_0) for every
// angle (kind 1), compound terms first, then the bridges' in bridge order.
template <typename F> void for_each_bonded(lima_engine* E, int r, int kind, F&& f) {
    const ReplicaInfo& ri = E->reps_h[r];
    if (kind == 0) {
        for (int b = E->bond_off_h[ri.comp_begin]; b < E->bond_off_h[ri.comp_end]; b++) f(E->bonds_h[b].kb, E->bonds_h[b].b0);
    } else {
        for (int a = E->angle_off_h[ri.comp_begin]; a < E->angle_off_h[ri.comp_end]; a++) f(E->angles_h[a].k, E->angles_h[a].t0);
    }
    for (int b = 0; b < E->NB; b++) {
        if (E->br_rep_h[b] != r) continue;
        if (kind == 0) {
            for (int t = E->brb_off_h[b]; t < E->brb_off_h[b + 1]; t++) f(E->brb_h[t].kb, E->brb_h[t].b0);
        } else {
            for (int t = E->bra_off_h[b]; t < E->bra_off_h[b + 1]; t++) f(E->bra_h[t].k, E->bra_h[t].t0);
        }
    }
}

void set_parameters(lima_engine* E, int r, const double* v) {
    for (int i = 0; i < LIMA_N_PARAMETERS; i++)
        if (!std::isfinite(v[i])) throw LimaError(LIMA_E_ARG, "parameters must be finite");
    // a type slot the force field leaves empty (sigma 0) may be passed back as it is; a new value
    // must be a valid one
    const lima_particle_params* pp_cur = E->ff_h[r].particle_parameters;
    for (int t = 0; t < kMaxTypes; t++) {
        const bool same = (float)v[t] == pp_cur[t].sigma && (float)v[kMaxTypes + t] == pp_cur[t].epsilon;
        if (!same && (v[t] <= 0 || v[kMaxTypes + t] < 0)) throw LimaError(LIMA_E_ARG, "sigma must be > 0 and epsilon >= 0");
    }
    // Entries 64-67 are one constant pair per kind shared by every term.  A system whose terms
    // carry their own constants (an ingested molecule) keeps them when the entries are passed
    // back unchanged, and refuses a change, which would replace the whole bonded force field.
    double cur[LIMA_N_PARAMETERS];
    get_parameters(E, r, cur);
    bool write_kind[2] = {false, false};
    for (int kind = 0; kind < 2; kind++) {
        const float k_new = (float)v[64 + 2 * kind], x_new = (float)v[65 + 2 * kind];
        if (k_new == (float)cur[64 + 2 * kind] && x_new == (float)cur[65 + 2 * kind]) continue;
        bool uniform = true;
        const float k0 = (float)cur[64 + 2 * kind], x0 = (float)cur[65 + 2 * kind];
        for_each_bonded(E, r, kind, [&](float& k, float& x) { uniform = uniform && k == k0 && x == x0; });
        if (!uniform)
            throw LimaError(LIMA_E_UNSUPPORTED, kind == 0 ? "the system's pair bonds differ per term: kb, b0 (entries 64, 65) cannot be set"
                                                          : "the system's angles differ per term: k_theta, theta_0 (entries 66, 67) cannot be set");
        write_kind[kind] = true;
    }
    HIP_TRY(hipSetDevice(E->device));
    SystemParams sp{};
    lima_particle_params* pp = E->ff_h[r].particle_parameters;
    for (int t = 0; t < kMaxTypes; t++) {
        sp.sigma[t] = pp[t].sigma = (float)v[t];
        sp.eps[t] = pp[t].epsilon = (float)v[kMaxTypes + t];
    }
    for (int kind = 0; kind < 2; kind++) {
        sp.write[kind] = write_kind[kind] ? 1 : 0;
        const float k_new = sp.bonded[kind][0] = (float)v[64 + 2 * kind], x_new = sp.bonded[kind][1] = (float)v[65 + 2 * kind];
        if (write_kind[kind]) for_each_bonded(E, r, kind, [&](float& k, float& x) { k = k_new; x = x_new; });
    }
    const ReplicaInfo& ri = E->reps_h[r];
    sp.bond0 = E->bond_off_h[ri.comp_begin]; sp.bond1 = E->bond_off_h[ri.comp_end];
    sp.angle0 = E->angle_off_h[ri.comp_begin]; sp.angle1 = E->angle_off_h[ri.comp_end];
    // a system's bridges are consecutive
    const auto br = std::equal_range(E->br_rep_h.begin(), E->br_rep_h.end(), r);
    if (br.first != br.second) {
        const int q0 = (int)(br.first - E->br_rep_h.begin()), q1 = (int)(br.second - E->br_rep_h.begin());
        sp.brb0 = E->brb_off_h[q0]; sp.brb1 = E->brb_off_h[q1];
        sp.bra0 = E->bra_off_h[q0]; sp.bra1 = E->bra_off_h[q1];
    }
    set_parameters_kernel<<<1, kMaxTypes * kMaxTypes, 0, E->stream>>>(sp, r, E->tab_sc.p, E->tab_cs.p, E->tab_ss.p, E->tab_inter.p,
                                                                      E->tab_intra.p, E->tab_inter_ab.p, E->tab_intra_ab.p, E->bonds.p,
                                                                      E->angles.p, E->brb.p, E->bra.p);
}

thread_local std::string g_last_error;

int fail(lima_engine* E, const LimaError& e) {
    if (E) E->last_error = e.msg;
    g_last_error = e.msg;
    return e.code;
}

template <typename F> int guarded(lima_engine* E, F&& f) {
    if (!E) return LIMA_E_ARG;
    try {
        return f();
    } catch (const LimaError& e) {
        return fail(E, e);
    }
}

// ---- autotune cache, keyed by the histogram of replica shapes ----
std::mutex g_tune_mu;
std::map<std::string, LaunchConfig> g_tune_cache;
bool g_tune_loaded = false;

std::string shape_key(const lima_engine* E) {
    std::map<std::pair<int, int>, int> hist;   // (chain particles / 128, solvents / 512) -> replicas
    for (const ReplicaInfo& ri : E->reps_h)
        hist[{(ri.chain_end - ri.chain_begin + 64) / 128, (ri.solv_end - ri.solv_begin + 256) / 512}]++;
    std::ostringstream os;
    os << "acc" << E->params.accumulation << "_sol" << E->params.enable_solvents;
    for (const auto& kv : hist) os << "_" << kv.first.first << "x" << kv.first.second << ":" << kv.second;
    return os.str();
}

std::string g_tune_path;

// reads the cache file once per path (a process may point LIMA_AUTOTUNE_CACHE elsewhere later)
void load_tune_file() {
    const char* path = std::getenv("LIMA_AUTOTUNE_CACHE");
    const std::string p = path ? path : "";
    if (g_tune_loaded && p == g_tune_path) return;
    g_tune_loaded = true;
    g_tune_path = p;
    if (!path) return;
    std::ifstream f(path);
    std::string line;
    while (std::getline(f, line)) {
        // key spt chunk_particles listed_grid [listed_lanes [listed_packed [fused_thermostat]]]
        std::istringstream is(line);
        std::string key;
        LaunchConfig c;
        if (!(is >> key >> c.spt >> c.chunk_particles >> c.listed_grid)) continue;
        if (!(is >> c.listed_lanes)) c.listed_lanes = 1;
        if (!(is >> c.listed_packed)) c.listed_packed = 1;
        if (!(is >> c.fused_thermostat)) c.fused_thermostat = 0;
        // only shapes the autotuner itself can pick: any other line is skipped
        const bool ok = (c.spt == 1 || c.spt == 2 || c.spt == 4) &&
                        (c.chunk_particles == 256 || c.chunk_particles == 512 || c.chunk_particles == 1024 ||
                         c.chunk_particles == 2048) && c.chunk_particles <= kChunkParticles &&
                        (c.listed_grid == 1024 || c.listed_grid == 2048 || c.listed_grid == 4096 || c.listed_grid == 8192) &&
                        (c.listed_lanes == 1 || c.listed_lanes == 4) && (c.listed_packed == 0 || c.listed_packed == 1 || c.listed_packed == 2) &&
                        (c.fused_thermostat >= 0 && c.fused_thermostat <= 2);
        if (!ok) continue;
        c.spt = 1;   // 2 and 4 solvents a lane, which files may name, were slower and are no longer a choice
        g_tune_cache[key] = c;
    }
}

void save_tune_entry(const std::string& key, const LaunchConfig& c) {
    const char* path = std::getenv("LIMA_AUTOTUNE_CACHE");
    if (!path) return;
    std::ofstream f(path, std::ios::app);
    f << key << " " << c.spt << " " << c.chunk_particles << " " << c.listed_grid << " " << c.listed_lanes << " "
      << c.listed_packed << " " << c.fused_thermostat << "\n";
}

// one system's energy record from the device sums (half of every directed-pair LJ sum)
void fill_energies(const lima_engine* E, int r, const double* v, float lam, lima_energies& o) {
    const ReplicaInfo& ri = E->reps_h[r];
    std::memset(&o, 0, sizeof(o));
    o.bond = v[kE_bond]; o.angle = v[kE_angle]; o.dihedral = v[kE_dih];
    o.lj_intra = 0.5 * v[kE_intra]; o.lj_inter = 0.5 * v[kE_inter];
    o.lj_compound_solvent = 0.5 * v[kE_cs]; o.lj_solvent_compound = 0.5 * v[kE_sc];
    o.lj_solvent_solvent = 0.5 * v[kE_ss];
    o.potential = o.bond + o.angle + o.dihedral + o.lj_intra + o.lj_inter + o.lj_compound_solvent +
                  o.lj_solvent_compound + o.lj_solvent_solvent;
    o.kinetic = 0.5 * v[kE_kin] / (ri.dt * ri.dt);
    const double ntot = (double)((ri.chain_end - ri.chain_begin) + (ri.solv_end - ri.solv_begin));
    o.temperature = ntot > 0 ? v[kE_kin] / (ri.dt * ri.dt) / (3.0 * ntot * 8.3145) : 0.0;
    o.virial = 0.5 * v[kE_virial];
    o.thermostat_scalar = lam;
}

// State and forces between the device's float4 arrays and the caller's triples: one kernel forms the
// triples of every array asked for, and they travel at once through a pinned buffer, or (over
// kIoPinned) straight between the caller's arrays and the device.  As a copy of each float4 array
// into a fresh vector and a loop over it, the state of production took 140 us, that of a million
// particles 3.6 ms.
constexpr size_t kIoPinned = (size_t)4 << 20;
struct IoArray {
    float4* dev;
    int n;
    float* host;
};
int io_layout(lima_engine* E, const IoArray (&io)[4], IoArrays& a) {
    size_t total = 0;
    for (int k = 0; k < 4; k++) {
        a.p[k] = io[k].dev;
        a.end[k] = (int)(total += io[k].host ? io[k].n : 0);
    }
    // as large as all four arrays of this engine need: a batch of small engines keeps as many buffers
    if (total && total * 12 <= kIoPinned && !E->io_pinned)
        HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&E->io_pinned), std::min(kIoPinned, E->io_dev.n * sizeof(float)), 0));
    return (int)total;
}
void io_get(lima_engine* E, const IoArray (&io)[4]) {
    IoArrays a{};
    const int total = io_layout(E, io, a);
    if (total == 0) {
        HIP_TRY(hipStreamSynchronize(E->stream));
        return;
    }
    const bool pinned = (size_t)total * 12 <= kIoPinned;
    io_pack_kernel<<<(total + 255) / 256, 256, 0, E->stream>>>(a, E->io_dev.p);
    if (pinned) {
        HIP_TRY(hipMemcpyAsync(E->io_pinned, E->io_dev.p, (size_t)total * 12, hipMemcpyDeviceToHost, E->stream));
        HIP_TRY(hipStreamSynchronize(E->stream));
    }
    size_t at = 0;
    for (const IoArray& x : io) {
        if (!x.host || !x.n) continue;
        if (pinned) std::memcpy(x.host, E->io_pinned + at, (size_t)x.n * 12);
        else HIP_TRY(hipMemcpyAsync(x.host, E->io_dev.p + at, (size_t)x.n * 12, hipMemcpyDeviceToHost, E->stream));
        at += (size_t)3 * x.n;
    }
    if (!pinned) HIP_TRY(hipStreamSynchronize(E->stream));
}
// chain positions (the first array) keep their type, solvent positions (the third) get their mark
void io_set(lima_engine* E, const IoArray (&io)[4]) {
    HIP_TRY(hipStreamSynchronize(E->stream));
    IoArrays a{};
    const int total = io_layout(E, io, a);
    if (total == 0) return;
    const bool pinned = (size_t)total * 12 <= kIoPinned;
    size_t at = 0;
    for (const IoArray& x : io) {
        if (!x.host || !x.n) continue;
        if (pinned) std::memcpy(E->io_pinned + at, x.host, (size_t)x.n * 12);
        else HIP_TRY(hipMemcpyAsync(E->io_dev.p + at, x.host, (size_t)x.n * 12, hipMemcpyHostToDevice, E->stream));
        at += (size_t)3 * x.n;
    }
    if (pinned) HIP_TRY(hipMemcpyAsync(E->io_dev.p, E->io_pinned, (size_t)total * 12, hipMemcpyHostToDevice, E->stream));
    io_unpack_kernel<<<(total + 255) / 256, 256, 0, E->stream>>>(a, E->io_dev.p, E->reps.p, E->solv_rep.p);
    HIP_TRY(hipStreamSynchronize(E->stream));   // the pinned buffer and the caller's arrays are free again
}

// The steps of lima_step_observed: record steps launched directly with their energy sums, each
// record's sums and lambda copied into series [record][system][kEnergyTerms] and lser
// [record][system] (every slot of a record is written before it is read), the plain steps
// between records as graph replays.  allow_capture false keeps to launches and replays of
// graphs already built (no capture or instantiation).
void observed_steps(lima_engine* E, int n, int every, double* series, float* lser, bool allow_capture) {
    const int R = E->R;
    int rec = 0;
    E->sync_step_count();
    for (int s = 0; s < n;) {
        // the recorded step: the step itself with its energy sums (Engine::step + the Analyzer's sums)
        HIP_TRY(hipMemsetAsync(E->energy.p, 0, E->energy.n * sizeof(double), E->stream));
        E->launch_step(E->cur, true);
        HIP_TRY(hipMemcpyAsync(series + (size_t)rec * R * kEnergyTerms, E->energy.p, (size_t)R * kEnergyTerms * 8,
                               hipMemcpyDeviceToDevice, E->stream));
        HIP_TRY(hipMemcpyAsync(lser + (size_t)rec * R, E->lambda_applied.p, (size_t)R * 4, hipMemcpyDeviceToDevice,
                               E->stream));
        E->cur ^= 1;
        E->step++;
        E->since_rebuild++;
        if (E->params.nlist_interval > 0 && E->since_rebuild >= E->params.nlist_interval) {
            E->launch_rebuild(E->cur);
            E->since_rebuild = 0;
            E->n_rebuilds++;
        }
        rec++;
        s++;
        // the plain steps up to the next record (graph replays where the cycle aligns)
        const int run = std::min(every - 1, n - s);
        if (run > 0) E->enqueue_steps(run, allow_capture);
        s += run;
    }
}

}  // namespace

extern "C" {

const char* lima_version(void) { return "lima-mi355x 0.1.0 (gfx950)"; }

int lima_device_count(int* count) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    if (count) *count = n;
    return LIMA_OK;
}

int lima_create(const lima_system* systems, int32_t n_systems, const lima_run_params* params, lima_engine** out) {
    if (!out || !systems || !params) return LIMA_E_ARG;
    *out = nullptr;
    lima_engine* E = new lima_engine();
    E->params = *params;
    try {
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw LimaError(LIMA_E_HIP, "no HIP device available");
        if (params->device < 0 || params->device >= ndev) throw LimaError(LIMA_E_ARG, "device ordinal out of range");
        E->device = params->device;
        HIP_TRY(hipSetDevice(E->device));
        E->scratch_d = scratch_address(E->device);
        E->create_streams();
        validate_and_build(E, systems, n_systems);
        E->fill_ab_tables();
        // Engine::Engine -> handleNLISTS(force) (Engine.cu:35)
        E->launch_rebuild(E->cur);
        HIP_TRY(hipStreamSynchronize(E->stream));
        int st = E->check_errors();
        if (st != LIMA_OK) {
            g_last_error = E->last_error;
            delete E;
            return st;
        }
    } catch (const LimaError& e) {
        g_last_error = e.msg;
        delete E;
        return e.code;
    }
    *out = E;
    return LIMA_OK;
}

void lima_destroy(lima_engine* E) {
    if (!E) return;
    (void)hipSetDevice(E->device);
    (void)hipStreamSynchronize(E->stream);
    delete E;
}

const char* lima_last_error(const lima_engine* E) { return E ? E->last_error.c_str() : g_last_error.c_str(); }

int lima_step_async(lima_engine* E, int32_t n) {
    return guarded(E, [&] {
        if (n < 0) throw LimaError(LIMA_E_ARG, "n_steps < 0");
        HIP_TRY(hipSetDevice(E->device));
        auto t0 = std::chrono::steady_clock::now();
        if (!E->async_open && n > 0) {
            // the device time of queued steps is read at the next lima_sync
            HIP_TRY(hipEventRecord(E->ev_t0, E->stream));
            E->async_open = true;
        }
        E->enqueue_steps(n);
        E->t_host_us += std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
        return LIMA_OK;
    });
}

int lima_sync(lima_engine* E) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        if (E->async_open) {
            HIP_TRY(hipEventRecord(E->ev_t1, E->stream));
            HIP_TRY(hipEventSynchronize(E->ev_t1));
            float ms = 0;
            HIP_TRY(hipEventElapsedTime(&ms, E->ev_t0, E->ev_t1));
            E->t_device_us += ms * 1000.0;
            E->async_open = false;
        }
        HIP_TRY(hipStreamSynchronize(E->stream));
        return E->check_errors();
    });
}

int lima_step(lima_engine* E, int32_t n) {
    return guarded(E, [&] {
        if (n < 0) throw LimaError(LIMA_E_ARG, "n_steps < 0");
        HIP_TRY(hipSetDevice(E->device));
        if (E->async_open) {   // steps queued by lima_step_async are timed up to here
            int st = lima_sync(E);
            if (st != LIMA_OK) return st;
        }
        auto t0 = std::chrono::steady_clock::now();
        HIP_TRY(hipEventRecord(E->ev_t0, E->stream));
        E->enqueue_steps(n);
        HIP_TRY(hipEventRecord(E->ev_t1, E->stream));
        E->fetch_errors();
        auto t1 = std::chrono::steady_clock::now();
        HIP_TRY(hipStreamSynchronize(E->stream));
        float ms = 0;
        HIP_TRY(hipEventElapsedTime(&ms, E->ev_t0, E->ev_t1));
        E->t_device_us += ms * 1000.0;
        E->t_host_us += std::chrono::duration<double, std::micro>(t1 - t0).count();
        return E->fetched_errors();
    });
}

int lima_rebuild_neighbors(lima_engine* E) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        E->launch_rebuild(E->cur);
        E->since_rebuild = 0;
        E->n_rebuilds++;
        return E->check_errors();
    });
}

int lima_get_state(lima_engine* E, float* cx, float* cxm, float* sx, float* sxm) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        io_get(E, {{E->cpos[E->cur].p, E->NCH, cx}, {E->cprev.p, E->NCH, cxm}, {E->spos[E->cur].p, E->NS, sx}, {E->sprev.p, E->NS, sxm}});
        return LIMA_OK;
    });
}

int lima_set_state(lima_engine* E, const float* cx, const float* cxm, const float* sx, const float* sxm) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        auto in = [](const float* p) { return const_cast<float*>(p); };   // read only
        io_set(E, {{E->cpos[E->cur].p, E->NCH, in(cx)}, {E->cprev.p, E->NCH, in(cxm)}, {E->spos[E->cur].p, E->NS, in(sx)}, {E->sprev.p, E->NS, in(sxm)}});
        return LIMA_OK;
    });
}

int lima_get_forces(lima_engine* E, float* cf, float* sf) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        io_get(E, {{E->cforce.p, E->NCH, cf}, {E->sforce.p, E->NS, sf}, {nullptr, 0, nullptr}, {nullptr, 0, nullptr}});
        return LIMA_OK;
    });
}

int lima_compute_forces(lima_engine* E, float* cf, float* sf) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        if (E->params.accumulation == LIMA_ACCUM_FIXED64) E->launch_forces<false, true, false>(E->cur);
        else E->launch_forces<false, false, false>(E->cur);
        int st = E->check_errors();
        if (st != LIMA_OK) return st;
        return lima_get_forces(E, cf, sf);
    });
}

int lima_get_energies(lima_engine* E, lima_energies* out) {
    return guarded(E, [&] {
        if (!out) throw LimaError(LIMA_E_ARG, "null output");
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipMemsetAsync(E->energy.p, 0, E->energy.n * sizeof(double), E->stream));
        if (E->params.accumulation == LIMA_ACCUM_FIXED64) E->launch_forces<false, true, true>(E->cur);
        else E->launch_forces<false, false, true>(E->cur);
        HIP_TRY(hipStreamSynchronize(E->stream));
        std::vector<double> e(E->energy.n);
        HIP_TRY(hipMemcpy(e.data(), E->energy.p, e.size() * sizeof(double), hipMemcpyDeviceToHost));
        std::vector<float> lam(E->R);
        HIP_TRY(hipMemcpy(lam.data(), E->lambda_applied.p, E->R * sizeof(float), hipMemcpyDeviceToHost));
        for (int r = 0; r < E->R; r++) fill_energies(E, r, &e[(size_t)r * kEnergyTerms], lam[r], out[r]);
        return E->check_errors();
    });
}

// Steps with the reference's per-step logs of one system: Engine::offloadLoggingData /
// offloadTrainData (Engine.cu:288-310) move device rings to the host every 100 steps
// (STEPS_PER_TRAINDATATRANSFER, Constants.cuh:99); here the rings are copied into the
// caller's arrays at the same cadence.
constexpr int kLogRing = 100;

int lima_step_logged(lima_engine* E, int32_t n, int32_t system, int32_t slots, float* logdata, float* traindata) {
    return guarded(E, [&] {
        if (n < 0 || system < 0 || system >= E->R) throw LimaError(LIMA_E_ARG, "n_steps < 0 or system out of range");
        if (n > 0 && !logdata && !traindata) throw LimaError(LIMA_E_ARG, "no output");
        const ReplicaInfo& ri = E->reps_h[system];
        const int nc = ri.comp_end - ri.comp_begin;
        int maxp = 0;
        for (int c = ri.comp_begin; c < ri.comp_end; c++) maxp = std::max(maxp, E->comp_off_h[c + 1] - E->comp_off_h[c]);
        if (traindata && (slots < std::max(maxp, 1) || slots > kCompoundBlock))
            throw LimaError(LIMA_E_ARG, "slots_per_compound must cover the largest compound and be at most 128");
        if (nc == 0) throw LimaError(LIMA_E_ARG, "the system has no compounds to log");
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipStreamSynchronize(E->stream));
        const size_t per_step = (size_t)nc * std::max(slots, 1) * 9;
        E->log_data.grow((size_t)kLogRing * 10);
        if (traindata) E->train_data.grow(kLogRing * per_step);
        // the rings enter the captured step through its arguments: recapture with them, and again without
        auto reset_graph = [&] {
            E->drop_graphs();
        };
        struct Off {   // logging is off again however the call ends
            lima_engine* E;
            ~Off() {
                E->log_rep = -1;
                E->log_train = false;
                E->drop_graphs();
            }
        } off{E};
        E->log_rep = system;
        E->log_train = traindata != nullptr;
        E->log_slots = traindata ? slots : 0;
        E->log_ring = kLogRing;
        reset_graph();
        std::vector<float> hl((size_t)kLogRing * 10), ht(traindata ? kLogRing * per_step : 0);
        int st = LIMA_OK;
        for (int done = 0; done < n && st == LIMA_OK;) {
            const int chunk = std::min(kLogRing, n - done);
            const long long step0 = E->step;
            E->enqueue_steps(chunk);
            HIP_TRY(hipStreamSynchronize(E->stream));
            st = E->check_errors();
            HIP_TRY(hipMemcpy(hl.data(), E->log_data.p, hl.size() * 4, hipMemcpyDeviceToHost));
            if (traindata) HIP_TRY(hipMemcpy(ht.data(), E->train_data.p, ht.size() * 4, hipMemcpyDeviceToHost));
            for (int i = 0; i < chunk; i++) {
                const size_t ring = (size_t)((step0 + i) % kLogRing);
                if (logdata) std::memcpy(logdata + (size_t)(done + i) * 10, hl.data() + ring * 10, 40);
                if (traindata) std::memcpy(traindata + (size_t)(done + i) * per_step, ht.data() + ring * per_step, per_step * 4);
            }
            done += chunk;
        }
        return st;
    });
}

int lima_step_observed(lima_engine* E, int32_t n, int32_t every, lima_energies* out) {
    return guarded(E, [&] {
        if (n < 0 || every <= 0) throw LimaError(LIMA_E_ARG, "n_steps < 0 or every <= 0");
        if (!out && n > 0) throw LimaError(LIMA_E_ARG, "null output");
        HIP_TRY(hipSetDevice(E->device));
        const int R = E->R;
        const int nrec = (n + every - 1) / every;
        std::vector<double> e((size_t)std::max(nrec, 1) * R * kEnergyTerms);
        std::vector<float> lam((size_t)std::max(nrec, 1) * R);
        DBuf<double> series;
        DBuf<float> lser;
        series.alloc(e.size());
        lser.alloc(lam.size());
        observed_steps(E, n, every, series.p, lser.p, true);
        HIP_TRY(hipStreamSynchronize(E->stream));
        if (nrec > 0) {
            HIP_TRY(hipMemcpy(e.data(), series.p, (size_t)nrec * R * kEnergyTerms * 8, hipMemcpyDeviceToHost));
            HIP_TRY(hipMemcpy(lam.data(), lser.p, (size_t)nrec * R * 4, hipMemcpyDeviceToHost));
        }
        for (int k = 0; k < nrec; k++)
            for (int r = 0; r < R; r++)
                fill_energies(E, r, &e[((size_t)k * R + r) * kEnergyTerms], lam[(size_t)k * R + r], out[(size_t)k * R + r]);
        return E->check_errors();
    });
}

int lima_step_observed_noalloc(lima_engine* E, int32_t n, int32_t every, lima_energies* out) {
    return guarded(E, [&] {
        if (n < 0 || every <= 0) throw LimaError(LIMA_E_ARG, "n_steps < 0 or every <= 0");
        if (!out && n > 0) throw LimaError(LIMA_E_ARG, "null output");
        HIP_TRY(hipSetDevice(E->device));
        const int R = E->R;
        const size_t nrec = (size_t)((n + every - 1) / every);
        const size_t ser_bytes = nrec * R * kEnergyTerms * sizeof(double);
        const size_t lam_off = (ser_bytes + 255) & ~(size_t)255;
        if (lam_off + nrec * R * sizeof(float) > kObservedScratchBytes) {
            char buf[200];
            snprintf(buf, sizeof(buf), "%zu records x %d systems exceed the no-alloc staging of %zu bytes (%zu bytes per record and system)",
                     nrec, R, kObservedScratchBytes, kEnergyTerms * sizeof(double) + sizeof(float));
            throw LimaError(LIMA_E_ARG, buf);
        }
        unsigned char* base = E->scratch_d;
        if (!base) throw LimaError(LIMA_E_UNSUPPORTED, "no-alloc staging is not set up on this device");
        double* series = reinterpret_cast<double*>(base);
        float* lser = reinterpret_cast<float*>(base + lam_off);
        observed_steps(E, n, every, series, lser, false);
        HIP_TRY(hipStreamSynchronize(E->stream));
        // out of the staging in fixed host chunks (no host allocation either)
        constexpr size_t kChunk = 64;
        double e[kChunk * kEnergyTerms];
        float lam[kChunk];
        const size_t total = nrec * R;
        for (size_t i = 0; i < total; i += kChunk) {
            const size_t m = std::min(kChunk, total - i);
            HIP_TRY(hipMemcpy(e, series + i * kEnergyTerms, m * kEnergyTerms * sizeof(double), hipMemcpyDeviceToHost));
            HIP_TRY(hipMemcpy(lam, lser + i, m * sizeof(float), hipMemcpyDeviceToHost));
            for (size_t j = 0; j < m; j++) fill_energies(E, (int)((i + j) % R), &e[j * kEnergyTerms], lam[j], out[i + j]);
        }
        return E->check_errors();
    });
}

int lima_get_neighbor_counts(lima_engine* E, int32_t* ccc, int32_t* csc, int32_t* ssc) {
    return guarded(E, [&] {
        HIP_TRY(hipStreamSynchronize(E->stream));
        if (ccc && E->NC) HIP_TRY(hipMemcpy(ccc, E->cc_cnt.p, E->NC * sizeof(int), hipMemcpyDeviceToHost));
        if (csc && E->NC) HIP_TRY(hipMemcpy(csc, E->cs_cnt.p, E->NC * sizeof(int), hipMemcpyDeviceToHost));
        if (ssc && E->NS) HIP_TRY(hipMemcpy(ssc, E->ss_cnt.p, E->NS * sizeof(int), hipMemcpyDeviceToHost));
        return LIMA_OK;
    });
}

int lima_get_neighbors(lima_engine* E, int32_t* cci, int32_t* csi, int32_t* ssi) {
    return guarded(E, [&] {
        HIP_TRY(hipStreamSynchronize(E->stream));
        const lima_run_params& P = E->params;
        if (cci && E->NC) HIP_TRY(hipMemcpy(cci, E->cc_ids.p, (size_t)E->NC * P.max_compound_neighbors * sizeof(int), hipMemcpyDeviceToHost));
        if (csi && E->NC) HIP_TRY(hipMemcpy(csi, E->cs_ids.p, (size_t)E->NC * P.max_compound_solvents * sizeof(int), hipMemcpyDeviceToHost));
        if (ssi && E->NS) {
            const size_t ld = E->ss_ld();
            std::vector<int> t((size_t)E->NS * ld);
            HIP_TRY(hipMemcpy(t.data(), E->ss_ids.p, t.size() * sizeof(int), hipMemcpyDeviceToHost));
            for (int s = 0; s < E->NS; s++)
                for (int k = 0; k < P.max_solvent_neighbors; k++) ssi[(size_t)s * P.max_solvent_neighbors + k] = t[(size_t)s * ld + k];
        }
        return LIMA_OK;
    });
}

int lima_set_neighbors(lima_engine* E, const int32_t* ccc, const int32_t* cci, const int32_t* csc, const int32_t* csi,
                       const int32_t* ssc, const int32_t* ssi) {
    return guarded(E, [&] {
        HIP_TRY(hipStreamSynchronize(E->stream));
        const lima_run_params& P = E->params;
        // every id must name an entity of the same replica (the kernels index per-replica ranges)
        std::vector<int> comp_rep_h(E->NC), solv_rep_h(E->NS);
        for (int r = 0; r < E->R; r++) {
            for (int c = E->reps_h[r].comp_begin; c < E->reps_h[r].comp_end; c++) comp_rep_h[c] = r;
            for (int s = E->reps_h[r].solv_begin; s < E->reps_h[r].solv_end; s++) solv_rep_h[s] = r;
        }
        if (ccc && cci && E->NC) {
            for (int c = 0; c < E->NC; c++) {
                if (ccc[c] < 0 || ccc[c] > P.max_compound_neighbors) throw LimaError(LIMA_E_CAPACITY, "compound list count exceeds capacity");
                const ReplicaInfo& ri = E->reps_h[comp_rep_h[c]];
                for (int k = 0; k < ccc[c]; k++) {
                    const int j = cci[(size_t)c * P.max_compound_neighbors + k];
                    if (j < ri.comp_begin || j >= ri.comp_end || j == c) throw LimaError(LIMA_E_ARG, "compound neighbour id outside the compound's system");
                }
            }
            HIP_TRY(hipMemcpy(E->cc_cnt.p, ccc, E->NC * sizeof(int), hipMemcpyHostToDevice));
            HIP_TRY(hipMemcpy(E->cc_ids.p, cci, (size_t)E->NC * P.max_compound_neighbors * sizeof(int), hipMemcpyHostToDevice));
        }
        if (csc && csi && E->NC) {
            for (int c = 0; c < E->NC; c++) {
                if (csc[c] < 0 || csc[c] > P.max_compound_solvents) throw LimaError(LIMA_E_CAPACITY, "compound solvent list count exceeds capacity");
                const ReplicaInfo& ri = E->reps_h[comp_rep_h[c]];
                for (int k = 0; k < csc[c]; k++) {
                    const int s = csi[(size_t)c * P.max_compound_solvents + k];
                    if (s < ri.solv_begin || s >= ri.solv_end) throw LimaError(LIMA_E_ARG, "solvent id outside the compound's system");
                }
            }
            HIP_TRY(hipMemcpy(E->cs_cnt.p, csc, E->NC * sizeof(int), hipMemcpyHostToDevice));
            HIP_TRY(hipMemcpy(E->cs_ids.p, csi, (size_t)E->NC * P.max_compound_solvents * sizeof(int), hipMemcpyHostToDevice));
        }
        if (ssc && ssi && E->NS) {
            for (int s = 0; s < E->NS; s++) {
                if (ssc[s] < 0 || ssc[s] > P.max_solvent_neighbors) throw LimaError(LIMA_E_CAPACITY, "solvent list count exceeds capacity");
                const ReplicaInfo& ri = E->reps_h[solv_rep_h[s]];
                for (int k = 0; k < ssc[s]; k++) {
                    const int j = ssi[(size_t)s * P.max_solvent_neighbors + k];
                    if (j < ri.solv_begin || j >= ri.solv_end || j == s) throw LimaError(LIMA_E_ARG, "solvent neighbour id outside the solvent's system");
                }
            }
            const size_t ld = E->ss_ld();
            std::vector<int> t((size_t)E->NS * ld, 0);
            for (int s = 0; s < E->NS; s++)
                for (int k = 0; k < ssc[s]; k++) t[(size_t)s * ld + k] = ssi[(size_t)s * P.max_solvent_neighbors + k];
            HIP_TRY(hipMemcpy(E->ss_cnt.p, ssc, E->NS * sizeof(int), hipMemcpyHostToDevice));
            HIP_TRY(hipMemcpy(E->ss_ids.p, t.data(), t.size() * sizeof(int), hipMemcpyHostToDevice));
        }
        if (E->NC) {
            E->launch_work_list(E->nlist_args(E->cur), E->stream);
            HIP_TRY(hipStreamSynchronize(E->stream));
        }
        return LIMA_OK;
    });
}

int lima_get_timings(lima_engine* E, double* out5) {
    return guarded(E, [&] {
        if (!out5) throw LimaError(LIMA_E_ARG, "null output");
        out5[0] = E->t_device_us;
        out5[1] = E->t_rebuild_us;
        out5[2] = E->t_host_us;
        out5[3] = (double)E->step;
        out5[4] = (double)E->n_rebuilds;
        return LIMA_OK;
    });
}

int lima_time_kernels(lima_engine* E, int32_t reps, double* out8) {
    return guarded(E, [&] {
        if (!out8 || reps <= 0) throw LimaError(LIMA_E_ARG, "bad arguments");
        double* out6 = out8;
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipStreamSynchronize(E->stream));
        hipEvent_t e0, e1;
        HIP_TRY(hipEventCreate(&e0));
        HIP_TRY(hipEventCreate(&e1));
        StepArgs a = E->step_args(E->cur);
        a.kclock = nullptr;   // these launches are not steps: they stay out of the in-step clock
        const bool fx = E->params.accumulation == LIMA_ACCUM_FIXED64;
        auto timeit = [&](auto&& launch) -> double {
            launch();   // warm
            HIP_TRY(hipEventRecord(e0, E->stream));
            for (int i = 0; i < reps; i++) launch();
            HIP_TRY(hipEventRecord(e1, E->stream));
            HIP_TRY(hipEventSynchronize(e1));
            float ms = 0;
            HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
            return ms * 1000.0 / reps;
        };
        for (int k = 0; k < 8; k++) out8[k] = 0.0;
        auto role = [&](int roles) {
            return timeit([&] {
                if (fx) E->launch_roles<true, false>(a, roles);
                else E->launch_roles<false, false>(a, roles);
            });
        };
        auto integrate = [&](bool compounds, bool solvents) {
            return timeit([&] {
                if (fx) E->launch_integrate<false, true, false>(a, compounds, solvents);
                else E->launch_integrate<false, false, false>(a, compounds, solvents);
            });
        };
        const bool solv = E->params.enable_solvents && E->NS > 0;
        if (E->NB > 0) out6[4] = role(lima_engine::kRoleBridges);
        if (E->NC > 0) out8[7] = role(lima_engine::kRoleLocal);
        if (solv && !E->scwork_h.empty()) out6[0] = role(lima_engine::kRoleAllPairs);
        if (solv) out8[6] = role(lima_engine::kRoleListedSolvents);
        if (E->NC > 0) {
            out6[1] = role(lima_engine::kRoleListed);
            out6[2] = integrate(true, false);
        }
        if (solv) out6[3] = integrate(false, true);
        out6[5] = timeit([&] { E->launch_rebuild(E->cur); });
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return E->check_errors();
    });
}

int lima_get_config(lima_engine* E, int32_t* out, int32_t n_out) {
    return guarded(E, [&] {
        if (!out || n_out < 0) throw LimaError(LIMA_E_ARG, "null output or negative count");
        int chunk = E->cfg.chunk_particles;
        for (const ReplicaInfo& ri : E->reps_h) chunk = std::max(chunk, E->chunk_target(ri));
        const int32_t v[12] = {E->cfg.spt, chunk, (int32_t)E->scwork_h.size(), E->kmax, E->cfg.use_graph,
                               E->n_cells, E->n_stiles, E->R, E->cfg.listed_grid > 0 ? E->cfg.listed_grid : 2 * E->listed_blocks(),
                               E->cfg.listed_lanes, E->listed_form(), E->thermo_form()};
        for (int i = 0; i < std::min<int32_t>(n_out, 12); i++) out[i] = v[i];
        return LIMA_OK;
    });
}

int lima_set_kernel_clock(lima_engine* E, int32_t on) {
    return guarded(E, [&] {
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipStreamSynchronize(E->stream));
        const bool want = on != 0;
        if (want) {
            ensure(E->kclock, (size_t)4);
            HIP_TRY(hipMemset(E->kclock.p, 0xFF, sizeof(unsigned long long)));
            HIP_TRY(hipMemset(E->kclock.p + 1, 0, 3 * sizeof(unsigned long long)));
        }
        if (want != E->kclock_on) {
            E->kclock_on = want;
            E->drop_graphs();
        }
        return LIMA_OK;
    });
}

int lima_get_kernel_clock(lima_engine* E, double* total_us, int64_t* launches) {
    return guarded(E, [&] {
        if (!total_us || !launches) throw LimaError(LIMA_E_ARG, "null output");
        if (!E->kclock_on) throw LimaError(LIMA_E_ARG, "the kernel clock is off (lima_set_kernel_clock)");
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipStreamSynchronize(E->stream));
        unsigned long long v[4];
        HIP_TRY(hipMemcpy(v, E->kclock.p, sizeof v, hipMemcpyDeviceToHost));
        int khz = 0;
        HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, E->device));
        if (khz <= 0) throw LimaError(LIMA_E_UNSUPPORTED, "the device reports no wall-clock rate");
        *total_us = (double)v[2] * 1000.0 / khz;
        *launches = (int64_t)v[3];
        return LIMA_OK;
    });
}

// Autotuner: picks the all-pairs role's chunk size, the listed compound role's grid and form, and where the
// thermostat runs, by timing whole steps of each from the current state, which is restored.  Results are
// cached per shape histogram in the process and, when LIMA_AUTOTUNE_CACHE names a file, across processes.
int lima_autotune(lima_engine* E, int32_t reps) {
    return guarded(E, [&] {
        if (reps <= 0) reps = 10;
        HIP_TRY(hipSetDevice(E->device));
        HIP_TRY(hipStreamSynchronize(E->stream));
        const std::string key = shape_key(E);
        LaunchConfig best = E->cfg;
        bool have = false;
        {
            std::lock_guard<std::mutex> lk(g_tune_mu);
            load_tune_file();
            auto it = g_tune_cache.find(key);
            if (it != g_tune_cache.end()) { best = it->second; have = true; }
        }
        if (!have) {
            // Each shape is timed on the whole step: captured cycles, rebuilds
            // included, from the same saved state, which is restored afterwards.  Isolated kernel
            // timings ranked the all-pairs chunk sizes differently from the step they run in.
            hipEvent_t e0, e1;
            HIP_TRY(hipEventCreate(&e0));
            HIP_TRY(hipEventCreate(&e1));
            const int NCH = E->NCH, NS = E->NS, R = E->R;
            DBuf<float4> st_save;
            DBuf<int> lists_save;
            st_save.alloc((size_t)2 * std::max(NCH + NS, 1));
            lists_save.alloc(std::max<size_t>(list_words(E), 1));
            save_state(E, st_save.p);
            save_lists(E, lists_save.p);
            std::vector<float> lam(R), lam_applied(R);
            HIP_TRY(hipStreamSynchronize(E->stream));
            HIP_TRY(hipMemcpy(lam.data(), E->lambda.p, R * sizeof(float), hipMemcpyDeviceToHost));
            HIP_TRY(hipMemcpy(lam_applied.data(), E->lambda_applied.p, R * sizeof(float), hipMemcpyDeviceToHost));
            const int cur0 = E->cur;
            const long long step0 = E->step, since0 = E->since_rebuild, nreb0 = E->n_rebuilds;
            auto restore = [&] {
                HIP_TRY(hipStreamSynchronize(E->stream));
                E->cur = cur0;
                load_state(E, st_save.p);
                load_lists(E, lists_save.p);
                HIP_TRY(hipStreamSynchronize(E->stream));
                HIP_TRY(hipMemcpy(E->lambda.p, lam.data(), R * sizeof(float), hipMemcpyHostToDevice));
                HIP_TRY(hipMemcpy(E->lambda_applied.p, lam_applied.data(), R * sizeof(float), hipMemcpyHostToDevice));
                E->step = step0;
                E->since_rebuild = since0;
                E->n_rebuilds = nreb0;
            };
            const int cyc = E->cycle_steps();
            int timed = std::max(reps, cyc);
            // ms per step of the current shape: one cycle to capture and warm, then the timed steps
            auto trial = [&]() -> double {
                E->drop_graphs();
                E->build_scwork();
                E->reps.upload(E->reps_h);
                E->enqueue_steps(cyc);
                HIP_TRY(hipEventRecord(e0, E->stream));
                E->enqueue_steps(timed);
                HIP_TRY(hipEventRecord(e1, E->stream));
                HIP_TRY(hipEventSynchronize(e1));
                float ms = 0;
                HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
                const int st = E->check_errors();
                restore();
                return st == LIMA_OK ? (double)ms / timed : 1e30;
            };
            // trials of at least 8 ms each, in whole list cycles, sized from one probe of the
            // current shape: 10-step trials (2 ms on the production system) picked a shape 27%
            // slower than the best on a freshly started device
            {
                const double ms = trial();
                if (ms > 0.0 && ms < 1e29) {
                    const int want = (int)std::ceil(8.0 / ms);
                    timed = std::max(timed, (want + cyc - 1) / cyc * cyc);
                }
            }
            // the chunk size that every system has by its own size, or 0
            int own_chunk = -1;
            E->cfg.chunk_particles = 0;
            for (const ReplicaInfo& ri : E->reps_h)
                own_chunk = own_chunk < 0 || own_chunk == E->chunk_target(ri) ? E->chunk_target(ri) : 0;
            // three sweeps, the fastest time of each shape (clocks ramp after idle periods)
            constexpr int kSweeps = 3;
            // the all-pairs shape, swept again after the listed kernels' choices below (a shape
            // picked while a slow listed form dominates the step can be the wrong one once it is gone)
            auto sweep_all_pairs = [&] {
                if (!(E->params.enable_solvents && E->NS > 0 && E->NCH > 0)) return;
                const int chunks[4] = {256, 512, 1024, 2048};
                double tmin[4] = {1e30, 1e30, 1e30, 1e30};
                for (int sweep = 0; sweep < kSweeps; sweep++) {
                    for (int j = 0; j < 4; j++) {
                        E->cfg.chunk_particles = chunks[j];
                        tmin[j] = std::min(tmin[j], trial());
                    }
                }
                const double tbest = *std::min_element(tmin, tmin + 4);
                // shapes within 1% of the best step are ties at the trials' resolution.  Among them, the
                // chunk that the engine takes untuned (the 256 replicas took 512 over their own 256, equal
                // in the trials, 1.3% slower over 60 steps and 2.3% over 2,000).  Else, of those
                // whose all-pairs role alone is within 5% of the fastest (a shape with too few
                // work items to fill the device alone leaves the step to the other roles
                // at this size and may not at another), the one writing the fewest
                // per-chunk partials (less HBM traffic; shapes that differ only in chunking run
                // within a few per cent alone), then the fastest alone
                double kms[4];
                long long parts[4];
                double kbest = 1e30;
                for (int j = 0; j < 4; j++) {
                    kms[j] = 1e30;
                    parts[j] = 0;
                    if (tmin[j] > 1.01 * tbest) continue;
                    E->cfg.chunk_particles = chunks[j];
                    E->build_scwork();
                    E->reps.upload(E->reps_h);
                    for (int r = 0; r < E->R; r++)
                        parts[j] += (long long)E->reps_h[r].chunk_count * (E->reps_h[r].solv_end - E->reps_h[r].solv_begin);
                    StepArgs ka = E->step_args(E->cur);
                    ka.kclock = nullptr;
                    auto launch = [&] {
                        if (E->params.accumulation == LIMA_ACCUM_FIXED64) E->launch_roles<true, false>(ka, lima_engine::kRoleAllPairs);
                        else E->launch_roles<false, false>(ka, lima_engine::kRoleAllPairs);
                    };
                    launch();
                    HIP_TRY(hipEventRecord(e0, E->stream));
                    for (int k = 0; k < 5; k++) launch();
                    HIP_TRY(hipEventRecord(e1, E->stream));
                    HIP_TRY(hipEventSynchronize(e1));
                    float ms = 0;
                    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
                    kms[j] = ms;
                    kbest = std::min(kbest, (double)ms);
                }
                long long pbest = -1;
                double kpick = 1e30;
                for (int j = 0; j < 4; j++) {
                    if (kms[j] > 1.05 * kbest) continue;   // not a step tie, or slow alone
                    if (pbest < 0 || parts[j] < pbest || (parts[j] == pbest && kms[j] < kpick)) {
                        pbest = parts[j];
                        kpick = kms[j];
                        best.chunk_particles = chunks[j];
                    }
                }
                for (int j = 0; j < 4; j++)
                    if (chunks[j] == own_chunk && tmin[j] <= 1.01 * tbest) best.chunk_particles = own_chunk;
                restore();
                E->cfg.chunk_particles = best.chunk_particles;
            };
            sweep_all_pairs();
            if (E->NC > 0) {
                // grid sizes, with the packed and the plain listed kernel where compounds allow both
                // (they give the same sums: a small system fills the device better with the plain one)
                // forms: packed (1), plain (0), plain with split small items (2, FP32 only)
                const int grids[4] = {1024, 2048, 4096, 8192};
                const int forms[3] = {1, 0, 2};
                const int nform = !E->pack_ppl() ? 1 : (E->params.accumulation == LIMA_ACCUM_FIXED64 ? 2 : 3);
                double gmin[3][4];
                for (auto& row : gmin)
                    for (double& v : row) v = 1e30;
                for (int sweep = 0; sweep < kSweeps; sweep++) {
                    for (int k = 0; k < nform; k++) {
                        E->cfg.listed_packed = forms[k];
                        for (int j = 0; j < 4; j++) {
                            E->cfg.listed_grid = grids[j];
                            gmin[k][j] = std::min(gmin[k][j], trial());
                        }
                    }
                }
                double gbest = 1e30;
                for (int k = 0; k < nform; k++)
                    for (int j = 0; j < 4; j++)
                        if (gmin[k][j] < gbest) { gbest = gmin[k][j]; best.listed_grid = grids[j]; best.listed_packed = forms[k]; }
                E->cfg.listed_grid = best.listed_grid;
                E->cfg.listed_packed = best.listed_packed;
            }
            if (E->thermo_ok) {
                // the thermostat as its own kernel (between the steps of a graph, beside the next one's
                // forces), or in the integrate launch's last blocks: that saves its launch, but every
                // integrator block then releases its partial at device scope, which writes back its XCD's L2
                double fmin[2] = {1e30, 1e30};
                for (int sweep = 0; sweep < kSweeps; sweep++) {
                    for (int j = 0; j < 2; j++) {
                        E->cfg.fused_thermostat = j;
                        fmin[j] = std::min(fmin[j], trial());
                    }
                }
                best.fused_thermostat = fmin[1] < fmin[0] ? 1 : 0;
                E->cfg.fused_thermostat = best.fused_thermostat;
            }
            sweep_all_pairs();
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            // choices that the systems did not offer (no solvents, no compounds) are kept as what the engine runs
            if (best.chunk_particles <= 0) best.chunk_particles = 1024;
            if (best.listed_packed < 0) best.listed_packed = E->listed_form();
            std::lock_guard<std::mutex> lk(g_tune_mu);
            g_tune_cache[key] = best;
            save_tune_entry(key, best);
        }
        E->cfg = best;
        E->build_scwork();
        E->reps.upload(E->reps_h);
        E->drop_graphs();
        return E->check_errors();
    });
}

int lima_get_parameters(lima_engine* E, int32_t system, double* params) {
    return guarded(E, [&] {
        if (!params || system < 0 || system >= E->R) throw LimaError(LIMA_E_ARG, "system index out of range or null output");
        get_parameters(E, system, params);
        return LIMA_OK;
    });
}

int lima_set_parameters(lima_engine* E, int32_t system, const double* params) {
    return guarded(E, [&] {
        if (!params || system < 0 || system >= E->R) throw LimaError(LIMA_E_ARG, "system index out of range or null input");
        set_parameters(E, system, params);
        return LIMA_OK;
    });
}

int lima_adjoint_run(lima_engine* E, const lima_adjoint_spec* spec, double* loss, double* grad) {
    return guarded(E, [&] {
        if (!spec) throw LimaError(LIMA_E_ARG, "null spec");
        return adjoint_run(E, *spec, loss, grad);
    });
}

int lima_record_frames(lima_engine* E, int32_t n_frames, float* chain_forces, float* solvent_forces, double* potential) {
    return guarded(E, [&] { return record_frames(E, n_frames, chain_forces, solvent_forces, potential); });
}

}  // extern "C"
