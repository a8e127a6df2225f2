// kernels.h — gfx950 kernels of one LIMA_MD step and of the neighbour-list build.
//
// Mapping to the reference (Quantom/Quantom/Engine.cu):
//   step_forces_kernel, by role
//     bridge_role                compoundBridgeKernel          1168-1223
//     local_role                 compoundKernel 918-937 (bonded, intra-compound LJ)
//     listed_role, listed_packed_role
//                                compoundKernel 939-974 (inter-compound and solvent-list LJ)
//     all_pairs_role             solventForceKernel 1099-1117 (solvent <- every chain particle)
//     solvent_listed_role        solventForceKernel 1111, 1121-1123 (solvent-solvent LJ)
//   step_integrate_kernel, by role
//     compound_integrate_role    compoundKernel 981-1056 (sums, integrate, PBC)
//     solvent_integrate_role     solventForceKernel 1129-1155 (sums, integrate, PBC)
//   thermostat_kernel            Engine::handleBoxtemp 362-393, as an FP64 device reduction
//   nl_*                         Engine::updateNeighborLists 146-287, on the device
//
// Every kernel is replica-aware: entities carry their replica id and read the
// box length, time step and type tables of that replica, so one launch covers
// any number of independent systems.
#pragma once
#include <algorithm>
#include <type_traits>
#include "bonded.h"
#include "device_common.h"

namespace lima {

struct I3 {
    long long x, y, z;
};

struct StepArgs {
    const ReplicaInfo* reps;
    int n_replicas;
    // chain particles
    const float4* cpos;      // current (x, y, z, type bits)
    float4* cpos_next;
    float4* cprev;
    float4* cforce;
    float4* fbridge;
    const uint32_t* intra_mask;   // [n_chain*4]
    const int* xoff;              // cross-compound exclusions [n_chain+1]
    const int2* xent;             // (compound, local)
    // compounds
    int n_comp;
    const int* comp_off;          // [n_comp+1]
    const int* comp_rep;
    const int* comp_key;          // compound-local key index
    const float* comp_sphere;
    const int* bond_off; const BondD* bonds;
    const int* angle_off; const AngleD* angles;
    const int* dih_off; const DihD* dihs;
    const int* inc_off; const uint32_t* inc;   // per chain particle: term incidences
    // bridges
    int n_bridges;
    const int* br_off; const int* br_glob; const int* br_rep;
    const int* brb_off; const BondD* brb;
    const int* bra_off; const AngleD* bra;
    const int* brd_off; const DihD* brd;
    // solvents
    int n_solv;
    const float4* spos;
    float4* spos_next;
    float4* sprev;
    float4* sforce;
    const int* solv_rep;
    const int4* stiles;           // (replica, begin, end, tile index) per solvent-integrate tile
    // type tables per replica
    const float* mass;            // [R*32]
    // pair parameters (sigma^2, 24 eps, -48 eps, sigma) with each call site's mixing rule
    const float4* tab_sc;         // [R*32] solvent <- chain type, arithmetic eps
    const float4* tab_cs;         // [R*32] chain type <- solvent, geometric eps
    const float4* tab_inter;      // [R*1024] arithmetic
    const float4* tab_intra;      // [R*1024] geometric
    const float4* tab_ss;         // [R]
    // lists
    int cap_cc, cap_cs, cap_ss;
    const int* cc_cnt; const int* cc_ids;
    const int* cs_cnt; const int* cs_ids;
    const int* ss_cnt; const int* ss_ids;   // rows: ss_ids[s*ss_ld + k], ss_ld = cap_ss rounded up to 4
    int ss_ld;
    float4* ss_part;              // solvent-solvent local sums
    float4* ss_img;               // the solvent's position after the reference's re-imaging sequence
    const int* cw_off; const int* cw_total;
    const int* item_comp;         // [work item] its compound (written with cw_off at each rebuild)
    const int* run_off; const int* run_cs_off; const int* run_total; const int* run_comp;   // listed_packed_role's runs
    const float2* tab_inter_ab;   // [R*1024] lj_ab of tab_inter, [source type * 32 + target type]
    const float2* tab_intra_ab;   // [R*1024] lj_ab of tab_intra
    // partial forces
    float4* partC;  I3* partC_fx;   // [slot*128 + p]
    float4* cloc;   I3* cloc_fx;    // [n_chain] bonded + intra-compound LJ (local_role); the integrator adds the bridges'
    float4* partS;  I3* partS_fx;   // [chunk*n_solv + s]
    const SCWork* scwork; int n_scwork;
    int chunk_cap;                // rows of the largest solvent<-chain chunk (LDS tile size)
    const int* comp_row;          // [n_comp+1] first row of each compound in all_pairs_role's tiles (multiples of kRowPad)
    const int* row_src;           // [rows] chain particle of each row, -1: padding
    // thermostat
    const float* lambda;          // [R] applied this step
    double* ke_comp;              // [n_comp]
    double* ke_stile;             // [n_stiles]
    int ke_ref;                   // 1: the thermostat sums read the reference's two-step kinetic energy
    // per-step logs of one replica (the compoundKernel's data log, Engine.cu:1019-1046)
    int log_rep;                  // logged replica, -1: none
    int log_slots;                // particle slots per compound (the reference's MAX_COMPOUND_PARTICLES)
    int log_ring;                 // steps the device rings hold; step k writes slot k % log_ring
    const long long* step_count;  // [R] steps done before this one
    // the step's thermostat, run by the last integrator block of each replica where thermo_cnt is
    // set (otherwise by thermostat_kernel after the integrators)
    int* thermo_cnt;              // [R] integrator blocks of the replica done this step (back to 0 after)
    const int* thermo_total;      // [R] its integrator blocks
    float* lambda_next;           // [R] the lambda array itself (the thermostat writes the next step's)
    float* lambda_applied;        // [R]
    double* temperature;          // [R]
    long long* step_count_w;      // [R] the step counters (the thermostat advances them)
    int thermo_mode;
    unsigned long long* kclock;   // [4] span of the step's all-pairs blocks and its running sum, or null
    float* log_data;              // [log_ring][10]
    float* train_data;            // [log_ring][compounds of log_rep][log_slots][3 x Float3], or null
    // energies: [R*kEnergyTerms]
    double* energy;
    uint32_t* err;                // [4]
    int enable_solvents, enable_dihedrals;
    int loc_nb, loc_na, loc_nd;   // most bonds, angles, dihedrals of any compound (local_role's LDS strides)
    int n_types;                  // atom types that any chain particle has, counted from type 0
    int local_stage;              // LDS bytes of one compound in local_role's wavefront form
    int listed_split;             // FP32: listed_role splits the rows of compounds of <= 32 particles over both halves of the wavefront
};

enum { kE_bond = 0, kE_angle, kE_dih, kE_intra, kE_inter, kE_cs, kE_sc, kE_ss, kE_virial, kE_kin, kEnergyTerms };

constexpr int kChunkParticles = 2048;   // chain particles staged per solvent<-chain work item
constexpr int kChunkCompounds = 64;

LIMA_DEV int ftype(float4 p) { return __float_as_int(p.w); }
// a stored solvent position: w is 0 inside the box, 1 outside (where no image rule holds)
__host__ LIMA_DEV float4 solvent_pos(float x, float y, float z, float L) {
    return make_float4(x, y, z, x >= 0.f && x <= L && y >= 0.f && y <= L && z >= 0.f && z <= L ? 0.f : 1.f);
}

// ===========================================================================
// One step is two launches on one stream.
//
//   step_forces_kernel     every force of the step: solvent lists, the compounds' local forces,
//                          bridges, the all-pairs solvent <- chain term and the listed compound term
//   step_integrate_kernel  the sums, integration, PBC and (optionally) the thermostat of every
//                          compound and solvent tile
//
// A launch holds blocks of several roles, chosen by the block index (ForceBlocks).  The roles of a
// launch do not depend on each other.  As separate kernels on four streams, the fork and the joins
// of a step cost about 30 us (a captured fork of four 10 us kernels, a join and a fifth take 52 us;
// two dependent kernels on one stream 22 us): more than the whole work of a small system's step.
// Blocks are dispatched in index order: first the bonded terms (latency-bound), then the all-pairs
// blocks, which fill the device, and the short listed items last, as its tail.  The solvent-list
// blocks, bound by their gathers, are spread over the launch in groups of eight, so that they share
// the CUs with the VALU-bound ones.  Every block has 256 threads; most roles work by wavefront and
// never meet a block barrier.
// ===========================================================================
constexpr int kStepThreads = 256;

// A launch of 2^32 threads or more in one dimension is refused (2^24 blocks of 256), which an all-pairs
// list of a million solvents and as many particles, or its list build, reaches: blocks beyond kGridWidth
// take a second dimension.  Whole rows, so the last one's rest have no work; widths are multiples of 8,
// which keeps a block's XCD that of its number.
constexpr long long kGridWidth = 1 << 14;
inline dim3 grid_of(long long blocks) {
    const long long rows = std::max<long long>(1, (blocks + kGridWidth - 1) / kGridWidth);
    return dim3(rows == 1 ? (unsigned)blocks : (unsigned)(((blocks + rows - 1) / rows + 7) / 8 * 8), (unsigned)rows);
}

LIMA_DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

LIMA_DEV void wave_atomic_energy(double v, double* dst) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0 && v != 0.0) atomicAdd(dst, v);
}

// ---------------------------------------------------------------------------
// compoundBridgeKernel (Engine.cu:1168-1223): bonded terms spanning two compounds
// (CompoundBridgeCompact, Bodies.cuh:644-700), at most 32 particles each
// (MAX_PARTICLES_IN_BRIDGE, Constants.cuh:110), one wavefront per bridge.  The bridge's
// particles are gathered into LDS and re-imaged against its first particle; the lanes
// evaluate up to kBridgeChunk terms of one kind at a time, and lane k then adds the
// results for particle k in term order (bonds, then angles, then dihedrals, each kind
// summed separately), the order of a serial pass over the terms, so the carry-in forces
// are the serial ones bit for bit.  They are stored (not added) into fbridge.
// ---------------------------------------------------------------------------
constexpr int kBridgeParticles = 32;
constexpr int kBridgeChunk = 64;
static_assert(kMaxTypes * kMaxTypes % kStepThreads == 0, "staging loops stride by the block size");

struct BridgeStage {
    double en[kBridgeChunk];
    F3 pos[kBridgeParticles];
    F3 res[kBridgeChunk * 4];
    int who[kBridgeChunk * 4];
};

template <bool ENERGY> LIMA_DEV void bridge_role(const StepArgs& a, int b, BridgeStage& st) {
    if (b >= a.n_bridges) return;
    const int lane = threadIdx.x & 63;
    const ReplicaInfo rp = a.reps[a.br_rep[b]];
    const int p0 = a.br_off[b], np = min(a.br_off[b + 1] - p0, kBridgeParticles);
    const int tb = a.brb_off[b], nb = a.brb_off[b + 1] - tb;
    const int ta = a.bra_off[b], na = a.bra_off[b + 1] - ta;
    const int td = a.brd_off[b], nd = a.enable_dihedrals ? a.brd_off[b + 1] - td : 0;
    // each kind's first chunk of term records is loaded together with the positions
    const BondD bd0 = lane < nb ? a.brb[tb + lane] : BondD{};
    const AngleD ad0 = lane < na ? a.bra[ta + lane] : AngleD{};
    const DihD dd0 = lane < nd ? a.brd[td + lane] : DihD{};
    F3 me = f3(0.f, 0.f, 0.f);
    if (lane < np) {
        const float4 q = a.cpos[a.br_glob[p0 + lane]];
        me = f3(q.x, q.y, q.z);
        st.pos[lane] = me;
    }
    wave_sync();
    if (lane > 0 && lane < np) {
        const F3 ref = st.pos[0];
        hyperpos(ref.x, ref.y, ref.z, me.x, me.y, me.z, make_box(rp.L, rp.half));
        st.pos[lane] = me;
    }
    wave_sync();
    F3 ps = f3(0.f, 0.f, 0.f), as = ps, ds = ps;
    double eb = 0, ea = 0, ed = 0;
    // one kind of term: compute a chunk into LDS, then each particle's lane adds its slots in order
    auto sweep = [&](int nterms, int slots, auto&& eval, F3& acc, double& esum) {
        for (int c0 = 0; c0 < nterms; c0 += kBridgeChunk) {
            const int nt = min(kBridgeChunk, nterms - c0);
            if (lane < nt) {
                double e = 0;
                eval(c0, &st.res[lane * 4], &st.who[lane * 4], &e);
                st.en[lane] = e;
            }
            wave_sync();
            if (lane < np)
                for (int t = 0; t < nt; t++)
                    for (int k = 0; k < slots; k++)
                        if (st.who[t * 4 + k] == lane) acc = f3_add(acc, st.res[t * 4 + k]);
            if (ENERGY && lane == 0)
                for (int t = 0; t < nt; t++) esum += st.en[t];
            wave_sync();
        }
    };
    const F3* pos = st.pos;
    sweep(nb, 2, [&](int c0, F3* r, int* w, double* e) {
        const BondD bd = c0 == 0 ? bd0 : a.brb[tb + c0 + lane];
        pairbond(pos[bd.a0], pos[bd.a1], bd.b0, bd.kb, r, e);
        w[0] = bd.a0; w[1] = bd.a1;
    }, ps, eb);
    sweep(na, 3, [&](int c0, F3* r, int* w, double* e) {
        const AngleD ad = c0 == 0 ? ad0 : a.bra[ta + c0 + lane];
        anglebond(pos[ad.a0], pos[ad.a1], pos[ad.a2], ad.t0, ad.k, r, e);
        w[0] = ad.a0; w[1] = ad.a1; w[2] = ad.a2;
    }, as, ea);
    sweep(nd, 4, [&](int c0, F3* r, int* w, double* e) {
        const DihD dd = c0 == 0 ? dd0 : a.brd[td + c0 + lane];
        dihedral(pos[dd.a0], pos[dd.a1], pos[dd.a2], pos[dd.a3], dd.p0, dd.k, dd.n, r, e);
        w[0] = dd.a0; w[1] = dd.a1; w[2] = dd.a2; w[3] = dd.a3;
    }, ds, ed);
    if (lane < np) {
        const F3 f = f3_add(f3_add(f3_add(f3(0.f, 0.f, 0.f), ps), as), ds);
        a.fbridge[a.br_glob[p0 + lane]] = make_float4(f.x, f.y, f.z, 0.0f);
    }
    if (ENERGY && lane == 0) {
        double* e = a.energy + a.br_rep[b] * kEnergyTerms;
        atomicAdd(e + kE_bond, eb);
        atomicAdd(e + kE_angle, ea);
        atomicAdd(e + kE_dih, ed);
    }
}

// ---------------------------------------------------------------------------
// compoundKernel's local forces (Engine.cu:918-937, 678-700): bonded terms (term forces
// computed once, then gathered per particle in term index order = the serialized scatter's
// order, Engine.cu:765-771) and the intra-compound LJ (geometric eps, exclusions), summed in
// that order; the integrator adds the bridge carry-in and the listed partials.  int64 sums in
// the fixed-point form.
//
// THREADS 256: one block per compound; the dihedrals run on its first two wavefronts and the
// bonds and angles on the other two, at the same time.  THREADS 64: one wavefront per compound,
// where every compound of the engine fits one.  Latency-bound: a few dependent loads, then one
// term of each kind a thread.
// ---------------------------------------------------------------------------
template <int THREADS> constexpr int local_particles() { return THREADS == 64 ? 64 : kCompoundBlock; }
template <int THREADS>
inline size_t local_lds_bytes(int nb, int na, int nd) {
    return ((size_t)local_particles<THREADS>() * sizeof(float4) +
            (THREADS == 64 ? 0 : (size_t)kMaxTypes * kMaxTypes * sizeof(float2)) +
            (size_t)(2 * nb + 3 * na + 4 * nd) * sizeof(F3) + 15) / 16 * 16;
}

template <bool FIXED, bool ENERGY, int THREADS>
LIMA_DEV void local_role(const StepArgs& a, int c, char* lds) {
    constexpr int P = local_particles<THREADS>();
    constexpr bool WAVE = THREADS == 64;
    if (c >= a.n_comp) return;
    const int p = WAVE ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
    auto sync = [] {
        if (WAVE) wave_sync();
        else __syncthreads();
    };
    float4* pos = reinterpret_cast<float4*>(lds);
    float2* tab = reinterpret_cast<float2*>(pos + P);
    F3* rb = reinterpret_cast<F3*>(WAVE ? reinterpret_cast<char*>(tab) : reinterpret_cast<char*>(tab + kMaxTypes * kMaxTypes));
    F3* ra = rb + 2 * a.loc_nb;
    F3* rd = ra + 3 * a.loc_na;
    const int r = a.comp_rep[c];
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
    const bool active = p < n;
    const int gi = base + (active ? p : 0);
    float4 me = a.cpos[gi];
    const float4 p0 = a.cpos[base];
    hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, box);                     // Engine.cu:923
    if (p < P) pos[p] = me;
    const float2* gtab = a.tab_intra_ab + (size_t)r * kMaxTypes * kMaxTypes;
    if (!WAVE) {
        // a compile-time stride, so that the loads of a lane are in flight together
        float2 v[kMaxTypes * kMaxTypes / kStepThreads];
#pragma unroll
        for (int u = 0; u < kMaxTypes * kMaxTypes / kStepThreads; u++) v[u] = gtab[p + u * kStepThreads];
#pragma unroll
        for (int u = 0; u < kMaxTypes * kMaxTypes / kStepThreads; u++) tab[p + u * kStepThreads] = v[u];
    }
    sync();
    double eb = 0, ea = 0, ed = 0;
    // Energies of the terms that thread 0 of the reference's 128 evaluates, for its potE slot of the
    // log: every 128th term, whatever this form's stride.  The thread of term 0 has them all.
    double slot_b = 0, slot_a = 0, slot_d = 0;
    auto count = [](double& sum, double& slot, int t, double e) {
        sum += e;
        slot += t % kCompoundBlock == 0 ? e : 0.0;
    };
    const int b0 = a.bond_off[c], nb = a.bond_off[c + 1] - b0;
    const int a0 = a.angle_off[c], na = a.angle_off[c + 1] - a0;
    const int d0 = a.dih_off[c], nd = a.dih_off[c + 1] - d0;
    auto P3 = [&](int i) { float4 q = pos[i]; return f3(q.x, q.y, q.z); };
    if (WAVE || p >= P) {
        for (int t = WAVE ? p : p - P; t < nb; t += P) {
            BondD bd = a.bonds[b0 + t];
            double e = 0;
            pairbond(P3(bd.a0), P3(bd.a1), bd.b0, bd.kb, &rb[t * 2], &e);
            count(eb, slot_b, t, e);
        }
        for (int t = WAVE ? p : p - P; t < na; t += P) {
            AngleD ad = a.angles[a0 + t];
            double e = 0;
            anglebond(P3(ad.a0), P3(ad.a1), P3(ad.a2), ad.t0, ad.k, &ra[t * 3], &e);
            count(ea, slot_a, t, e);
        }
    }
    if (a.enable_dihedrals && p < P) {
        for (int t = p; t < nd; t += P) {
            DihD dd = a.dihs[d0 + t];
            double e = 0;
            dihedral(P3(dd.a0), P3(dd.a1), P3(dd.a2), P3(dd.a3), dd.p0, dd.k, dd.n, &rd[t * 4], &e);
            count(ed, slot_d, t, e);
        }
    }
    sync();
    F3 bs = f3(0.f, 0.f, 0.f), as = bs, ds = bs;
    if (active) {
        for (int e = a.inc_off[gi]; e < a.inc_off[gi + 1]; e++) {
            const uint32_t v = a.inc[e];
            const uint32_t kind = v >> 30, slot = v & 3u, term = (v >> 2) & 0xFFFFFFFu;
            if (kind == 0) bs = f3_add(bs, rb[term * 2 + slot]);
            else if (kind == 1) as = f3_add(as, ra[term * 3 + slot]);
            else ds = f3_add(ds, rd[term * 4 + slot]);
        }
    }
    F3 force = f3(0.f, 0.f, 0.f);
    long long fx_i = 0, fy_i = 0, fz_i = 0;
    uint32_t bad = 0;
    if (FIXED) {
        fx_i = to_fixed(bs.x, bad) + to_fixed(as.x, bad) + (a.enable_dihedrals ? to_fixed(ds.x, bad) : 0);
        fy_i = to_fixed(bs.y, bad) + to_fixed(as.y, bad) + (a.enable_dihedrals ? to_fixed(ds.y, bad) : 0);
        fz_i = to_fixed(bs.z, bad) + to_fixed(as.z, bad) + (a.enable_dihedrals ? to_fixed(ds.z, bad) : 0);
    } else {
        force = f3_add(bs, as);
        if (a.enable_dihedrals) force = f3_add(force, ds);
    }
    // computeIntramolecularLJForces (Engine.cu:678-700)
    float lx = 0.f, ly = 0.f, lz = 0.f;
    double e_intra = 0, vir = 0;
    if (active) {
        const int tp = ftype(me);
        const uint32_t* mk = a.intra_mask + (size_t)gi * 4;
        const uint32_t m[4] = {mk[0], mk[1], mk[2], mk[3]};
#pragma unroll
        for (int g = 0; g < P / 32; g++) {
            const int jend = min(n, g * 32 + 32);
#pragma unroll 4
            for (int j = g * 32; j < jend; j++) {
                const float4 q = pos[j];
                const float2 pr = WAVE ? gtab[ftype(q) * kMaxTypes + tp] : tab[ftype(q) * kMaxTypes + tp];
                float dx = q.x - me.x, dy = q.y - me.y, dz = q.z - me.z;
                float r2 = pair_r2(dx, dy, dz);
                float inv;
                float fs = lj_scalar(r2, pr.x, pr.y, inv);
                const bool ex = (j == p) || ((m[g] >> (j & 31)) & 1u);
                fs = ex ? 0.0f : fs;
                pair_add(dx, dy, dz, fs, lx, ly, lz);
                if (ENERGY && !ex) {
                    e_intra += lj_energy(inv, pr.x, pr.y);
                    pair_virial(r2, fs, vir);
                }
            }
        }
    }
    if (FIXED) {
        fx_i += to_fixed(lx, bad); fy_i += to_fixed(ly, bad); fz_i += to_fixed(lz, bad);
        if (bad) atomicOr(a.err, bad);
    } else force = f3_add(force, f3(lx, ly, lz));
    if (active) {
        if (FIXED) a.cloc_fx[gi] = I3{fx_i, fy_i, fz_i};
        else a.cloc[gi] = make_float4(force.x, force.y, force.z, 0.f);
    }
    // thread 0's potE slot of the logged replica's first compound (Engine.cu:1027): the dihedral
    // assigns it (Engine.cu:612), else its bond and angle terms (which thread P evaluates here)
    if (a.log_rep == r && c == rp.comp_begin) {
        float* o = a.log_data + (size_t)(a.step_count[r] % a.log_ring) * 10;
        const bool by_dihedral = a.enable_dihedrals && nd > 0;
        if (by_dihedral && p == 0) o[2] = (float)slot_d;
        if (!by_dihedral && p == (WAVE ? 0 : P)) o[2] = (float)(slot_b + slot_a);
    }
    if (ENERGY) {
        double* e = a.energy + r * kEnergyTerms;
        wave_atomic_energy(eb, e + kE_bond);
        wave_atomic_energy(ea, e + kE_angle);
        wave_atomic_energy(ed, e + kE_dih);
        wave_atomic_energy(e_intra, e + kE_intra);
        wave_atomic_energy(vir, e + kE_virial);
    }
}

// ---------------------------------------------------------------------------
// The solvent's own position is re-imaged against each compound's particle 0 in
// compound order before its LJ sums (Engine.cu:1111).  replay_images continues
// that sequence over compounds [cb, ce) for the solvent of each lane, from
// particle-0 positions staged in LDS; every thread of the block calls it.
// ---------------------------------------------------------------------------
constexpr int kReplayStage = 256;

template <typename F> LIMA_DEV void each_particle0(const StepArgs& a, int cb, int ce, float4* p0s, F&& f) {
    for (int c0 = cb; c0 < ce; c0 += kReplayStage) {
        const int nc = min(kReplayStage, ce - c0);
        __syncthreads();
        for (int i = threadIdx.x; i < nc; i += blockDim.x) p0s[i] = a.cpos[a.comp_off[c0 + i]];
        __syncthreads();
        for (int i = 0; i < nc; i++) f(p0s[i]);
    }
}
LIMA_DEV void replay_images(const StepArgs& a, int cb, int ce, float4* p0s, float& sx, float& sy, float& sz, const Box& box) {
    each_particle0(a, cb, ce, p0s, [&](const float4& q) { hyperpos(q.x, q.y, q.z, sx, sy, sz, box); });
}

// ---------------------------------------------------------------------------
// solventForceKernel's compound loop (Engine.cu:1099-1117): every solvent
// against every chain particle of its replica, no cutoff.  Work item =
// (solvent tile, compound chunk).  The chunk's particles are staged in LDS as
// rows (x, y, z, A) + B (the pair constants of lj_ab), each compound padded to a multiple of
// kRowPad rows (comp_row, row_src; padding rows have zero constants), so the pair loop has no
// remainder; every lane holds one solvent.  Per-compound partial sums match computeLJForces' local sum (Engine.cu:640-651).
//
// The solvent's image next to each compound's particle 0 is taken from its stored position.  The
// reference carries the image from compound to compound (Engine.cu:1111).  With the solvent and
// every particle 0 inside the box both are the image nearest to particle 0 (a carried image lies
// within [-L/2, 3L/2], one shift from it), and the direct one is rounded once instead of once a
// shift.  Where the two are exactly half a box apart both images are as near and the carried one
// depends on the compounds before: there, and for a whole block where a solvent or a particle 0 lies
// outside (positions as a caller first set them), the sequence is replayed from the first compound.
// The replay had cost 7% of the kernel on the production system's 100 compounds and 14% on the 18 nm
// box's 400; the test for a tie costs the demo's step (compounds of 30 to 43 particles) 1%, larger
// compounds' less.
//
// Bound: VALU issue, 14 instructions a pair at the full rate (2.3 cycles) and a reciprocal (12-16
// cycles among FMAs): 50 cycles a pair of 64 lanes measured with one solvent a lane, 51-54 with
// two, 59 with four.  Subtractions moved to the matrix cores (exact bfloat16 pieces) cost the same
// issue time, one reciprocal shared by two or four pairs saves 1-2% and loses accuracy.
// ---------------------------------------------------------------------------
constexpr int kRowPad = 4;
constexpr float kFarAway = 1e18f;   // outside any box; r^2 = 3e36 is finite, its reciprocal's square is zero
constexpr int kAllPairsHead = 528;   // the constants and row offsets before the tile, 16-byte aligned
static_assert(kMaxTypes * 8 + (kChunkCompounds + 1) * 4 <= kAllPairsHead && kAllPairsHead % 16 == 0, "head of the tile");
inline size_t all_pairs_lds_bytes(int rows) {
    const size_t tile = (size_t)rows * (sizeof(float4) + sizeof(float));
    return kAllPairsHead + (tile > kReplayStage * sizeof(float4) ? tile : kReplayStage * sizeof(float4));
}
LIMA_DEV bool in_box(float4 p, float L) {
    return p.x >= 0.f && p.x <= L && p.y >= 0.f && p.y <= L && p.z >= 0.f && p.z <= L;
}

// In-step timing of all_pairs_role, on the device's constant-rate clock (wall_clock64):
// kclock[0] = the earliest start of the first kClockHead blocks (dispatched first, one per
// XCD), kclock[1] = the latest end of any block (work items differ in length, so any block
// may be the last); the step's thermostat kernel, which runs after it on the same stream,
// adds the span to kclock[2] and counts it in kclock[3], then clears kclock[0..1].  A clock
// read stalls its wave, so the start is read by the first blocks only.
constexpr int kClockHead = 8;

template <bool FIXED, bool ENERGY> LIMA_DEV void all_pairs_role(const StepArgs& a, int item, char* lds) {
    // [kMaxTypes] float2 constants, [kChunkCompounds + 1] row offsets, [cap] float4 + [cap] float rows
    float2* tab = reinterpret_cast<float2*>(lds);
    int* tile_off = reinterpret_cast<int*>(tab + kMaxTypes);
    float4* tile = reinterpret_cast<float4*>(lds + kAllPairsHead);
    float* tile_b = reinterpret_cast<float*>(tile + a.chunk_cap);
    const int tid = threadIdx.x;
    if (a.kclock && tid == 0 && item < kClockHead) atomicMin(&a.kclock[0], (unsigned long long)wall_clock64());
    const SCWork wk = a.scwork[item];
    const ReplicaInfo rp = a.reps[wk.replica];
    const float L = rp.L;
    const Box box = make_box(L, rp.half);
    if (tid < kMaxTypes) {
        const float4 v = a.tab_sc[wk.replica * kMaxTypes + tid];
        tab[tid] = lj_ab(v.x, v.y);
    }
    const int c0 = wk.comp_begin, ncomp = wk.comp_end - wk.comp_begin;
    const int base = a.comp_row[c0], total = a.comp_row[wk.comp_end] - base;
    for (int k = tid; k <= ncomp; k += kStepThreads) tile_off[k] = a.comp_row[c0 + k] - base;
    const int s = wk.solv_begin + tid;
    const bool active = s < wk.solv_end;
    const float4 me = a.spos[active ? s : wk.solv_begin];
    float rx = me.x, ry = me.y, rz = me.z;
    bool inside = in_box(me, L);
    for (int c = rp.comp_begin + tid; c < wk.comp_end; c += kStepThreads) inside = inside && in_box(a.cpos[a.comp_off[c]], L);
    const bool direct = __syncthreads_and(inside) != 0;   // also: tab and tile_off are written
    if (!direct) {   // the reference's sequential re-imaging over the compounds before the chunk
        replay_images(a, rp.comp_begin, c0, tile, rx, ry, rz, box);
        __syncthreads();
    }
    for (int k = tid; k < total; k += kStepThreads) {
        const int src = a.row_src[base + k];
        float4 p = make_float4(kFarAway, kFarAway, kFarAway, 0.f);   // padding: zero constants, at a distance that is not zero
        float2 ab = make_float2(0.f, 0.f);
        if (src >= 0) {
            p = a.cpos[src];
            ab = tab[ftype(p)];
        }
        tile[k] = make_float4(p.x, p.y, p.z, ab.x);
        tile_b[k] = ab.y;
    }
    __syncthreads();
    float fx = 0.f, fy = 0.f, fz = 0.f;
    long long ix = 0, iy = 0, iz = 0;
    double en = 0.0, vir = 0.0;
    for (int ci = 0; ci < ncomp; ci++) {
        const int j0 = tile_off[ci], j1 = tile_off[ci + 1];
        const float4 q0 = tile[j0];
        float sx = rx, sy = ry, sz = rz, lx = 0.f, ly = 0.f, lz = 0.f;
        hyperpos(q0.x, q0.y, q0.z, sx, sy, sz, box);
        if (!direct) {
            rx = sx; ry = sy; rz = sz;
        } else if (__ballot(half_a_box(fsub(q0.x, rx), fsub(q0.y, ry), fsub(q0.z, rz), rp.half)) != 0ull) {
            // A tie (one or two a step of production's 7 million): the image carried from the last
            // compound before that ties with none of these solvents, where it is the nearest again.
            int c = c0 + ci - 1;
            for (; c >= rp.comp_begin; c--) {
                const float4 q = a.cpos[a.comp_off[c]];
                if (__ballot(half_a_box(fsub(q.x, rx), fsub(q.y, ry), fsub(q.z, rz), rp.half)) == 0ull) break;
            }
            float cx = rx, cy = ry, cz = rz;
            for (c = max(c, rp.comp_begin); c <= c0 + ci; c++) {
                const float4 q = a.cpos[a.comp_off[c]];
                hyperpos(q.x, q.y, q.z, cx, cy, cz, box);
            }
            if (fabsf(fsub(q0.x, rx)) == rp.half) sx = cx;
            if (fabsf(fsub(q0.y, ry)) == rp.half) sy = cy;
            if (fabsf(fsub(q0.z, rz)) == rp.half) sz = cz;
        }
        for (int j = j0; j < j1; j += kRowPad) {
            float4 q[kRowPad];
#pragma unroll
            for (int u = 0; u < kRowPad; u++) q[u] = tile[j + u];
            const float4 b4 = *reinterpret_cast<const float4*>(tile_b + j);
#pragma unroll
            for (int u = 0; u < kRowPad; u++) {
                const float b = u == 0 ? b4.x : u == 1 ? b4.y : u == 2 ? b4.z : b4.w;
                if (ENERGY) lj_acc_energy(sx, sy, sz, q[u].x, q[u].y, q[u].z, q[u].w, b, lx, ly, lz, en, vir);
                else lj_acc(sx, sy, sz, q[u].x, q[u].y, q[u].z, q[u].w, b, lx, ly, lz);
            }
        }
        if (FIXED) {
            uint32_t bad = 0;
            ix += to_fixed(lx, bad); iy += to_fixed(ly, bad); iz += to_fixed(lz, bad);
            if (bad) atomicOr(a.err, bad);
        } else { fx += lx; fy += ly; fz += lz; }
    }
    if (active) {
        const size_t slot = (size_t)wk.chunk * a.n_solv + s;
        if (FIXED) a.partS_fx[slot] = I3{ix, iy, iz};
        else a.partS[slot] = make_float4(fx, fy, fz, 0.f);
    }
    if (ENERGY) {
        wave_atomic_energy(active ? en : 0.0, a.energy + wk.replica * kEnergyTerms + kE_sc);
        wave_atomic_energy(active ? vir : 0.0, a.energy + wk.replica * kEnergyTerms + kE_virial);
    }
    if (a.kclock) {
        __syncthreads();   // every wave of the block is done
        if (tid == 0) atomicMax(&a.kclock[1], (unsigned long long)wall_clock64());
    }
}

// ---------------------------------------------------------------------------
// compoundKernel's listed LJ (Engine.cu:939-974): work item = (compound,
// source chunk); sources are one neighbour compound (arithmetic eps, LJ
// exclusions) or 256 entries of the compound's solvent list (geometric eps).
// Sources are re-imaged against the compound's particle 0 (Engine.cu:949, 967).
// An item's sum for a target is that of its parts, each in list order, added in order, and goes to
// the item's slot.  A system of few items and with a compound of more than 32 particles
// (ReplicaInfo::listed_split) has an item of more than 32 sources in four parts, so that four
// wavefronts can share it; others have one part, which saves them the parts' ends (18 nm: 373 us
// alone in four parts, 355 in one; 256 replicas 332 and 312).  Each lane holds
// one target particle, or two (lane, lane + 64) for compounds of more than 64, so that a row is read
// from LDS once for two pairs.
//   WIDE false: a wavefront per item.  WIDE true: a block per item and a wavefront per part, for
// engines with few items (ForceBlocks::listed_wide); the sums are the same.
// A wavefront reads only the LDS rows that it staged.  Rows are padded to a multiple of 4 with
// positions whose force is exactly zero (r^-8 underflows).  The type table of the block's first item
// is staged in LDS; an item of another system reads its constants from the global table.  With
// a.listed_split (FP32, an autotuner choice, WIDE false) a compound of at most 32 particles has each
// half of the wavefront sum one half of the rows, the halves added in order.
// ---------------------------------------------------------------------------
constexpr int kListedParts = 4;
// rows of a part of an item of `nsrc` sources: a quarter, in whole fours, or all of them
LIMA_DEV int listed_part(int nsrc, int split) { return nsrc <= 32 || !split ? (nsrc + 3) & ~3 : ((nsrc + 15) >> 4) * 4; }

constexpr size_t kListedLds = (size_t)kMaxTypes * kMaxTypes * sizeof(float2) + 4 * kSolventChunk * sizeof(float4);
static_assert(kListedParts == kStepThreads / 64 && kSolventChunk + kListedParts * kCompoundBlock <= 4 * kSolventChunk,
              "a wavefront per part; the rows and the parts' sums of the wide form");

template <bool FIXED, bool ENERGY, bool WIDE>
LIMA_DEV void listed_role(const StepArgs& a, int blk, int nblk, char* lds) {
    float2* tab = reinterpret_cast<float2*>(lds);   // (A, B) of lj_ab: 8-byte entries keep the per-lane reads conflict-light
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float4* src = reinterpret_cast<float4*>(tab + kMaxTypes * kMaxTypes) + (WIDE ? 0 : wid * kSolventChunk);
    float4* part_sums = src + kSolventChunk;   // WIDE: [kListedParts][kCompoundBlock]
    constexpr int PER = WIDE ? 1 : 4;
    const int total = *a.cw_total;
    int cached_rep = -1;
    for (int w0 = blk * PER; w0 < total; w0 += nblk * PER) {
        const bool valid = WIDE || w0 + wid < total;
        const int w = WIDE ? w0 : valid ? w0 + wid : w0;
        const int c = a.item_comp[w], r = a.comp_rep[c], r0 = a.comp_rep[a.item_comp[w0]];
        if (r0 != cached_rep) {   // the same for the whole block
            float2 v[kMaxTypes * kMaxTypes / kStepThreads];
#pragma unroll
            for (int u = 0; u < kMaxTypes * kMaxTypes / kStepThreads; u++)
                v[u] = a.tab_inter_ab[(size_t)r0 * kMaxTypes * kMaxTypes + threadIdx.x + u * kStepThreads];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kMaxTypes * kMaxTypes / kStepThreads; u++) tab[threadIdx.x + u * kStepThreads] = v[u];
            __syncthreads();
            cached_rep = r0;
        }
        if (!valid) continue;
        const int k = w - a.cw_off[c];
        const ReplicaInfo rp = a.reps[r];
        const Box box = make_box(rp.L, rp.half);
        const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
        const float4 p0 = a.cpos[base];
        const bool split = !WIDE && !FIXED && a.listed_split && n <= 32;
        const int h = split ? lane >> 5 : 0;
        float mx[2], my[2], mz[2];
        int tp[2], gi[2];
        bool active[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int pi = split ? lane & 31 : lane + 64 * q;
            active[q] = pi < n && !(split && q);
            gi[q] = base + (active[q] ? pi : 0);
            float4 me = a.cpos[gi[q]];
            hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, box);                     // Engine.cu:923
            mx[q] = me.x; my[q] = me.y; mz[q] = me.z;
            tp[q] = ftype(me);
        }
        const int ncc = a.cc_cnt[c];
        const bool is_cc = k < ncc;
        float lx[2] = {0.f, 0.f}, ly[2] = {0.f, 0.f}, lz[2] = {0.f, 0.f};
        double en = 0.0, vir = 0.0;
        int nsrc;
        uint32_t m[2][4] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
        wave_sync();   // the wavefront is done with the previous item's rows
        // the rows that this wavefront stages and sums
        int part = 0, row_lo = 0, row_hi = 0;
        auto rows_of = [&]() {
            part = listed_part(nsrc, rp.listed_split);
            row_lo = WIDE ? wid * part : 0;
            row_hi = WIDE ? min(row_lo + part, (nsrc + 3) & ~3) : kSolventChunk;
        };
        if (is_cc) {
            const int nb = a.cc_ids[(size_t)c * a.cap_cc + k];
            const int nbase = a.comp_off[nb];
            nsrc = a.comp_off[nb + 1] - nbase;
            rows_of();
#pragma unroll
            for (int u = 0; u < (WIDE ? 1 : kCompoundBlock / 64); u++) {
                const int jj = row_lo + lane + 64 * u;
                if (jj >= row_hi) continue;
                float4 q = make_float4(kFarAway, kFarAway, kFarAway, 0.f);
                if (jj < nsrc) {
                    q = a.cpos[nbase + jj];
                    hyperpos(p0.x, p0.y, p0.z, q.x, q.y, q.z, box);                // Engine.cu:949
                    q.w = __int_as_float(ftype(q) * (int)(kMaxTypes * sizeof(float2)));   // byte offset of the type's table row
                }
                src[jj] = q;
            }
            // LJ_Ignores of the targets against the neighbour (Engine.cu:660)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                if (!active[t]) continue;
                for (int e = a.xoff[gi[t]]; e < a.xoff[gi[t] + 1]; e++) {
                    const int2 x = a.xent[e];
                    if (x.x == nb) {
                        const uint32_t bit = 1u << (x.y & 31);
                        const int ws = x.y >> 5;
                        m[t][0] |= ws == 0 ? bit : 0u; m[t][1] |= ws == 1 ? bit : 0u;
                        m[t][2] |= ws == 2 ? bit : 0u; m[t][3] |= ws == 3 ? bit : 0u;
                    }
                }
            }
        } else {
            const int j0 = (k - ncc) * kSolventChunk;
            nsrc = min(kSolventChunk, a.cs_cnt[c] - j0);
            rows_of();
            const int* ids = a.cs_ids + (size_t)c * a.cap_cs + j0;
#pragma unroll
            for (int u = 0; u < (WIDE ? 1 : kSolventChunk / 64); u++) {
                const int jj = row_lo + lane + 64 * u;
                if (jj >= row_hi) continue;
                float4 q = make_float4(kFarAway, kFarAway, kFarAway, 0.f);
                if (jj < nsrc) {
                    q = a.spos[ids[jj]];
                    hyperpos(p0.x, p0.y, p0.z, q.x, q.y, q.z, box);                // Engine.cu:967
                }
                src[jj] = q;
            }
        }
        wave_sync();
        const int rows = (nsrc + 3) & ~3;
        const int half_rows = (rows / 2 + 3) & ~3;
        const char* gtab = reinterpret_cast<const char*>(a.tab_inter_ab + (size_t)r * kMaxTypes * kMaxTypes);
        auto pair = [&](const float4& q, float2 pr, bool ex, int t) {
            const float dx = q.x - mx[t], dy = q.y - my[t], dz = q.z - mz[t];
            const float r2 = pair_r2(dx, dy, dz);
            float inv;
            float fs = lj_scalar(r2, pr.x, pr.y, inv);
            fs = ex ? 0.0f : fs;
            pair_add(dx, dy, dz, fs, lx[t], ly[t], lz[t]);
            if (ENERGY && active[t] && !ex) {
                en += lj_energy(inv, pr.x, pr.y);
                pair_virial(r2, fs, vir);
            }
        };
        // KIND 0: solvents (each target's own constants); 1: neighbour compound, table in LDS.  NQ targets a lane
        auto sums = [&](auto kind_tag, auto nq_tag, int lo, int hi) {
            constexpr int KIND = decltype(kind_tag)::value, NQ = decltype(nq_tag)::value;
            const char* trow[NQ];
            float2 own[NQ];
#pragma unroll
            for (int t = 0; t < NQ; t++) {
                trow[t] = reinterpret_cast<const char*>(tab + tp[t]);
                own[t] = make_float2(0.f, 0.f);
                if (KIND == 0) {
                    const float4 pv = a.tab_cs[r * kMaxTypes + tp[t]];
                    own[t] = lj_ab(pv.x, pv.y);
                }
            }
            for (int j = lo; j < hi; j += 4) {
                float4 q[4];
#pragma unroll
                for (int u = 0; u < 4; u++) q[u] = src[j + u];
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int t = 0; t < NQ; t++)
                        pair(q[u], KIND == 1 ? *reinterpret_cast<const float2*>(trow[t] + ftype(q[u])) : own[t], false, t);
            }
        };
        constexpr std::integral_constant<int, 0> solvents{};
        constexpr std::integral_constant<int, 1> one{};
        constexpr std::integral_constant<int, 2> two{};
        const bool clean = !is_cc || (__ballot((m[0][0] | m[0][1] | m[0][2] | m[0][3] | m[1][0] | m[1][1] | m[1][2] | m[1][3]) != 0u) == 0ull && r == r0);
        // rows [lo, hi) (the same for the wavefront unless it splits)
        auto run = [&](int lo, int hi) {
            if (!is_cc) {
                if (n > 64) sums(solvents, two, lo, hi);
                else sums(solvents, one, lo, hi);
            } else if (clean) {
                if (n > 64) sums(one, two, lo, hi);
                else sums(one, one, lo, hi);
            } else {
                // a bridged neighbour (exclusions exist only between bridged compounds), or another system's table
#pragma unroll
                for (int g = 0; g < kCompoundBlock / 32; g++)
                    for (int j = max(lo, 32 * g); j < min(hi, 32 * g + 32); j++) {
                        const float4 q = src[j];
#pragma unroll
                        for (int t = 0; t < 2; t++)
                            pair(q, *reinterpret_cast<const float2*>(gtab + ftype(q) + tp[t] * (int)sizeof(float2)),
                                 ((m[t][g] >> (j & 31)) & 1u) != 0u, t);
                    }
            }
        };
        if (split) {
            run(h * half_rows, min(rows, (h + 1) * half_rows));
        } else if (WIDE) {
            run(row_lo, row_hi);
        } else {
            float sx[2] = {0.f, 0.f}, sy[2] = {0.f, 0.f}, sz[2] = {0.f, 0.f};
            for (int lo = 0; lo < rows; lo += part) {
                run(lo, min(lo + part, rows));
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    sx[t] += lx[t]; sy[t] += ly[t]; sz[t] += lz[t];
                    lx[t] = ly[t] = lz[t] = 0.f;
                }
            }
#pragma unroll
            for (int t = 0; t < 2; t++) { lx[t] = sx[t]; ly[t] = sy[t]; lz[t] = sz[t]; }
        }
        if (split) {
            lx[0] += __shfl_down(lx[0], 32, 64); ly[0] += __shfl_down(ly[0], 32, 64); lz[0] += __shfl_down(lz[0], 32, 64);
        }
        auto store = [&](int p, float x, float y, float z) {
            const size_t slot = (size_t)w * kCompoundBlock + p;
            if (FIXED) {
                uint32_t bad = 0;
                a.partC_fx[slot] = I3{to_fixed(x, bad), to_fixed(y, bad), to_fixed(z, bad)};
                if (bad) atomicOr(a.err, bad);
            } else a.partC[slot] = make_float4(x, y, z, 0.f);
        };
        if (WIDE) {
#pragma unroll
            for (int t = 0; t < 2; t++) part_sums[wid * kCompoundBlock + lane + 64 * t] = make_float4(lx[t], ly[t], lz[t], 0.f);
            __syncthreads();
            const int p = threadIdx.x;
            if (p < n) {
                float4 v = part_sums[p];
                for (int q = 1; q * part < rows; q++) {
                    const float4 o = part_sums[q * kCompoundBlock + p];
                    v.x += o.x; v.y += o.y; v.z += o.z;
                }
                store(p, v.x, v.y, v.z);
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++)
                if (active[t] && !h) store(lane + 64 * t, lx[t], ly[t], lz[t]);
        }
        if (ENERGY) {
            wave_atomic_energy(en, a.energy + r * kEnergyTerms + (is_cc ? kE_inter : kE_cs));
            wave_atomic_energy(vir, a.energy + r * kEnergyTerms + kE_virial);
        }
    }
}

// ---------------------------------------------------------------------------
// listed_role for engines whose compounds all hold at most 16 * PPL particles
// (PPL 1, 2 or 4 particles per lane).  A wavefront is four groups of 16 lanes and
// takes four runs at once, one per group.  A run is either one solvent-chunk work item (its
// 256 sources staged and summed in two halves of 128), or up to cc_run(PPL) = 8 / PPL
// consecutive neighbour-compound items of one compound (at most 128 sources, staged together).
// Lane pi of a group holds particles pi, pi + 16, ... of the run's compound and sums each
// item's sources in list order, in the parts that listed_role sums them in, into the item's
// own partial slot: the sums are the same.  A group reads only
// its own LDS row, so wavefront-level ordering is the only synchronisation.  Groups may belong
// to different replicas: the inter-compound pair constants come from a table of the used types in
// LDS when every group is of the system of the block's first run, else from the global table
// tab_inter_ab (whose gathers, two a row from up to four lines a group, kept L1 busier than the VALU).
// ---------------------------------------------------------------------------
constexpr int kPackLanes = 16;
constexpr int kPackGroups = 64 / kPackLanes;
constexpr int kPackRow = 128;                 // staged sources per group
__host__ __device__ constexpr int cc_run(int ppl) { return kPackRow / (kPackLanes * ppl); }

template <int W> LIMA_DEV double group_sum(double v) {
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <int PPL> struct PackedStage {   // one wavefront's LDS
    // rows padded by one entry: the four groups' rows start in different LDS banks
    float4 src[kPackGroups][kPackRow + 1];
    int run_nb[kPackGroups][cc_run(PPL)], run_off[kPackGroups][cc_run(PPL) + 1];
};

template <bool FIXED, bool ENERGY, int PPL>
LIMA_DEV void listed_packed_role(const StepArgs& a, int blk, int nblk, char* lds) {
    static_assert(PPL == 1 || PPL == 2 || PPL == 4, "16, 32 or 64 particles per compound");
    constexpr int RUN = cc_run(PPL);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float2* ltab = reinterpret_cast<float2*>(lds + 4 * sizeof(PackedStage<PPL>));   // [n_types][n_types]
    PackedStage<PPL>& st = reinterpret_cast<PackedStage<PPL>*>(lds)[wid];
    int table_rep = -1;
    auto& src = st.src;
    auto& run_nb = st.run_nb;
    auto& run_off = st.run_off;
    const int p = threadIdx.x & 63, g = p / kPackLanes, pi = p % kPackLanes;
    float4* sg = src[g];
    const int n_ccr = a.run_total[0], total = n_ccr + a.run_total[1];
    for (int sb = blk * 4 * kPackGroups; sb < total; sb += nblk * 4 * kPackGroups) {
        const int r0 = sb < n_ccr ? a.comp_rep[a.run_comp[sb]] : table_rep;
        if (r0 != table_rep) {   // the same for the whole block
            __syncthreads();
            for (int e = threadIdx.x; e < a.n_types * a.n_types; e += kStepThreads)
                ltab[e] = a.tab_inter_ab[(size_t)r0 * kMaxTypes * kMaxTypes + e / a.n_types * kMaxTypes + e % a.n_types];
            __syncthreads();
            table_rep = r0;
        }
        const int s0 = sb + wid * kPackGroups;
        if (s0 >= total) continue;
        const int sr = s0 + g;
        const bool valid = sr < total;
        const int si = valid ? sr : s0;
        const int c = a.run_comp[si];
        const bool is_cc = si < n_ccr;
        const int ncc = a.cc_cnt[c];
        const int r = a.comp_rep[c];
        const ReplicaInfo rp = a.reps[r];
        const Box box = make_box(rp.L, rp.half);
        const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
        const float4 p0 = a.cpos[base];
        float mx[PPL], my[PPL], mz[PPL];
        int tp[PPL], xb[PPL], xe[PPL];
        bool act[PPL];
#pragma unroll
        for (int q = 0; q < PPL; q++) {
            const int pidx = pi + kPackLanes * q;
            act[q] = valid && pidx < n;
            const int gi = base + (act[q] ? pidx : 0);
            float4 me = a.cpos[gi];
            hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, box);                 // Engine.cu:923
            mx[q] = me.x; my[q] = me.y; mz[q] = me.z;
            tp[q] = ftype(me);
            xb[q] = act[q] ? a.xoff[gi] : 0;
            xe[q] = act[q] ? a.xoff[gi + 1] : 0;
        }
        // the run's items: neighbour items w_first .. w_first + nitems - 1, or one solvent chunk
        const int k0 = is_cc ? (si - a.run_off[c]) * RUN : ncc + (si - n_ccr - a.run_cs_off[c]);
        const int nitems = is_cc ? min(RUN, ncc - k0) : 1;
        const int w_first = a.cw_off[c] + k0;
        double en = 0.0, vir = 0.0;
        auto store = [&](int w, int q, float lx, float ly, float lz) {
            const size_t slot = (size_t)w * kCompoundBlock + pi + kPackLanes * q;
            if (FIXED) {
                uint32_t bad = 0;
                a.partC_fx[slot] = I3{to_fixed(lx, bad), to_fixed(ly, bad), to_fixed(lz, bad)};
                if (bad) atomicOr(a.err, bad);
            } else a.partC[slot] = make_float4(lx, ly, lz, 0.f);
        };
        // The pair loops, for the first NQ particle slots of each lane: when every group of the
        // wavefront holds a compound of at most 16 particles the second slot is idle, and the
        // loops skip it (a wavefront-uniform choice; the active slots' sums are unchanged)
        // LT: the groups' pair constants come from the table in LDS
        auto pairs = [&](auto nq_tag, auto lt_tag) {
        constexpr int NQ = decltype(nq_tag)::value;
        constexpr bool LT = decltype(lt_tag)::value;
        const int row = LT ? a.n_types : kMaxTypes;
        wave_sync();   // every group of the wavefront is done with the previous round's rows
        if (valid && is_cc) {
            // the run's neighbour compounds, re-imaged against this compound's particle 0 (Engine.cu:949)
            if (pi < nitems) {
                const int nb = a.cc_ids[(size_t)c * a.cap_cc + k0 + pi];
                run_nb[g][pi] = nb;
                run_off[g][pi + 1] = a.comp_off[nb + 1] - a.comp_off[nb];
            }
            wave_sync();
            if (pi == 0) {
                run_off[g][0] = 0;
                for (int t = 0; t < nitems; t++) run_off[g][t + 1] += run_off[g][t];
            }
            wave_sync();
            for (int t = 0; t < nitems; t++) {
                const int nbase = a.comp_off[run_nb[g][t]], o = run_off[g][t], nn = run_off[g][t + 1] - o;
                for (int j = pi; j < nn; j += kPackLanes) {
                    float4 qv = a.cpos[nbase + j];
                    hyperpos(p0.x, p0.y, p0.z, qv.x, qv.y, qv.z, box);
                    qv.w = __int_as_float(ftype(qv) * row);   // the type's table row
                    sg[o + j] = qv;
                }
            }
            wave_sync();
            const float2* gtab = a.tab_inter_ab + (size_t)r * kMaxTypes * kMaxTypes;
            for (int t = 0; t < nitems; t++) {
                const int nb = run_nb[g][t], j0 = run_off[g][t], j1 = run_off[g][t + 1];
                // LJ_Ignores of each particle against this neighbour (Engine.cu:660); only
                // particles at a bridged junction have entries
                uint32_t m0[PPL], m1[PPL];
                bool clean = true;
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    m0[q] = m1[q] = 0u;
                    for (int e = xb[q]; e < xe[q]; e++) {
                        const int2 x = a.xent[e];
                        if (x.x == nb) {
                            const uint32_t bit = 1u << (x.y & 31);
                            m0[q] |= x.y < 32 ? bit : 0u;
                            m1[q] |= x.y >= 32 ? bit : 0u;
                        }
                    }
                    clean = clean && (m0[q] | m1[q]) == 0u;
                }
                float lx[PPL], ly[PPL], lz[PPL], tx[PPL], ty[PPL], tz[PPL];
#pragma unroll
                for (int q = 0; q < NQ; q++) tx[q] = ty[q] = tz[q] = 0.f;
                const int part = PPL <= 2 ? j1 - j0 : listed_part(j1 - j0, rp.listed_split);
                for (int p0 = j0; p0 < j1; p0 += part) {
                const int p1 = min(p0 + part, j1);
#pragma unroll
                for (int q = 0; q < NQ; q++) lx[q] = ly[q] = lz[q] = 0.f;
                if (clean) {
#pragma unroll 2
                    for (int j = p0; j < p1; j++) {
                        const float4 qv = sg[j];
                        const int ts = ftype(qv);
#pragma unroll
                        for (int q = 0; q < NQ; q++) {
                            const float2 pr = LT ? ltab[ts + tp[q]] : gtab[ts + tp[q]];
                            const float dx = qv.x - mx[q], dy = qv.y - my[q], dz = qv.z - mz[q];
                            const float r2 = pair_r2(dx, dy, dz);
                            float inv;
                            const float fs = lj_scalar(r2, pr.x, pr.y, inv);
                            pair_add(dx, dy, dz, fs, lx[q], ly[q], lz[q]);
                            if (ENERGY && act[q]) {
                                en += lj_energy(inv, pr.x, pr.y);
                                pair_virial(r2, fs, vir);
                            }
                        }
                    }
                } else {
                    for (int j = p0; j < p1; j++) {
                        const float4 qv = sg[j];
                        const int ts = ftype(qv), jl = j - j0;
#pragma unroll
                        for (int q = 0; q < NQ; q++) {
                            const float2 pr = LT ? ltab[ts + tp[q]] : gtab[ts + tp[q]];
                            const float dx = qv.x - mx[q], dy = qv.y - my[q], dz = qv.z - mz[q];
                            const float r2 = pair_r2(dx, dy, dz);
                            float inv;
                            float fs = lj_scalar(r2, pr.x, pr.y, inv);
                            const bool ex = (((jl < 32 ? m0[q] : m1[q]) >> (jl & 31)) & 1u) != 0u;
                            fs = ex ? 0.0f : fs;
                            pair_add(dx, dy, dz, fs, lx[q], ly[q], lz[q]);
                            if (ENERGY && act[q] && !ex) {
                                en += lj_energy(inv, pr.x, pr.y);
                                pair_virial(r2, fs, vir);
                            }
                        }
                    }
                }
#pragma unroll
                for (int q = 0; q < NQ; q++) { tx[q] += lx[q]; ty[q] += ly[q]; tz[q] += lz[q]; }
                }
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    if (act[q]) store(w_first + t, q, tx[q], ty[q], tz[q]);
            }
        } else if (valid) {
            // 256 entries of the compound's solvent list (Engine.cu:967), staged in two halves
            const int j0 = (k0 - ncc) * kSolventChunk;
            const int nsrc = min(kSolventChunk, a.cs_cnt[c] - j0);
            const int* ids = a.cs_ids + (size_t)c * a.cap_cs + j0;
            float2 pr_cs[PPL];
#pragma unroll
            for (int q = 0; q < PPL; q++) {
                const float4 pv = a.tab_cs[r * kMaxTypes + tp[q]];
                pr_cs[q] = lj_ab(pv.x, pv.y);
            }
            float lx[PPL], ly[PPL], lz[PPL], tx[PPL], ty[PPL], tz[PPL];
#pragma unroll
            for (int q = 0; q < NQ; q++) lx[q] = ly[q] = lz[q] = tx[q] = ty[q] = tz[q] = 0.f;
            const int part = PPL <= 2 ? nsrc : listed_part(nsrc, rp.listed_split);
            int part_end = min(part, nsrc);
            for (int h0 = 0; h0 < nsrc; h0 += kPackRow) {
                const int hn = min(kPackRow, nsrc - h0);
                if (h0 > 0) wave_sync();   // the first half is summed before the row is rewritten
#pragma unroll
                for (int u = 0; u < kPackRow / kPackLanes; u++) {
                    const int jj = pi + u * kPackLanes;
                    if (jj < hn) {
                        float4 qv = a.spos[ids[h0 + jj]];
                        hyperpos(p0.x, p0.y, p0.z, qv.x, qv.y, qv.z, box);
                        sg[jj] = qv;
                    }
                }
                wave_sync();
                for (int b0 = 0; b0 < hn;) {
                const int b1 = PPL <= 2 ? hn : min(hn, part_end - h0);
#pragma unroll 2
                for (int j = b0; j < b1; j++) {
                    const float4 qv = sg[j];
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        if (ENERGY) {
                            double e0 = 0.0, w0 = 0.0;
                            lj_acc_energy(mx[q], my[q], mz[q], qv.x, qv.y, qv.z, pr_cs[q].x, pr_cs[q].y, lx[q], ly[q],
                                          lz[q], e0, w0);
                            if (act[q]) { en += e0; vir += w0; }
                        } else lj_acc(mx[q], my[q], mz[q], qv.x, qv.y, qv.z, pr_cs[q].x, pr_cs[q].y, lx[q], ly[q], lz[q]);
                    }
                }
                b0 = b1;
                if (PPL <= 2) continue;   // one part
                if (h0 + b1 == part_end) {   // the part's end (parts may run over the halves')
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        tx[q] += lx[q]; ty[q] += ly[q]; tz[q] += lz[q];
                        lx[q] = ly[q] = lz[q] = 0.f;
                    }
                    part_end = min(part_end + part, nsrc);
                }
                }
            }
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (act[q]) store(w_first, q, tx[q] + lx[q], ty[q] + ly[q], tz[q] + lz[q]);
        }
        };
        const bool lt = __ballot(valid && is_cc && r != table_rep) == 0ull;
        if (PPL > 1 && __ballot(valid && n > kPackLanes) == 0ull) {
            if (lt) pairs(std::integral_constant<int, 1>{}, std::true_type{});
            else pairs(std::integral_constant<int, 1>{}, std::false_type{});
        } else {
            if (lt) pairs(std::integral_constant<int, PPL>{}, std::true_type{});
            else pairs(std::integral_constant<int, PPL>{}, std::false_type{});
        }
        if (ENERGY) {
            en = group_sum<kPackLanes>(en);
            vir = group_sum<kPackLanes>(vir);
            if (valid && pi == 0) {
                if (en != 0.0) atomicAdd(a.energy + r * kEnergyTerms + (is_cc ? kE_inter : kE_cs), en);
                if (vir != 0.0) atomicAdd(a.energy + r * kEnergyTerms + kE_virial, vir);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// solventForceKernel's listed part (Engine.cu:1111, 1121-1123, 706-720): the
// solvent's own position is re-imaged against every compound's particle 0 in
// compound order, then against every listed neighbour in list order, as the
// reference mutates it; the solvent-solvent LJ local sum and the final self
// image are written for the integrator.
//
// With the solvent, its neighbours and every particle 0 inside the box, each image of the sequence
// is the one nearest to its entry: on each axis the stored coordinate, or that one moved by L
// towards the far side (up for a coordinate below L/2, down above it).  So an entry's separation is
// taken from the stored position, with one flag an axis, and the sequence's last image, bit for bit,
// from the last entry and from whether any flag was set: a coordinate once moved keeps the rounding
// of the move.  The particle 0s set one if the farthest of them on that side does.  Entries are then
// independent: a quad of lanes walks a row, lane x of it entries 4x .. 4x + 3 of every 16, and the
// four sums are added in a fixed order.  Where any position lies outside (a solvent's w, particle 0
// as a caller first set it), or an entry is exactly half a box away, where the sequence keeps the image
// that it has, the wavefront replays the sequence, with the same split of the sums.
//
// Bound by the gathers: an entry takes 24 full-rate instructions and a reciprocal, 70 cycles a
// wavefront, and 64 lines of L1.  The carried image had taken 32 and made a row one serial chain.
// Alone, us, before and now: t4 17.5 -> 8.7, small 15.7 -> 8.6, production (24,071 solvents) 43 ->
// 15, 18 nm (158,512) 105 -> 65, 256 replicas 379 -> 338.
// Tiles are taken in XCD-contiguous order (xcd_item), so the tiles of one replica share one L2.
// ---------------------------------------------------------------------------
constexpr int kListChunk = 16;                 // row length granule of the solvent lists
constexpr int kXcds = 8;

// Workgroups are dispatched round-robin over the XCDs (block b runs on XCD
// b % 8).  With the grid padded to a multiple of 8, XCD x takes the contiguous
// item range [x * per, (x + 1) * per).
LIMA_DEV int xcd_item(int b, int nblocks) {
    const int per = nblocks / kXcds;
    return (b % kXcds) * per + b / kXcds;
}
inline int xcd_grid(int n) { return (n + kXcds - 1) / kXcds * kXcds; }

constexpr int kQuadSolvents = kStepThreads / 4;   // solvents of a block

template <int CTRL> LIMA_DEV float quad_perm(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
// the quad's sum ((0 + 1) + (2 + 3)) in each of its lanes
LIMA_DEV float quad_sum(float v) {
    v += quad_perm<0xB1>(v);   // lanes 1, 0, 3, 2
    return v + quad_perm<0x4E>(v);   // lanes 2, 3, 0, 1
}
// One axis of a position inside the box: the side to which its other image lies.
struct Side {
    float step, shift;   // +-2^60, -+L
};
LIMA_DEV Side side_of(float m, float half, const Box& box) {
    const bool up = m < half;
    return {up ? box.step : -box.step, up ? -box.L : box.L};
}
// 1 if a separation d = q - m is beyond half a box, else 0 (above_half on that side alone)
LIMA_DEV float beyond(float d, const Side& sd, const Box& box) {
    return __builtin_amdgcn_fmed3f(__builtin_fmaf(d, sd.step, box.nstep), 0.f, 1.f);
}
// the last image of a coordinate m: `last` the last entry's coordinate, `ever` whether any moved it
LIMA_DEV float last_image(float m, float last, float ever, const Side& sd, const Box& box) {
    const float other = m - sd.shift;
    return ever == 0.f ? m : beyond(fsub(last, m), sd, box) != 0.f ? other : other + sd.shift;
}

// `rounds` of 64 solvents a block
template <bool ENERGY> LIMA_DEV void solvent_listed_role(const StepArgs& a, int item, int rounds) {
    const int per_tile = 256 / kQuadSolvents / rounds;
    constexpr int SEG = 16;   // entries of a row a quad takes at a time
    static_assert(kListChunk % SEG == 0, "segments tile the rows");
    const int4 tile = a.stiles[item / per_tile];
    const int lane = threadIdx.x & 63, ax = lane & 3;
    const int first = tile.y + (item % per_tile) * rounds * kQuadSolvents + (int)(threadIdx.x >> 6) * 16;   // the wavefront's
    if (first >= tile.z) return;
    const int r = tile.x;
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const float4 pv = a.tab_ss[r];
    float2 pss = lj_ab(pv.x, pv.y);
    asm("" : "+v"(pss.x), "+v"(pss.y));   // full rate, as the box's
    // Entries can be half a box away only where that is within the lists' radius and what solvents drift
    // between builds (a quarter of it); tested for everywhere, they cost the 256 replicas' step 1%.
    const bool near_ties = rp.half * rp.half < 1.5625f * rp.ss_bound;
    // the particle 0s: inside the box, and the farthest on either side of each axis
    float p0_outside = 0.f;
    const int last = rp.comp_end - 1;
    float lo[3], hi[3];
    if (last >= rp.comp_begin) {
        for (int c = rp.comp_begin + lane; c <= last || c < rp.comp_begin + 64; c += 64) {   // lanes past the end repeat the last
            const float4 q = a.cpos[a.comp_off[min(c, last)]];
            p0_outside += in_box(q, rp.L) ? 0.f : 1.f;
            const float v[3] = {q.x, q.y, q.z};
            const bool first_of = c < rp.comp_begin + 64;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                lo[k] = first_of ? v[k] : fminf(lo[k], v[k]);
                hi[k] = first_of ? v[k] : fmaxf(hi[k], v[k]);
            }
        }
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int k = 0; k < 3; k++) {
                lo[k] = fminf(lo[k], __shfl_xor(lo[k], off, 64));
                hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], off, 64));
            }
    }
    double en = 0.0, vir = 0.0;
    for (int round = 0; round < rounds; round++) {
        const int s0 = first + round * kQuadSolvents, s = s0 + (lane >> 2);
        if (s0 >= tile.z) break;
        const bool active = s < tile.z;
        const int si = active ? s : tile.y;
        const int cnt = active ? a.ss_cnt[si] : 0;
        const float4 me = a.spos[si];
        const int* row = a.ss_ids + (size_t)si * a.ss_ld;
        int wmax = cnt;
        for (int off = 32; off >= 4; off >>= 1) wmax = max(wmax, __shfl_xor(wmax, off, 64));
        float outside = p0_outside + me.w;
        const Side sdx = side_of(me.x, rp.half, box), sdy = side_of(me.y, rp.half, box), sdz = side_of(me.z, rp.half, box);
        auto farthest = [&](float m, int k, const Side& sd) {
            return last < rp.comp_begin ? 0.f : beyond(fsub(m < rp.half ? hi[k] : lo[k], m), sd, box);
        };
        float evx = farthest(me.x, 0, sdx), evy = farthest(me.y, 1, sdy), evz = farthest(me.z, 2, sdz);
        float lx = 0.f, ly = 0.f, lz = 0.f;
        bool tie = false;
        double e_round = 0.0, w_round = 0.0;
        // past the row's count a lane re-reads its entries of the first segment (in bounds, not used)
        // and its own position
        auto load_ids = [&](int k0) { return *reinterpret_cast<const int4*>(row + (k0 < cnt ? k0 : 0) + 4 * ax); };
        struct Four {
            float4 q[4];
        };
        auto gather = [&](int4 id, int k0) {
            const int n = cnt - k0 - 4 * ax;
            return Four{{a.spos[0 < n ? id.x : si], a.spos[1 < n ? id.y : si], a.spos[2 < n ? id.z : si], a.spos[3 < n ? id.w : si]}};
        };
        auto add = [&](float dx, float dy, float dz, bool take) {
            const float r2 = pair_r2(dx, dy, dz);
            float inv;
            float fs = lj_scalar(r2, pss.x, pss.y, inv);
            fs = take ? fs : 0.f;
            pair_add(dx, dy, dz, fs, lx, ly, lz);
            if (ENERGY) {
                const double e = lj_energy(inv, pss.x, pss.y);
                e_round += take ? e : 0.0;
                pair_virial(r2, fs, w_round);
            }
        };
        if (wmax > 0) {
            // a segment's positions are requested while the one before is summed, its ids another
            // segment earlier
            int4 ids = load_ids(SEG);
            Four cur = gather(load_ids(0), 0);
            for (int k0 = 0; k0 < wmax; k0 += SEG) {
                const Four nxt = gather(ids, k0 + SEG);
                ids = load_ids(k0 + 2 * SEG);
                __builtin_amdgcn_sched_barrier(0);
                const int n = cnt - k0 - 4 * ax;   // this lane's entries in the segment (may be <= 0)
                auto sums = [&](auto full_tag) {
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const float4 q = cur.q[u];
                        outside += q.w;
                        const float dx = fsub(q.x, me.x), dy = fsub(q.y, me.y), dz = fsub(q.z, me.z);
                        const float fx = beyond(dx, sdx, box), fy = beyond(dy, sdy, box), fz = beyond(dz, sdz, box);
                        evx += fx; evy += fy; evz += fz;
                        add(__builtin_fmaf(sdx.shift, fx, dx), __builtin_fmaf(sdy.shift, fy, dy), __builtin_fmaf(sdz.shift, fz, dz),
                            decltype(full_tag)::value || u < n);
                    }
                };
                if (__ballot(n < 4) == 0ull) sums(std::true_type{});
                else sums(std::false_type{});
                if (near_ties)
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        tie = tie | half_a_box(fsub(cur.q[u].x, me.x), fsub(cur.q[u].y, me.y), fsub(cur.q[u].z, me.z), rp.half);
                cur = nxt;
            }
        }
        float mx = me.x, my = me.y, mz = me.z;
        float4 end = me;   // the sequence's last entry
        if (cnt > 0) end = a.spos[row[cnt - 1]];
        else if (last >= rp.comp_begin) end = a.cpos[a.comp_off[last]];
        tie = tie | half_a_box(fsub(end.x, me.x), fsub(end.y, me.y), fsub(end.z, me.z), rp.half);
        if (__ballot(outside != 0.f || tie) == 0ull) {
            evx = quad_sum(evx);
            evy = quad_sum(evy);
            evz = quad_sum(evz);
            if (cnt > 0 || last >= rp.comp_begin) {
                mx = last_image(me.x, end.x, evx, sdx, box);
                my = last_image(me.y, end.y, evy, sdy, box);
                mz = last_image(me.z, end.z, evz, sdz, box);
            }
        } else {
            lx = ly = lz = 0.f;
            e_round = w_round = 0.0;
            for (int c = rp.comp_begin; c < rp.comp_end; c++) {
                const float4 q = a.cpos[a.comp_off[c]];
                hyperpos(q.x, q.y, q.z, mx, my, mz, box);
            }
            for (int k = 0; k < cnt; k++) {
                const float4 q = a.spos[row[k]];
                hyperpos(q.x, q.y, q.z, mx, my, mz, box);
                if (((k >> 2) & 3) == ax) add(q.x - mx, q.y - my, q.z - mz, true);
            }
        }
        lx = quad_sum(lx);
        ly = quad_sum(ly);
        lz = quad_sum(lz);
        if (active && ax == 0) a.ss_part[s] = make_float4(lx, ly, lz, 0.f);
        if (active && ax == 1) a.ss_img[s] = make_float4(mx, my, mz, 0.f);
        en += e_round;
        vir += w_round;
    }
    if (ENERGY) {
        wave_atomic_energy(en, a.energy + r * kEnergyTerms + kE_ss);
        wave_atomic_energy(vir, a.energy + r * kEnergyTerms + kE_virial);
    }
}

// ---------------------------------------------------------------------------
// Thermostat (Engine::handleBoxtemp, Engine.cu:362-393, made a device FP64
// reduction).  One wavefront per replica, fixed summation order.
//   mode 1 (Berendsen): T = sum m|dx|^2 / dt^2 / (3 N R) every step;
//     lambda = sqrt(1 + dt/tau (T0/T - 1)), clamped to [0.9, 1.1], T=0 guard.
//   mode 2 (the reference's cadence, Engine.cu:49-75, 314-393): after step k,
//     with s = k + 1 steps done, s % 40 == 0 evaluates T from the per-particle
//     FP32 kinetic energies of the positions two steps apart,
//     T = (float)(sum / N * 2 / (3 * 8.3145)), and, when s > 20, sets
//     lambda = clamp((float)T0 / T, 0.9, 1.1) for step s only; every other
//     step runs with lambda = 1.  step_count[r] counts the steps done.
// ---------------------------------------------------------------------------
constexpr int kThermostatEvery = 40;   // STEPS_PER_THERMOSTAT (Constants.cuh:82)

// One replica's thermostat by one wavefront (lane = its lane index).
LIMA_DEV void thermostat_replica(int r, const ReplicaInfo& rp, int lane, const double* ke_comp, const double* ke_stile,
                                 float* lambda, float* lambda_applied, double* temperature, long long* step_count,
                                 int mode, unsigned long long* kclock) {
    double s = 0.0;
    for (int c = rp.comp_begin + lane; c < rp.comp_end; c += 64) s += ke_comp[c];
    for (int t = rp.stile_begin + lane; t < rp.stile_end; t += 64) s += ke_stile[t];
    s = wave_sum(s);
    if (lane == 0) {
        lambda_applied[r] = lambda[r];
        const long long done = step_count[r] + 1;
        step_count[r] = done;
        if (kclock && r == 0) {   // this step's span of the all-pairs blocks
            const unsigned long long b = kclock[0], e = kclock[1];
            if (b != ~0ull && e > b) {
                kclock[2] += e - b;
                kclock[3] += 1;
            }
            kclock[0] = ~0ull;
            kclock[1] = 0ull;
        }
        const double ntot = (double)((rp.chain_end - rp.chain_begin) + (rp.solv_end - rp.solv_begin));
        float lam = 1.0f;
        if (mode == 2) {
            if (done % kThermostatEvery == 0) {
                const double avg = ntot > 0 ? s / ntot : 0.0;
                float temp = (float)(avg * 2.0f / (3.0f * 8.3145));
                temp = temp == 0.f ? 1.f : temp;
                temperature[r] = temp;
                float sc = rp.T0 / temp;
                sc = fminf(sc, 1.1f);
                sc = fmaxf(sc, 0.9f);
                if (done > 20) lam = sc;
            }
        } else {
            const double temp = ntot > 0 ? s / (rp.dt * rp.dt) / (3.0 * ntot * 8.3145) : 0.0;
            temperature[r] = temp;
            if (mode == 1) {
                double t = temp == 0.0 ? 1.0 : temp;
                double l = sqrt(1.0 + rp.dt / rp.tau * ((double)rp.T0 / t - 1.0));
                l = l < 1.1 ? l : 1.1;
                l = l > 0.9 ? l : 0.9;
                lam = (float)l;
            }
        }
        lambda[r] = lam;
    }
}

// ---------------------------------------------------------------------------
// The force launch.  PPL 0: listed_role, else listed_packed_role.  Four wavefronts a SIMD (128
// registers): the all-pairs role runs within 3% of its rate at eight with three.
// ---------------------------------------------------------------------------
struct ForceBlocks {
    int listed_solvents, local, bridges, all_pairs, listed;   // blocks of each role, in this order
    int thermostat;       // blocks of the step before's thermostat, first among the others
    int solvent_items, solvent_rounds;
    int local_waves;      // 1: one wavefront per compound
    int listed_wide;      // 1: a block per listed item
    int spread;           // groups of eight other blocks after each group of eight solvent-list blocks
    int mix;              // all-pairs blocks after each listed block; 0: all of them first
    int width;            // the grid's (grid_of)
};

template <bool FIXED, bool ENERGY, int PPL>
__global__ __launch_bounds__(kStepThreads, ENERGY ? 2 : 4) void step_forces_kernel(StepArgs a, ForceBlocks f) {
    extern __shared__ float4 dyn_lds[];
    char* lds = reinterpret_cast<char*>(dyn_lds);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int block = blockIdx.y * f.width + blockIdx.x;
    const int unit = block / kXcds, turn = unit / (f.spread + 1), lists = f.listed_solvents / kXcds;
    if (turn < lists && unit % (f.spread + 1) == 0) {
        const int item = xcd_item(turn * kXcds + block % kXcds, f.listed_solvents);
        if (item >= f.solvent_items) return;
        solvent_listed_role<ENERGY>(a, item, f.solvent_rounds);
        return;
    }
    int b = block - min(turn + 1, lists) * kXcds;   // among the other roles' blocks
    // Between the steps of a captured graph the thermostat of one runs beside the forces of the
    // next, which do not read what it writes (lambda, the counters): its own launch took 3.9 us of
    // a small system's 31 us step.
    if (b < f.thermostat) {
        const int r = 4 * b + wid;
        if (r < a.n_replicas)
            thermostat_replica(r, a.reps[r], threadIdx.x & 63, a.ke_comp, a.ke_stile, a.lambda_next, a.lambda_applied, a.temperature,
                               a.step_count_w, a.thermo_mode, nullptr);
        return;
    }
    b -= f.thermostat;
    if (b < f.local) {
        if (f.local_waves) local_role<FIXED, ENERGY, 64>(a, 4 * b + wid, lds + (size_t)wid * a.local_stage);
        else local_role<FIXED, ENERGY, kStepThreads>(a, b, lds);
        return;
    }
    b -= f.local;
    if (b < f.bridges) {
        bridge_role<ENERGY>(a, 4 * b + wid, reinterpret_cast<BridgeStage*>(lds)[wid]);
        return;
    }
    b -= f.bridges;
    // the all-pairs and listed blocks: one after the other, or (mix > 0, the packed form)
    // that many all-pairs blocks after each listed one
    int all_pairs = b, listed = b - f.all_pairs;
    if (f.mix > 0) {
        const int t = b / (f.mix + 1), rest = b % (f.mix + 1);
        const bool mixed = t < f.listed;
        all_pairs = mixed ? (rest ? b - t - 1 : f.all_pairs) : b - f.listed;
        listed = mixed && rest == 0 ? t : f.listed;
    }
    if (all_pairs < f.all_pairs) {
        all_pairs_role<FIXED, ENERGY>(a, all_pairs, lds);
        return;
    }
    if (listed >= f.listed) return;   // the launch is padded to whole groups of eight, and to whole rows
    if constexpr (PPL == 0) {
        if (f.listed_wide) listed_role<FIXED, ENERGY, true>(a, listed, f.listed, lds);
        else listed_role<FIXED, ENERGY, false>(a, listed, f.listed, lds);
    }
    else listed_packed_role<FIXED, ENERGY, PPL>(a, listed, f.listed, lds);
}

// lj_ab of every inter- or intra-compound table entry: the global copies
__global__ void ab_table_kernel(const float4* t, float2* ab, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) ab[i] = lj_ab(t[i].x, t[i].y);
}

// Triples of up to four float4 arrays, one after the other: array k takes triples end[k - 1] .. end[k].
struct IoArrays {
    float4* p[4];
    int end[4];
};
LIMA_DEV float4* io_element(const IoArrays& a, int i, int& k, int& e) {
    k = i < a.end[0] ? 0 : i < a.end[1] ? 1 : i < a.end[2] ? 2 : 3;
    e = i - (k == 0 ? 0 : k == 1 ? a.end[0] : k == 2 ? a.end[1] : a.end[2]);
    return (k == 0 ? a.p[0] : k == 1 ? a.p[1] : k == 2 ? a.p[2] : a.p[3]) + e;
}
__global__ __launch_bounds__(256) void io_pack_kernel(IoArrays a, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.end[3]) return;
    int k, e;
    const float4 v = *io_element(a, i, k, e);
    float* o = out + 3 * (size_t)i;
    o[0] = v.x; o[1] = v.y; o[2] = v.z;
}
__global__ __launch_bounds__(256) void io_unpack_kernel(IoArrays a, const float* in, const ReplicaInfo* reps, const int* solv_rep) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.end[3]) return;
    int k, e;
    float4* v = io_element(a, i, k, e);
    const float* q = in + 3 * (size_t)i;
    *v = k == 0 ? make_float4(q[0], q[1], q[2], v->w) : k == 2 ? solvent_pos(q[0], q[1], q[2], reps[solv_rep[e]].L)
                                                               : make_float4(q[0], q[1], q[2], 0.f);
}

// New parameters of one system, written where the kernels read them.  The values travel as kernel
// arguments and the tables are mixed here, so an update is one launch in stream order: as five
// copies, two launches and three synchronisations it took 140 us, 9 ms for a batch of 64 systems.
// The mixing is the host's fill_tables, rounded alike.
struct SystemParams {
    float sigma[kMaxTypes], eps[kMaxTypes];
    float bonded[2][2];    // force constant and equilibrium value of every pair bond, every angle
    int write[2];          // whether they change
    int bond0, bond1, angle0, angle1, brb0, brb1, bra0, bra1;   // the system's terms
};
LIMA_DEV float4 pair_table_entry(float sigma, float eps) {
    const float e24 = fmul(24.f, eps);
    return make_float4(fmul(sigma, sigma), e24, -2.0f * e24, sigma);
}
__global__ __launch_bounds__(kMaxTypes * kMaxTypes) void set_parameters_kernel(SystemParams p, int r, float4* tab_sc, float4* tab_cs,
                                                                              float4* tab_ss, float4* tab_inter, float4* tab_intra,
                                                                              float2* inter_ab, float2* intra_ab, BondD* bonds,
                                                                              AngleD* angles, BondD* brb, AngleD* bra) {
    const int i = threadIdx.x, t = i / kMaxTypes, u = i % kMaxTypes;
    const size_t e = (size_t)r * kMaxTypes * kMaxTypes + i;
    const float sigma = fmul(fadd(p.sigma[t], p.sigma[u]), 0.5f);
    const float ea = fmul(fadd(p.eps[t], p.eps[u]), 0.5f), eg = sqrtf(fmul(p.eps[t], p.eps[u]));
    const float4 inter = pair_table_entry(sigma, ea), intra = pair_table_entry(sigma, eg);
    tab_inter[e] = inter;
    tab_intra[e] = intra;
    inter_ab[e] = lj_ab(inter.x, inter.y);
    intra_ab[e] = lj_ab(intra.x, intra.y);
    if (t == 0) {
        tab_sc[r * kMaxTypes + u] = inter;
        tab_cs[r * kMaxTypes + u] = intra;
    }
    if (i == 0) tab_ss[r] = pair_table_entry(p.sigma[0], p.eps[0]);
    const auto bond = [&](BondD* b, int k0, int k1) {
        for (int k = k0 + i; k < k1; k += kMaxTypes * kMaxTypes) { b[k].kb = p.bonded[0][0]; b[k].b0 = p.bonded[0][1]; }
    };
    const auto angle = [&](AngleD* a, int k0, int k1) {
        for (int k = k0 + i; k < k1; k += kMaxTypes * kMaxTypes) { a[k].k = p.bonded[1][0]; a[k].t0 = p.bonded[1][1]; }
    };
    if (p.write[0]) { bond(bonds, p.bond0, p.bond1); bond(brb, p.brb0, p.brb1); }
    if (p.write[1]) { angle(angles, p.angle0, p.angle1); angle(bra, p.bra0, p.bra1); }
}

__global__ __launch_bounds__(64) void thermostat_kernel(const ReplicaInfo* reps, int n_rep, const double* ke_comp,
                                                      const double* ke_stile, float* lambda, float* lambda_applied,
                                                      double* temperature, long long* step_count, int mode,
                                                      unsigned long long* kclock) {
    const int r = blockIdx.x;
    if (r >= n_rep) return;
    thermostat_replica(r, reps[r], threadIdx.x, ke_comp, ke_stile, lambda, lambda_applied, temperature, step_count, mode,
                       kclock);
}

// The thermostat at the end of an integrator block: the replica's last block to finish runs
// it (a count per replica, no waiting), so no separate launch follows the integrators.  A block of
// solvents counts once, a block of two compounds once for each (`sub`, its half of the threads).
// The release fence orders the block's kinetic-energy partials before its counts; the last block's
// acquire fence makes every partial of the replica visible.  The sums are thermostat_kernel's.
// Every thread of the block calls it.
LIMA_DEV void thermostat_if_last(const StepArgs& a, int r, bool counts, int sub) {
    if (!a.thermo_cnt) return;
    __shared__ int last[2];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if ((threadIdx.x & 127) == 0) last[sub] = counts && atomicAdd(a.thermo_cnt + r, 1) == a.thermo_total[r] - 1;
    __syncthreads();
    if (last[sub]) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if ((threadIdx.x & 127) < 64)
            thermostat_replica(r, a.reps[r], threadIdx.x & 63, a.ke_comp, a.ke_stile, a.lambda_next, a.lambda_applied,
                               a.temperature, a.step_count_w, a.thermo_mode, a.kclock);
        if ((threadIdx.x & 127) == 0) a.thermo_cnt[r] = 0;
    }
}

// ---------------------------------------------------------------------------
// The integrate launch.
//
// Compounds (compoundKernel's remainder, Engine.cu:939-1056), two a block: the bridge carry-in,
// the local sum and the listed partials in list order, integration, PBC.  Solvent tiles
// (solventForceKernel's remainder, Engine.cu:1129-1155): force = compound contributions (chunk
// partials in order) + the solvent-solvent local sum; integrate, PBC, NaN check; tiles never
// straddle replicas.  ADVANCE=false computes forces (and the kinetic energy) without changing the
// state.  Bound by the partials' bytes on large systems, by the chain of loads on small ones.
// ---------------------------------------------------------------------------
template <bool ADVANCE, bool FIXED, bool ENERGY, int SLOTS> LIMA_DEV void compound_integrate_role(const StepArgs& a, int pair) {
    __shared__ float4 first[2];     // each compound's particle 0 after its step
    __shared__ double red[4];
    const int sub = threadIdx.x >> 7, p = threadIdx.x & 127;   // two compounds a block, 128 threads each
    const bool valid = 2 * pair + sub < a.n_comp;
    const int c = valid ? 2 * pair + sub : 2 * pair;
    const int r = a.comp_rep[c];
    const ReplicaInfo rp = a.reps[r];
    const float L = rp.L;
    const Box box = make_box(rp.L, rp.half);
    const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
    const bool active = valid && p < n;
    const int gi = base + (active ? p : 0);
    float4 me = a.cpos[gi];
    const float4 p0 = a.cpos[base];
    hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, box);                 // Engine.cu:923
    F3 force = f3(0.f, 0.f, 0.f);
    long long fx_i = 0, fy_i = 0, fz_i = 0;
    if (active) {
        const float4 fb = a.fbridge[gi];                                    // Engine.cu:918
        if (FIXED) {
            const I3 v = a.cloc_fx[gi];
            uint32_t bad = 0;
            fx_i = v.x + to_fixed(fb.x, bad); fy_i = v.y + to_fixed(fb.y, bad); fz_i = v.z + to_fixed(fb.z, bad);
            if (bad) atomicOr(a.err, bad);
        } else {
            const float4 v = a.cloc[gi];
            force = f3(fadd(fb.x, v.x), fadd(fb.y, v.y), fadd(fb.z, v.z));
        }
    }
    // listed partials: neighbour compounds (list order), then solvent chunks
    const bool logged = ADVANCE && valid && a.log_rep == r;
    F3 f_sol = f3(-1.f, -1.f, -1.f);   // computeSolventToCompoundLJForces' result, Float3(-1) when unset (Engine.cu:919)
    if (active) {
        const int s0 = a.cw_off[c], s1 = a.cw_off[c + 1];
        // SLOTS slots' loads in flight at once, then added in slot order
        for (int s = s0; s < s1; s += SLOTS) {
            if (FIXED) {
                I3 v[SLOTS];
#pragma unroll
                for (int u = 0; u < SLOTS; u++) v[u] = s + u < s1 ? a.partC_fx[(size_t)(s + u) * kCompoundBlock + p] : I3{0, 0, 0};
#pragma unroll
                for (int u = 0; u < SLOTS; u++) { fx_i += v[u].x; fy_i += v[u].y; fz_i += v[u].z; }
            } else {
                float4 v[SLOTS];
#pragma unroll
                for (int u = 0; u < SLOTS; u++)
                    v[u] = s + u < s1 ? a.partC[(size_t)(s + u) * kCompoundBlock + p] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int u = 0; u < SLOTS; u++)
                    if (s + u < s1) { force.x += v[u].x; force.y += v[u].y; force.z += v[u].z; }
            }
        }
        if (logged && a.enable_solvents) {
            long long sx_i = 0, sy_i = 0, sz_i = 0;
            float gx = 0.f, gy = 0.f, gz = 0.f;
            for (int s = s0 + a.cc_cnt[c]; s < s1; s++) {
                const size_t slot = (size_t)s * kCompoundBlock + p;
                if (FIXED) { I3 v = a.partC_fx[slot]; sx_i += v.x; sy_i += v.y; sz_i += v.z; }
                else { float4 v = a.partC[slot]; gx += v.x; gy += v.y; gz += v.z; }
            }
            f_sol = FIXED ? f3(from_fixed(sx_i), from_fixed(sy_i), from_fixed(sz_i)) : f3(gx, gy, gz);
        }
    }
    if (FIXED) force = f3(from_fixed(fx_i), from_fixed(fy_i), from_fixed(fz_i));
    if (active) a.cforce[gi] = make_float4(force.x, force.y, force.z, 0.f);
    if (active && exact_len(force.x, force.y, force.z) > 2e12f) atomicOr(a.err, kErrCriticalForce);   // Engine.cu:1050
    double ke = 0.0, kt = 0.0;   // one-step m|dx|^2; what the thermostat sums
    const double m = (double)a.mass[r * kMaxTypes + ftype(me)];
    float4 pv = a.cprev[gi];
    if (ADVANCE) {
        float px = me.x, py = me.y, pz = me.z, qx = pv.x, qy = pv.y, qz = pv.z, dx, dy, dz;
        const double mts = rp.dt / m * rp.dt;
        integrate(px, py, pz, qx, qy, qz, force.x, force.y, force.z, mts, a.lambda[r], box, dx, dy, dz);
        if (active) {
            a.cprev[gi] = make_float4(qx, qy, qz, 0.f);
            ke = m * ((double)dx * dx + (double)dy * dy + (double)dz * dz);
        }
        if (p == 0) first[sub] = make_float4(px, py, pz, me.w);
        __syncthreads();
        // PBC on particle 0, then re-image every particle against it (Engine.cu:993-996)
        const float4 z = first[sub];
        float zx = pbc1(z.x, L), zy = pbc1(z.y, L), zz = pbc1(z.z, L);
        hyperpos(zx, zy, zz, px, py, pz, box);
        if (active) a.cpos_next[gi] = make_float4(px, py, pz, me.w);
        if (logged) {
            const long long k = a.step_count[r];
            const int ring = (int)(k % a.log_ring);
            const int cl = c - rp.comp_begin;
            if (a.train_data && p < a.log_slots) {
                // data_GAN (Engine.cu:1036-1043): position, solvent LJ force, and a third Float3 left zero
                float* t = a.train_data + (((size_t)ring * (rp.comp_end - rp.comp_begin) + cl) * a.log_slots + p) * 9;
                const bool in = p < n;
                t[0] = in ? px : -1.f; t[1] = in ? py : -1.f; t[2] = in ? pz : -1.f;
                t[3] = f_sol.x; t[4] = f_sol.y; t[5] = f_sol.z;
                t[6] = 0.f; t[7] = 0.f; t[8] = 0.f;
            }
            if (cl == 0 && p == 0) {
                // outdata of compound 0, particle 0 (Engine.cu:1019-1028): speed, kinetic energy of the
                // one-step-apart positions, |F| (thread 0's potE slot comes from local_role)
                float bx = qx, by = qy, bz = qz;
                hyperpos(px, py, pz, bx, by, bz, box);
                float* o = a.log_data + (size_t)ring * 10;
                o[0] = (float)((double)exact_len(fsub(px, bx), fsub(py, by), fsub(pz, bz)) / rp.dt);
                o[1] = ref_kinetic(px, py, pz, bx, by, bz, m, rp.dt, box);
                o[3] = exact_len(force.x, force.y, force.z);
                for (int j = 4; j < 10; j++) o[j] = 0.f;
            }
        }
        // the logged position of this step against the one two steps back (Engine.cu:333-337)
        kt = !active ? 0.0 : a.ke_ref ? (double)ref_kinetic(px, py, pz, pv.x, pv.y, pv.z, m, rp.dt, box) : ke;
    } else if (active) {
        float qx = pv.x, qy = pv.y, qz = pv.z;
        hyperpos(me.x, me.y, me.z, qx, qy, qz, box);
        float dx = me.x - qx, dy = me.y - qy, dz = me.z - qz;
        ke = m * ((double)dx * dx + (double)dy * dy + (double)dz * dz);
    }
    // kinetic-energy partials of this compound (FP64, fixed order)
    if (ADVANCE) {
        const double ks = wave_sum(kt);
        if ((p & 63) == 0) red[threadIdx.x >> 6] = ks;
        __syncthreads();
        if (p == 0 && valid) a.ke_comp[c] = red[2 * sub] + red[2 * sub + 1];
        thermostat_if_last(a, r, valid, sub);
    }
    if (ENERGY) wave_atomic_energy(active ? ke : 0.0, a.energy + r * kEnergyTerms + kE_kin);
}

template <bool ADVANCE, bool FIXED, bool ENERGY> LIMA_DEV void solvent_integrate_role(const StepArgs& a, int tile_index) {
    __shared__ double red[4];
    const int4 tile = a.stiles[tile_index];
    const int r = tile.x;
    const ReplicaInfo rp = a.reps[r];
    const float L = rp.L;
    const Box box = make_box(rp.L, rp.half);
    const int s = tile.y + threadIdx.x;
    const bool active = s < tile.z;
    const int si = active ? s : tile.y;
    const float4 me = a.spos[si];
    const float4 img = a.ss_img[si];
    float sx = img.x, sy = img.y, sz = img.z;
    float fx = 0.f, fy = 0.f, fz = 0.f;
    long long ix = 0, iy = 0, iz = 0;
    // eight chunks' loads in flight at once, then added in chunk order
    for (int k = 0; k < rp.chunk_count; k += 8) {
        if (FIXED) {
            I3 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = k + u < rp.chunk_count ? a.partS_fx[(size_t)(k + u) * a.n_solv + si] : I3{0, 0, 0};
#pragma unroll
            for (int u = 0; u < 8; u++) { ix += v[u].x; iy += v[u].y; iz += v[u].z; }
        } else {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++)
                v[u] = k + u < rp.chunk_count ? a.partS[(size_t)(k + u) * a.n_solv + si] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (k + u < rp.chunk_count) { fx += v[u].x; fy += v[u].y; fz += v[u].z; }
        }
    }
    const float4 l = a.ss_part[si];
    if (FIXED) {
        uint32_t bad = 0;
        ix += to_fixed(l.x, bad); iy += to_fixed(l.y, bad); iz += to_fixed(l.z, bad);
        if (bad) atomicOr(a.err, bad);
        fx = from_fixed(ix); fy = from_fixed(iy); fz = from_fixed(iz);
    } else {
        fx += l.x; fy += l.y; fz += l.z;
    }
    if (active) a.sforce[s] = make_float4(fx, fy, fz, 0.f);
    const double m = (double)a.mass[r * kMaxTypes + 0];
    double ke = 0.0, kt = 0.0;   // one-step m|dx|^2; what the thermostat sums
    float4 pv = a.sprev[si];
    if (ADVANCE) {
        float qx = pv.x, qy = pv.y, qz = pv.z, dx, dy, dz;
        const double mts = rp.dt / m * rp.dt;
        integrate(sx, sy, sz, qx, qy, qz, fx, fy, fz, mts, a.lambda[r], box, dx, dy, dz);
        sx = pbc1(sx, L); sy = pbc1(sy, L); sz = pbc1(sz, L);
        if (active) {
            if (sx != sx) atomicOr(a.err, kErrNaN);                        // Engine.cu:1151
            a.spos_next[s] = solvent_pos(sx, sy, sz, L);
            a.sprev[s] = make_float4(qx, qy, qz, 0.f);
            ke = m * ((double)dx * dx + (double)dy * dy + (double)dz * dz);
            // the logged position of this step against the one two steps back (Engine.cu:347-351)
            kt = a.ke_ref ? (double)ref_kinetic(sx, sy, sz, pv.x, pv.y, pv.z, m, rp.dt, box) : ke;
        }
    } else if (active) {
        float qx = pv.x, qy = pv.y, qz = pv.z;
        hyperpos(me.x, me.y, me.z, qx, qy, qz, box);
        float dx = me.x - qx, dy = me.y - qy, dz = me.z - qz;
        ke = m * ((double)dx * dx + (double)dy * dy + (double)dz * dz);
    }
    if (ADVANCE) {
        const double ks = wave_sum(kt);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ks;
        __syncthreads();
        if (threadIdx.x == 0) a.ke_stile[tile.w] = ((red[0] + red[1]) + red[2]) + red[3];
        thermostat_if_last(a, r, threadIdx.x < 128, threadIdx.x >> 7);
    }
    if (ENERGY) wave_atomic_energy(ke, a.energy + r * kEnergyTerms + kE_kin);
}

// SLOTS: partials of a compound in flight at a time, 16 in small engines (a round of loads is most of
// a small one's kernel), 8 in others, which the registers of 16 cost a wavefront.
template <bool ADVANCE, bool FIXED, bool ENERGY, int SLOTS>
__global__ __launch_bounds__(kStepThreads) void step_integrate_kernel(StepArgs a, int compound_blocks) {
    if ((int)blockIdx.x < compound_blocks) compound_integrate_role<ADVANCE, FIXED, ENERGY, SLOTS>(a, blockIdx.x);
    else solvent_integrate_role<ADVANCE, FIXED, ENERGY>(a, blockIdx.x - compound_blocks);
}

// sets every replica's step counter (graph-safe: a kernel, not a memset)
__global__ void set_step_count_kernel(long long* step_count, int n_rep, long long v) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n_rep) step_count[r] = v;
}

// ===========================================================================
// Neighbour lists (Engine::updateNeighborLists, Engine.cu:208-287).
// The reference's incremental cull/add with hash dedupe yields, per pair:
//   compound-compound (lo < hi): member = (was && d < C+((r_lo+r_hi)+C)) || d < C+((r_lo+r_lo)+C)
//                                 (the add threshold reads the lower id's radius twice, Engine.cu:243)
//   compound-solvent:            member = d < C + (r_c + C)
//   solvent-solvent (lo < hi):   member = d < C + C
// with d = |a - hyperpos(a, b)| in FP32, a = the lower id (or the compound key).
// Lists are produced in ascending id order (compound lists) or cell-scan order
// (solvent lists); the sets are bit-exact, the order is this build's own.
// ===========================================================================
struct NlistArgs {
    const ReplicaInfo* reps;
    const float4* cpos;
    const float4* spos;
    int n_comp, n_solv;
    const int* comp_off; const int* comp_rep; const int* comp_key; const float* comp_sphere;
    const int* solv_rep;
    float cutoff;
    int cap_cc, cap_cs, cap_ss;
    int* cc_cnt; int* cc_ids;
    int* cs_cnt; int* cs_ids;
    int* ss_cnt; int* ss_ids;   // rows of ss_ld
    int ss_ld;
    int n_cells;
    int* cell_cnt; int* cell_start; int* cell_cursor; int* cell_ids; int* solv_cell;
    const int* cell_rep;          // replica of each cell
    const float* comp_cs_bound;   // per compound: bound(C + (r + C)) for the squared distance
    int* seg_cnt;                 // [n_comp * max_segs] compound-solvent members per solvent segment
    int max_segs;
    int* cw_off; int* cw_total;
    int* item_comp;
    int run_len;                  // neighbour items per run of listed_packed_role (0: not used)
    int* run_off; int* run_cs_off; int* run_total; int* run_comp;   // run_total[2]: neighbour runs, solvent chunks
    uint32_t* err;
    int enable_solvents;
};

LIMA_DEV float4 key_pos(const NlistArgs& a, int c) { return a.cpos[a.comp_off[c] + a.comp_key[c]]; }

// One wavefront per compound, candidates of its replica in ascending id order.
// The compound's previous list is first turned into an LDS bitmask (it is the
// only reader of its own list), then overwritten with the new one.
constexpr int kMaxReplicaCompounds = 8192;

__global__ __launch_bounds__(64) void nl_compound_compound_kernel(NlistArgs a) {
    __shared__ uint32_t was_bits[kMaxReplicaCompounds / 32];
    const int i = blockIdx.x;
    const int lane = threadIdx.x;
    const int r = a.comp_rep[i];
    const ReplicaInfo rp = a.reps[r];
    const int ncr = rp.comp_end - rp.comp_begin;
    if (ncr > kMaxReplicaCompounds) {
        if (lane == 0) atomicOr(a.err, kErrCapacity);
        return;
    }
    const float C = a.cutoff;
    const Box box = make_box(rp.L, rp.half);
    for (int w = lane; w < (ncr + 31) / 32; w += 64) was_bits[w] = 0u;
    __syncthreads();
    const int old_cnt = a.cc_cnt[i];
    for (int e = lane; e < old_cnt; e += 64) {
        const int j = a.cc_ids[(size_t)i * a.cap_cc + e] - rp.comp_begin;
        atomicOr(&was_bits[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    const float4 ki = key_pos(a, i);
    int count = 0;
    for (int j0 = rp.comp_begin; j0 < rp.comp_end; j0 += 64) {
        const int j = j0 + lane;
        bool member = false;
        if (j < rp.comp_end && j != i) {
            const int lo = min(i, j), hi = max(i, j);
            const float4 klo = lo == i ? ki : key_pos(a, j);
            const float4 khi = hi == i ? ki : key_pos(a, j);
            const float rlo = a.comp_sphere[lo], rhi = a.comp_sphere[hi];
            const int jl = j - rp.comp_begin;
            const bool was = (was_bits[jl >> 5] >> (jl & 31)) & 1u;
            const bool keep = within(klo.x, klo.y, klo.z, khi.x, khi.y, khi.z, fadd(fadd(rlo, rhi), C), C, box);
            const bool add = within(klo.x, klo.y, klo.z, khi.x, khi.y, khi.z, fadd(fadd(rlo, rlo), C), C, box);
            member = (was && keep) || add;
        }
        const unsigned long long ball = __ballot(member);
        const int before = __popcll(ball & ((1ull << lane) - 1ull));
        if (member) {
            const int pos = count + before;
            if (pos < a.cap_cc) a.cc_ids[(size_t)i * a.cap_cc + pos] = j;
        }
        count += __popcll(ball);
    }
    if (lane == 0) {
        if (count > a.cap_cc) { atomicOr(a.err, kErrCapacity); atomicMax(a.err + 1, count); }
        a.cc_cnt[i] = min(count, a.cap_cc);
    }
}

// Compound -> solvent lists in ascending solvent order, in two passes over a
// (compound, 2048-solvent segment) grid: count members per segment, then write
// each segment's members at the prefix of the counts before it.
constexpr int kSegSolvents = 2048;

LIMA_DEV bool cs_member(const NlistArgs& a, float4 ki, float bound, int s, const Box& box) {
    const float4 q = a.spos[s];
    // |d| < C + (r + C)  <=>  d^2 < bound (correctly rounded sqrt is monotone)
    return dist2_reimaged(ki.x, ki.y, ki.z, q.x, q.y, q.z, box) < bound;
}

LIMA_DEV void nl_cs_count(const NlistArgs& a, int i, int seg) {
    __shared__ int wsum[4];
    const ReplicaInfo rp = a.reps[a.comp_rep[i]];
    const int s0 = rp.solv_begin + seg * kSegSolvents;
    const int s1 = min(s0 + kSegSolvents, rp.solv_end);
    const float4 ki = key_pos(a, i);
    const float bound = a.comp_cs_bound[i];
    int c = 0;
    for (int s = s0 + (int)threadIdx.x; s < s1; s += blockDim.x) c += cs_member(a, ki, bound, s, make_box(rp.L, rp.half));
    for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) a.seg_cnt[(size_t)i * a.max_segs + seg] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

LIMA_DEV void nl_cs_write(const NlistArgs& a, int i, int seg) {
    __shared__ int wave_cnt[4];
    const ReplicaInfo rp = a.reps[a.comp_rep[i]];
    const int nseg = (rp.solv_end - rp.solv_begin + kSegSolvents - 1) / kSegSolvents;
    const int* sc = a.seg_cnt + (size_t)i * a.max_segs;
    if (seg == 0 && threadIdx.x == 0) {
        int total = 0;
        for (int k = 0; k < nseg; k++) total += sc[k];
        if (total > a.cap_cs) { atomicOr(a.err, kErrCapacity); atomicMax(a.err + 2, total); }
        a.cs_cnt[i] = min(total, a.cap_cs);
    }
    if (seg >= nseg) return;
    int count = 0;
    for (int k = 0; k < seg; k++) count += sc[k];
    const int s0 = rp.solv_begin + seg * kSegSolvents;
    const int s1 = min(s0 + kSegSolvents, rp.solv_end);
    const float4 ki = key_pos(a, i);
    const float bound = a.comp_cs_bound[i];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int b = s0; b < s1; b += 256) {
        const int s = b + threadIdx.x;
        const bool member = s < s1 && cs_member(a, ki, bound, s, make_box(rp.L, rp.half));
        const unsigned long long ball = __ballot(member);
        if (lane == 0) wave_cnt[wid] = __popcll(ball);
        __syncthreads();
        int before = __popcll(ball & ((1ull << lane) - 1ull));
        for (int w = 0; w < wid; w++) before += wave_cnt[w];
        if (member && count + before < a.cap_cs) a.cs_ids[(size_t)i * a.cap_cs + count + before] = s;
        count += wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
        __syncthreads();
    }
}

LIMA_DEV int cell_coord(float v, float inv, int n) {
    int c = (int)(v * inv);
    c = c < 0 ? 0 : c;
    return c >= n ? n - 1 : c;
}

// Wavefront-aggregated counter update: the lanes of each distinct cell in the wavefront add their
// number with one atomic, made by the cell's first lane; returns each lane's slot (the counter's
// old value plus the lane's rank among the cell's lanes).  Consecutive solvents mostly share a
// few cells, so the atomics on one counter drop from one per solvent to one per wavefront.
LIMA_DEV int wave_cell_add(int* counter, int cell, bool valid) {
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long todo = __ballot(valid);
    int slot = 0;
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const int lc = __shfl(cell, leader);
        const unsigned long long same = __ballot(valid && cell == lc) & todo;
        int base = 0;
        if (lane == leader) base = atomicAdd(counter + lc, __popcll(same));
        base = __shfl(base, leader);
        if ((same >> lane) & 1ull) slot = base + __popcll(same & below);
        todo &= ~same;
    }
    return slot;
}

// (the counters are zero: at creation, and again after each rebuild's sort)
LIMA_DEV void nl_cell_count(const NlistArgs& a, int block) {
    const int s = block * (int)blockDim.x + (int)threadIdx.x;
    const bool valid = s < a.n_solv;
    int cell = 0;
    if (valid) {
        const ReplicaInfo rp = a.reps[a.solv_rep[s]];
        const float4 q = a.spos[s];
        const int n = rp.ncell;
        const int cx = cell_coord(q.x, rp.cell_inv, n), cy = cell_coord(q.y, rp.cell_inv, n), cz = cell_coord(q.z, rp.cell_inv, n);
        cell = rp.cell_begin + (cx * n + cy) * n + cz;
        a.solv_cell[s] = cell;
    }
    wave_cell_add(a.cell_cnt, cell, valid);
}

// exclusive scan of cell counts (single block of 1024)
__global__ __launch_bounds__(1024) void nl_cell_scan_kernel(NlistArgs a) {
    __shared__ int part[1024];
    const int n = a.n_cells;
    const int per = (n + 1023) / 1024;
    const int b = threadIdx.x * per;
    int s = 0;
    for (int k = 0; k < per && b + k < n; k++) s += a.cell_cnt[b + k];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        int v = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (int k = 0; k < per && b + k < n; k++) {
        a.cell_start[b + k] = run;
        a.cell_cursor[b + k] = run;
        run += a.cell_cnt[b + k];
    }
    if (threadIdx.x == 1023) a.cell_start[n] = part[1023];
}

LIMA_DEV void nl_cell_scatter(const NlistArgs& a, int block) {
    const int s = block * (int)blockDim.x + (int)threadIdx.x;
    const bool valid = s < a.n_solv;
    const int cell = valid ? a.solv_cell[s] : 0;
    const int pos = wave_cell_add(a.cell_cursor, cell, valid);
    if (valid) a.cell_ids[pos] = s;
}

// The compounds' solvent lists and the solvents' cells do not depend on each other, so their passes
// share launches: counting, then (after the scan of the cells) writing.  A rebuild of a small system
// is its launches, about 5 us each: eleven took 54 us, seven (the counters cleared by the sort, few
// compounds' items written by the work list's block) save 10 to 13 of a rebuild.
__global__ __launch_bounds__(256) void nl_count_kernel(NlistArgs a) {
    const long long b = (long long)blockIdx.y * gridDim.x + blockIdx.x, cs = (long long)a.n_comp * a.max_segs;
    if (b < cs) nl_cs_count(a, (int)(b % a.n_comp), (int)(b / a.n_comp));
    else nl_cell_count(a, (int)(b - cs));
}
__global__ __launch_bounds__(256) void nl_write_kernel(NlistArgs a) {
    const long long b = (long long)blockIdx.y * gridDim.x + blockIdx.x, cs = (long long)a.n_comp * a.max_segs;
    if (b < cs) nl_cs_write(a, (int)(b % a.n_comp), (int)(b / a.n_comp));
    else nl_cell_scatter(a, (int)(b - cs));
}

// sort each cell's ids ascending (rank sort in LDS), making the lists deterministic, and clear its
// counter for the next rebuild
__global__ __launch_bounds__(256) void nl_cell_sort_kernel(NlistArgs a) {
    constexpr int CAP = 2048;
    __shared__ int ids[CAP];
    const int cell = blockIdx.y * gridDim.x + blockIdx.x;
    if (cell >= a.n_cells) return;
    if (threadIdx.x == 0) a.cell_cnt[cell] = 0;
    const int b = a.cell_start[cell], n = a.cell_start[cell + 1] - b;
    if (n > CAP) {
        if (threadIdx.x == 0) { atomicOr(a.err, kErrCapacity); atomicMax(a.err + 3, n); }
        return;
    }
    for (int k = threadIdx.x; k < n; k += blockDim.x) ids[k] = a.cell_ids[b + k];
    __syncthreads();
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const int v = ids[k];
        int rank = 0;
        for (int e = 0; e < n; e++) rank += ids[e] < v;
        a.cell_ids[b + rank] = v;
    }
}

// One block per home cell: the solvents of the (deduplicated) 27 neighbouring
// cells are staged in LDS in a fixed cell order (each cell sorted by id); every
// wavefront tests one home solvent against all candidates.  The pair predicate is
// evaluated with the lower id as the static point, as the reference's add loop
// does (Engine.cu:262-264), and compared as d^2 < bound(C + C).
// 3456 staged candidates (54 KB of positions, 13.5 KB of ids, 8 KB of queues)
// let two blocks share a CU.
constexpr int kCellCandidates = 3456;
constexpr int kSsQueue = 256;   // per-wavefront ring of prefiltered candidate slots
static_assert(kCellCandidates <= 65535 && kCellCandidates % 128 == 0, "16-bit slots, whole passes of 128");

LIMA_DEV bool ss_member(int s, float4 me, int j, float4 q, const Box& box, float bound) {
    const bool lo_self = s < j;
    const float ax = lo_self ? me.x : q.x, ay = lo_self ? me.y : q.y, az = lo_self ? me.z : q.z;
    const float bx = lo_self ? q.x : me.x, by = lo_self ? q.y : me.y, bz = lo_self ? q.z : me.z;
    return (j != s) & (dist2_reimaged(ax, ay, az, bx, by, bz, box) < bound);
}

// 1024 threads: each block carries 16 waves to hide LDS and ballot latency, and
// two blocks fit one CU
constexpr int kSolventListThreads = 1024;

__global__ __launch_bounds__(kSolventListThreads) void nl_solvent_solvent_kernel(NlistArgs a) {
    __shared__ float4 cand_pos[kCellCandidates];
    __shared__ int cand_id[kCellCandidates];
    __shared__ unsigned short queue[kSolventListThreads / 64][kSsQueue];
    __shared__ int cell_b[27], cell_n[27], cell_off[28];
    // cells of one replica are contiguous: XCD-contiguous order keeps a replica's positions in one L2
    const int cell = xcd_item(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    if (cell >= a.n_cells) return;
    const int h0 = a.cell_start[cell], h1 = a.cell_start[cell + 1];
    if (h0 == h1) return;
    const ReplicaInfo rp = a.reps[a.cell_rep[cell]];
    const float L = rp.L, bound = rp.ss_bound;
    const Box box = make_box(rp.L, rp.half);
    const int n = rp.ncell;
    const int local = cell - rp.cell_begin;
    const int cx = local / (n * n), cy = (local / n) % n, cz = local % n;
    const int span = n >= 3 ? 3 : n;
    const int nnb = span * span * span;
    // neighbour cell k = (ox, oy, oz) in a fixed order; grids narrower than 3 cells take every cell once
    auto nb_cell = [&](int k) {
        const int ox = k / (span * span), oy = (k / span) % span, oz = k % span;
        const int x = (n >= 3) ? (cx - 1 + ox + n) % n : ox;
        const int y = (n >= 3) ? (cy - 1 + oy + n) % n : oy;
        const int z = (n >= 3) ? (cz - 1 + oz + n) % n : oz;
        return rp.cell_begin + (x * n + y) * n + z;
    };
    // all cell ranges at once, then an exclusive scan of their sizes
    if (threadIdx.x < nnb) {
        const int c = nb_cell(threadIdx.x);
        const int b = a.cell_start[c];
        cell_b[threadIdx.x] = b;
        cell_n[threadIdx.x] = a.cell_start[c + 1] - b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int k = 0; k < nnb; k++) {
            cell_off[k] = acc;
            acc += cell_n[k];
        }
        cell_off[nnb] = acc;
    }
    __syncthreads();
    const int total = cell_off[nnb];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    // With 3 or more cells per side each neighbour cell has one image next to the home cell, and
    // its candidates are staged shifted into it, so that the prefilter below is a plain distance
    // (the exact test reads the raw positions); narrower grids stage them raw.
    const bool shifted = n >= 3;
    const unsigned long long below = (1ull << lane) - 1ull;
    const int nhome = h1 - h0;
    const float rb = sqrtf(bound) + 1e-5f * L + 1e-6f;
    const float pre = rb * rb;
    // below this the cheap distance certifies membership: per axis it differs from the exactly
    // rounded re-imaged difference by a few roundings of coordinates up to 2L, far below the margin
    const float ri = sqrtf(bound) - (1e-5f * L + 1e-6f);
    const float inner = ri * ri;
    unsigned short* q = queue[wid];
    // The candidates, in the fixed cell order, pass through LDS kCellCandidates at a time; each
    // home solvent takes every chunk in turn, so its row is in candidate order whatever the chunks.
    // Between chunks the row's running count (not yet clamped to the capacity) waits in ss_cnt.
    for (int c0 = 0; c0 < total; c0 += kCellCandidates) {
        const int c1 = min(total, c0 + kCellCandidates);
        const bool last = c1 == total;
        if (c0 > 0) {
            // every wavefront is done with the previous chunk, and the running counts it stored
            // are visible to the loads below
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __syncthreads();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        // stage: wavefront w copies the parts of cells w, w + nw, ... that fall in [c0, c1)
        for (int k = wid; k < nnb; k += nw) {
            const int b = cell_b[k], o = cell_off[k], m = cell_n[k];
            const int e0 = max(0, c0 - o), e1 = min(m, c1 - o);
            if (e0 >= e1) continue;
            float sx = 0.f, sy = 0.f, sz = 0.f;
            if (shifted) {
                const int ux = cx - 1 + k / 9, uy = cy - 1 + (k / 3) % 3, uz = cz - 1 + k % 3;
                sx = ux < 0 ? -L : ux >= n ? L : 0.f;
                sy = uy < 0 ? -L : uy >= n ? L : 0.f;
                sz = uz < 0 ? -L : uz >= n ? L : 0.f;
            }
            for (int e = e0 + lane; e < e1; e += 64) {
                const int id = a.cell_ids[b + e];
                const float4 x = a.spos[id];
                cand_id[o + e - c0] = id;
                cand_pos[o + e - c0] = make_float4(x.x + sx, x.y + sy, x.z + sz, x.w);
            }
        }
        // pad to whole passes of 128 with NaN positions, which no distance test accepts
        const int nc = c1 - c0;
        const int padded = (nc + 127) & ~127;
        if (threadIdx.x < padded - nc) {
            const float nan = __builtin_nanf("");
            cand_pos[nc + threadIdx.x] = make_float4(nan, nan, nan, nan);
        }
        __syncthreads();
        // Each wavefront takes home solvents in turn.  A cheap distance (minimum image on grids
        // narrower than 3 cells), with a margin far above its rounding error against the exact
        // re-imaged one, drops the candidates that cannot be members; the rest enter the
        // wavefront's queue in candidate order.  Whenever 64 are queued, the exact predicate
        // runs on them and the members are appended in that order (ballot compaction), so each
        // list is the one a test of every candidate in order would give.
        for (int h = wid; h < nhome; h += nw) {
            const int s = a.cell_ids[h0 + h];
            const float4 me = a.spos[s];
            int* row = a.ss_ids + (size_t)s * a.ss_ld;
            int count = c0 == 0 ? 0 : a.ss_cnt[s];
            unsigned head = 0, tail = 0;   // wavefront-uniform queue cursors
            auto dist2 = [&](float4 c) {   // the cheap distance of a staged candidate
                float dx = c.x - me.x, dy = c.y - me.y, dz = c.z - me.z;
                if (!shifted) {
                    dx = fabsf(dx); dy = fabsf(dy); dz = fabsf(dz);
                    dx = fminf(dx, fabsf(L - dx)); dy = fminf(dy, fabsf(L - dy)); dz = fminf(dz, fabsf(L - dz));
                }
                return dx * dx + dy * dy + dz * dz;
            };
            auto drain = [&](int m) {      // membership of the m <= 64 oldest queued slots
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // other lanes' queue writes
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const bool has = lane < m;
                const int e = has ? (int)q[(head + lane) & (kSsQueue - 1)] : 0;
                const int j = cand_id[e];
                const float d2 = dist2(cand_pos[e]);
                bool mem = has & (j != s) & (d2 < inner);
                // the exact predicate only for slots near the bound (wavefront-uniform branch)
                const bool band = has & !mem & (j != s);
                if (__ballot(band) != 0ull)
                    mem = mem | (band && ss_member(s, me, j, shifted ? a.spos[j] : cand_pos[e], box, bound));
                const unsigned long long bm = __ballot(mem);
                const int pos = count + __popcll(bm & below);
                if (mem & (pos < a.cap_ss)) row[pos] = j;
                count += __popcll(bm);
                head += m;
            };
            auto near = [&](int e) { return dist2(cand_pos[e]) < pre; };
            for (int e0 = 0; e0 < padded; e0 += 128) {
                const int ea = e0 + lane, eb = ea + 64;
                const bool ma = near(ea), mb = near(eb);
                const unsigned long long ba = __ballot(ma), bb = __ballot(mb);
                const unsigned ta = tail + __popcll(ba);
                if (ma) q[(tail + __popcll(ba & below)) & (kSsQueue - 1)] = (unsigned short)ea;
                if (mb) q[(ta + __popcll(bb & below)) & (kSsQueue - 1)] = (unsigned short)eb;
                tail = ta + __popcll(bb);
                while (tail - head >= 64u) drain(64);   // at most 191 queued, 63 left
            }
            while (tail != head) drain((int)min(64u, tail - head));
            if (lane == 0) {
                if (!last) {
                    a.ss_cnt[s] = count;
                } else {
                    if (count > a.cap_ss) { atomicOr(a.err, kErrCapacity); atomicMax(a.err + 3, count); }
                    a.ss_cnt[s] = min(count, a.cap_ss);
                }
            }
        }
    }
}

// per compound work slots: listed neighbours + ceil(solvent list / 256); exclusive scan.  With
// run_len > 0 (listed_packed_role), also the compound's runs: ceil(neighbours / run_len)
// + ceil(solvent list / 256), scanned into run_off.
// run_len > 0: the compound's runs of run_len neighbours; run_len == 0: its work items (one per
// listed neighbour, then one per solvent chunk); run_len < 0: its solvent chunks alone
LIMA_DEV int work_count(const NlistArgs& a, int c, int run_len) {
    const int chunks = a.enable_solvents ? (a.cs_cnt[c] + kSolventChunk - 1) / kSolventChunk : 0;
    if (run_len > 0) return (a.cc_cnt[c] + run_len - 1) / run_len;
    if (run_len < 0) return chunks;
    return a.cc_cnt[c] + chunks;
}

LIMA_DEV void block_exclusive_scan(int* part, const NlistArgs& a, int run_len, int* off, int* total) {
    const int n = a.n_comp;
    const int per = (n + 1023) / 1024;
    const int b = threadIdx.x * per;
    int s = 0;
    for (int k = 0; k < per && b + k < n; k++) s += work_count(a, b + k, run_len);
    part[threadIdx.x] = s;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        int v = threadIdx.x >= o ? part[threadIdx.x - o] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (int k = 0; k < per && b + k < n; k++) {
        off[b + k] = run;
        run += work_count(a, b + k, run_len);
    }
    if (threadIdx.x == 1023) { off[n] = part[1023]; *total = part[1023]; }
    __syncthreads();
}

// the compound of every work item, and of every run, of compound c (a wavefront)
constexpr int kWorkItemsInPlace = 64;
LIMA_DEV void nl_items(const NlistArgs& a, int c, int lane) {
    for (int w = a.cw_off[c] + lane; w < a.cw_off[c + 1]; w += 64) a.item_comp[w] = c;
    if (a.run_len > 0) {
        for (int w = a.run_off[c] + lane; w < a.run_off[c + 1]; w += 64) a.run_comp[w] = c;
        const int cs0 = a.run_total[0];
        for (int w = a.run_cs_off[c] + lane; w < a.run_cs_off[c + 1]; w += 64) a.run_comp[cs0 + w] = c;
    }
}
// With run_len > 0 (listed_packed_role) the run list holds every compound's neighbour
// runs first (run_off, run_total[0] of them), then every compound's solvent chunks (run_cs_off,
// run_total[1]), so that the groups of a wavefront mostly take runs of one kind.
__global__ __launch_bounds__(1024) void nl_work_kernel(NlistArgs a) {
    __shared__ int part[1024];
    block_exclusive_scan(part, a, 0, a.cw_off, a.cw_total);
    if (a.run_len > 0) {
        block_exclusive_scan(part, a, a.run_len, a.run_off, a.run_total);
        block_exclusive_scan(part, a, -1, a.run_cs_off, a.run_total + 1);
    }
    // few compounds: their items at once, without a launch
    if (a.n_comp <= kWorkItemsInPlace) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (int c = threadIdx.x >> 6; c < a.n_comp; c += 16) nl_items(a, c, threadIdx.x & 63);
    }
}

__global__ __launch_bounds__(64) void nl_item_kernel(NlistArgs a) { nl_items(a, blockIdx.x, threadIdx.x); }

}  // namespace lima
