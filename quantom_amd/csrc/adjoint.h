// adjoint.h — reverse-mode (adjoint) kernels of the LIMA_MD step for parameter
// gradients of trajectory losses.
//
// Forward model (thermostat off, lambda = 1, neighbour lists piecewise constant):
//     x_{k+1} = 2 x_k - x_{k-1} + c * F(x_k; theta),   c = dt^2 / m   (Engine.cu:849-869)
// Loss over frames k = 0..K-1:
//     L = sum_k [ alpha_r (E_k - E*_k)^2 + beta_r sum_i |F_k,i - F*_k,i|^2 ]
// Backward recurrence (a_k = dL/dx_k):
//     w_k = a_{k+1} * c + 2 beta (F_k - F*_k),  g_k = 2 alpha (E_k - E*_k)
//     a_k = G_x(x_k; w_k, g_k) + 2 a_{k+1} - a_{k+2},   dL/dtheta += G_theta(x_k; w_k, g_k)
// where G(w, g) is the gradient of  w . F(x) + g E(x)  with respect to x and theta.
//
// LJ pairs (calcLJForce, Engine.cu:475-522): f = d phi(q), d = x_j - x_i, q = |d|^2.  With the
// force's own constants A = 24e sigma^6, B = -48e sigma^12 (lj_ab):
//     phi = A q^-4 + B q^-7,  psi = -dphi/dq = 4 A q^-5 + 7 B q^-8,
//     d(w.f)/dd = phi w - 2 psi (w.d) d,   U = -(A q^-3 + B/2 q^-6) / 6,  dU/dd = phi d.
// A directed pair weighs (w.f) by its receiver's w and U by half the frame's g.  As A and B enter
// linearly, a pair's derivatives are q^-3 ((w.d)/q - gU/6) and q^-6 ((w.d)/q - gU/12); the chain
// rule to sigma and epsilon follows once per pair of types where a thread sums one.
// Position gradients are gathered only, by each end's thread.  Parameter derivatives are credited
// to both types of a pair: where each end's thread sees the pair (solvent-solvent, inter- and
// intra-compound) each credits its own type, and the solvent <-> chain sites are credited to both
// by the chain's thread.  That is exactly the mixing-rule chain rule (both types receive
// d/dsigma^2 * sigma_m; arithmetic eps 12 x, geometric eps e24/(2 eps_t) x).  Bonded terms are
// differentiated in forward mode, one direction (a coordinate or a constant) a lane.
#pragma once
#include "kernels.h"

namespace lima {

constexpr int kAdjTypeBins = 3 * kMaxTypes;   // per type: sigma, eps (arithmetic sites), eps*e24 (geometric sites)

// ---- dual numbers: a value and its derivative in one direction ----------------
struct Dual {
    float v, d;
};
LIMA_DEV Dual dconst(float v) { return {v, 0.f}; }
LIMA_DEV Dual dvar(float v, bool on) { return {v, on ? 1.f : 0.f}; }
LIMA_DEV Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
LIMA_DEV Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
LIMA_DEV Dual operator-(Dual a) { return {-a.v, -a.d}; }
LIMA_DEV Dual operator*(Dual a, Dual b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
LIMA_DEV Dual operator*(Dual a, float s) { return {a.v * s, a.d * s}; }
LIMA_DEV Dual operator/(Dual a, Dual b) {
    const float inv = 1.0f / b.v, v = a.v * inv;
    return {v, (a.d - v * b.d) * inv};
}
LIMA_DEV Dual dsqrt(Dual a) {
    const float v = sqrtf(a.v);
    return {v, a.d * (v > 0.f ? 0.5f / v : 0.f)};
}

struct V3d {
    Dual x, y, z;
};
LIMA_DEV V3d vadd(const V3d& a, const V3d& b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
LIMA_DEV V3d vsub(const V3d& a, const V3d& b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
LIMA_DEV V3d vneg(const V3d& a) { return {-a.x, -a.y, -a.z}; }
LIMA_DEV V3d vscale(const V3d& a, Dual s) { return {a.x * s, a.y * s, a.z * s}; }
LIMA_DEV V3d vscalef(const V3d& a, float s) { return {a.x * s, a.y * s, a.z * s}; }
LIMA_DEV Dual vdot(const V3d& a, const V3d& b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
LIMA_DEV V3d vcross(const V3d& a, const V3d& b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
LIMA_DEV Dual vlen(const V3d& a) { return dsqrt(vdot(a, a)); }
LIMA_DEV V3d vnorm(const V3d& a) {
    const Dual l = vlen(a);
    if (l.v != 0.f) return vscale(a, dconst(1.f) / l);
    return {dconst(0.f), dconst(0.f), dconst(0.f)};
}
// Float3::getAngle with its clamp (QuantomTypes.cuh:74-83)
LIMA_DEV Dual dangle(const V3d& a, const V3d& b) {
    const Dual val = vdot(a, b) / (vlen(a) * vlen(b));
    if (val.v >= 1.f) return dconst(0.f);
    if (val.v <= -1.f) return dconst(3.14159265358979f);
    return {acosf(val.v), val.d * (-1.0f / sqrtf(1.0f - val.v * val.v))};
}

// coordinates k0, k0 + 1, k0 + 2 of a term; `dir` is the differentiated one
LIMA_DEV V3d dpos(float4 p, int k0, int dir) { return {dvar(p.x, dir == k0), dvar(p.y, dir == k0 + 1), dvar(p.z, dir == k0 + 2)}; }
LIMA_DEV float dot_w(const V3d& f, float4 w) { return w.x * f.x.d + w.y * f.y.d + w.z * f.z.d; }

// Derivative of  sum_atoms w.F + g E  in one direction, for one bond (calcPairbondForces,
// Engine.cu:525-548): directions 0..5 positions, 6 b0, 7 kb
constexpr int kBondDirs = 8, kAngleDirs = 11, kDihedralDirs = 12;
LIMA_DEV float bond_vjp(float4 a, float4 b, float b0, float kb, float4 wa, float4 wb, float g, int dir) {
    const V3d A = dpos(a, 0, dir), B = dpos(b, 3, dir);
    const Dual B0 = dvar(b0, dir == 6), KB = dvar(kb, dir == 7);
    const V3d diff = vsub(A, B);
    const Dual err = vlen(diff) - B0;
    const Dual E = KB * err * err * 0.5f;
    const V3d fa = vscale(vnorm(diff), -(KB * err));
    return dot_w(fa, wa) + dot_w(vneg(fa), wb) + g * E.d;
}

// one angle (calcAnglebondForces, Engine.cu:552-578): directions 0..8 positions, 9 theta0, 10 k
LIMA_DEV float angle_vjp(float4 l, float4 m, float4 r, float t0, float k, float4 wl, float4 wm, float4 wr, float g, int dir) {
    const V3d L = dpos(l, 0, dir), M = dpos(m, 3, dir), R = dpos(r, 6, dir);
    const Dual T0 = dvar(t0, dir == 9), K = dvar(k, dir == 10);
    const V3d v1 = vsub(L, M), v2 = vsub(R, M);
    const V3d dir1 = vnorm(vcross(v1, vcross(v2, v1)));
    const V3d dir2 = vnorm(vcross(v2, vcross(v1, v2)));
    const Dual err = dangle(v1, v2) - T0;
    const Dual E = K * err * err * 0.25f;
    const Dual fsc = K * err;
    const V3d fl = vscale(dir1, fsc), fr = vscale(dir2, fsc);
    const V3d fm = vneg(vadd(fl, fr));
    return dot_w(fl, wl) + dot_w(fm, wm) + dot_w(fr, wr) + g * E.d;
}

// one dihedral (calcDihedralbondForces, Engine.cu:580-637): directions 0..11 positions
LIMA_DEV float dihedral_vjp(float4 l, float4 lm, float4 rm, float4 r, float phi0, float k, int n, float4 wl, float4 wlm,
                            float4 wrm, float4 wr, float g, int dir) {
    const V3d L = dpos(l, 0, dir), LM = dpos(lm, 3, dir), RM = dpos(rm, 6, dir), R = dpos(r, 9, dir);
    V3d n1 = vnorm(vcross(vsub(L, LM), vsub(RM, LM)));
    V3d n2 = vnorm(vcross(vsub(LM, RM), vsub(R, RM)));
    const Dual tors = dangle(n1, n2);
    const float lp = vlen(vsub(vadd(L, n1), R)).v, lmn = vlen(vsub(vsub(L, n1), R)).v;
    if (lp < lmn) n2 = vneg(n2);
    else n1 = vneg(n1);
    const Dual arg = tors * (float)n - dconst(phi0);
    const float sn = sinf(arg.v), cs = cosf(arg.v);
    const Dual fs{k * sn, arg.d * (k * cs)};
    const V3d fl = vscale(n1, fs), fr = vscale(n2, fs);
    const V3d fmid = vscalef(vadd(fl, fr), -0.5f);
    return dot_w(fl, wl) + dot_w(fmid, wlm) + dot_w(fmid, wrm) + dot_w(fr, wr) + g * (arg.d * (k * sn));
}

// ---- LJ pair derivatives -----------------------------------------------------
struct D3 {
    double x, y, z;
};
LIMA_DEV float3 xyz(float4 v) { return make_float3(v.x, v.y, v.z); }
LIMA_DEV float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
struct Powers {
    float inv, i3, i4, i5, i6;   // q^-1 .. q^-6; the reciprocal is 1 ulp, as the force's
};
LIMA_DEV Powers powers(float3 d) {
    Powers p;
    p.inv = __builtin_amdgcn_rcpf(pair_r2(d.x, d.y, d.z));
    const float i2 = p.inv * p.inv;
    p.i3 = i2 * p.inv;
    p.i4 = i2 * i2;
    p.i5 = p.i4 * p.inv;
    p.i6 = p.i3 * p.i3;
    return p;
}
// phi and psi of constants (A, B)
LIMA_DEV void phi_psi(const Powers& p, float A, float B, float& phi, float& psi) {
    const float x = B * p.i3, y = A + x;
    phi = p.i4 * y;
    psi = p.i5 * __builtin_fmaf(4.f, y, 3.f * x);
}
// derivatives of  ud phi + gU U  by A and B
LIMA_DEV void pair_dab(const Powers& p, float ud, float gU, float& dA, float& dB) {
    dA = p.i3 * __builtin_fmaf(ud, p.inv, gU * (-1.f / 6.f));
    dB = p.i6 * __builtin_fmaf(ud, p.inv, gU * (-1.f / 12.f));
}
// Sums over a particle's thousands of pairs cancel heavily, so the gathers
// accumulate in FP64 (the per-pair terms stay FP32).
LIMA_DEV void gather(D3& acc, float x, float y, float z) {
    acc.x -= (double)x;
    acc.y -= (double)y;
    acc.z -= (double)z;
}
// One directed LJ site seen from particle P: d = x_other - x_P, u = the force
// weight as seen from P (w_P when P receives the force, -w_receiver when P is
// the source), gU = weight of the site's energy.
LIMA_DEV void site(const Powers& p, float3 d, float3 u, float ud, float gU, float A, float B, D3& acc) {
    float phi, psi;
    phi_psi(p, A, B, phi, psi);
    const float c = __builtin_fmaf(gU, phi, -2.f * ud * psi);
    gather(acc, __builtin_fmaf(phi, u.x, c * d.x), __builtin_fmaf(phi, u.y, c * d.y), __builtin_fmaf(phi, u.z, c * d.z));
}
// sums dA, dB of one pair of types, of 24 eps = e24: d/dsigma_t (half of both types' sum) and d/d(24 eps)
LIMA_DEV void chain_rule(double dA, double dB, float4 pr, double e24, double& ds, double& de) {
    const double s2 = pr.x, s6 = s2 * s2 * s2, v = dB * s6;
    de = s6 * (dA - 2.0 * v);
    ds = e24 * s2 * s2 * (double)pr.w * (3.0 * dA - 12.0 * v);
}

constexpr int kAdjStride = kAdjTypeBins + 4;   // per replica: type bins, then kb, b0, k_theta, theta0

// ===========================================================================
// A frame is two launches: adj_frame_kernel, whose blocks take one role each (as
// step_forces_kernel's do), and adj_update_kernel.  As five kernels one after the other a frame of
// 4 compounds and 1,488 solvents took 235 us, each bound by its own chain of loads.
// ===========================================================================
struct AdjArgs {
    StepArgs s;              // the frame's positions (cpos, spos), its lists and the type tables
    const float4* wc;        // [NCH] weight of the chain forces
    const float4* ws;        // [NS] weight of the solvent forces
    const float* gE;         // [R] weight of the frame's potential energy
    float4* gxc;             // [kAdjChainSlots + solvent slices][NCH] parts: bonded, bridges, intra-compound, then the slices
    float4* gxs;             // [chain chunks + 1][NS]
    double* gpar;            // [R][kAdjStride]
    const uint32_t* cs_mask; // per compound, bitmask over its replica's solvents: listed by the compound
    const int* mask_off;     // [n_comp] first word of each compound's mask
    const int* comp_of;      // [NCH] compound of each chain particle
    int n_chain;             // NCH: stride of the chain parts
    float4* gpart;           // [work item][128]: neighbour-compound parts, per step work item
    int comp_chunk;          // compounds per block of the solvent-side role
    int comp_split;          // blocks per compound of it (comp_chunk 1)
    int n_cchunks;           // blocks per solvent tile of it
    int solv_slice;          // solvents per block of the chain-side role
    int n_sslices;
    int nb, na;              // most bonds and angles of any compound (LDS strides)
};
struct AdjBlocks {
    int bonded, bridges, intra, listed, solvent, chain, pairs;   // blocks of each role
    int width;                                                   // the grid's (grid_of)
};
constexpr int kAdjThreads = 256;
constexpr int kAdjChainSlots = 3;
constexpr int kAdjRows = 256;            // rows staged by the solvent- and chain-side roles
constexpr int kAdjPairLanes = 16;        // lanes per solvent of the solvent-solvent role
constexpr int kAdjBridgeTerms = 16;      // terms of a bridge evaluated at a time
constexpr size_t kAdjHead = kAdjStride * sizeof(double);   // the block's parameter bins

LIMA_DEV void bins_zero(double* bins) {
    for (int i = threadIdx.x; i < kAdjStride; i += kAdjThreads) bins[i] = 0.0;
    __syncthreads();
}
// type t's credits: sigma, arithmetic 24eps, geometric 24eps (already times 24eps)
LIMA_DEV void bins_credit(double* bins, int t, double s, double ea, double eg) {
    if (s != 0.0) atomicAdd(&bins[t], s);
    if (ea != 0.0) atomicAdd(&bins[kMaxTypes + t], ea);
    if (eg != 0.0) atomicAdd(&bins[2 * kMaxTypes + t], eg);
}
// add the block's bins to the replica's and clear them (each thread clears the entries it added)
LIMA_DEV void bins_flush(double* bins, double* g) {
    __syncthreads();
    for (int i = threadIdx.x; i < kAdjStride; i += kAdjThreads) {
        if (bins[i] != 0.0) atomicAdd(&g[i], bins[i]);
        bins[i] = 0.0;
    }
    __syncthreads();
}

// Threads of a block on the n <= 128 target particles of a compound: `lanes` of them (a power of
// two from 16) hold one target each, and the 256 / lanes groups share the sources.
struct Targets {
    int lanes, p, group, groups;
    bool active;
};
LIMA_DEV Targets targets(int n) {
    Targets t;
    t.lanes = n <= 16 ? 16 : n <= 32 ? 32 : n <= 64 ? 64 : 128;
    t.p = threadIdx.x & (t.lanes - 1);
    t.group = threadIdx.x / t.lanes;
    t.groups = kAdjThreads / t.lanes;
    t.active = t.p < n;
    return t;
}
// sums N values of each target over the groups, in group order, into the first group's threads;
// red: [N][256] doubles
template <int N> LIMA_DEV void group_reduce(const Targets& t, double* red, double (&v)[N]) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) red[k * kAdjThreads + threadIdx.x] = v[k];
    __syncthreads();
    if (t.group) return;
#pragma unroll
    for (int k = 0; k < N; k++)
        for (int g = 1; g < t.groups; g++) v[k] += red[k * kAdjThreads + g * t.lanes + t.p];
}

// ---------------------------------------------------------------------------
// Solvent side of the solvent <-> chain sites.  Block = (solvent tile of 256, chunk of compounds,
// or part of one).  For every chain particle j of the chunk: the all-pairs site "solvent <- j"
// (arithmetic eps, Engine.cu:1099-1117) and, when the solvent is in j's compound list, the
// transpose of "j <- solvent" (geometric eps, Engine.cu:964-974).  The two see the same distance
// unless the second's re-imaging of j against its compound's particle 0 moves it (possible only in
// positions as a caller first set them), and both sites mix sigma arithmetically, so they are one
// site of 24 eps = 1 with the weight  ea w - eg w_j  and the energy weight  (ea + eg) g/2.
// ---------------------------------------------------------------------------
LIMA_DEV void adj_solvent_role(const AdjArgs& A, int blk, char* lds) {
    const StepArgs& a = A.s;
    float4* rows = reinterpret_cast<float4*>(lds);               // x, y, z, 24 eps (arithmetic)
    float4* roww = rows + kAdjRows;                              // -eg w, eg = 24 eps (geometric)
    float2* rowab = reinterpret_cast<float2*>(roww + kAdjRows);  // A, B of 24 eps = 1
    const int4 tile = a.stiles[blk / A.n_cchunks];
    const int y = blk % A.n_cchunks;
    const int r = tile.x;
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const int s = tile.y + threadIdx.x;
    const bool active = s < tile.z;
    const int si = active ? s : tile.y;
    const float4 me = a.spos[si];
    const float3 w = xyz(A.ws[si]);
    const float gh = 0.5f * A.gE[r];
    const int sl = si - rp.solv_begin;
    D3 acc{0.0, 0.0, 0.0};
    const int c0 = rp.comp_begin + y / A.comp_split * A.comp_chunk;
    const int c1 = min(c0 + A.comp_chunk, rp.comp_end);
    if (c0 < c1) {
        int pb = a.comp_off[c0], pe = a.comp_off[c1];
        if (A.comp_split > 1) {   // a part of compound c0
            const int per = (pe - pb + A.comp_split - 1) / A.comp_split, part = y % A.comp_split;
            const int b = min(pb + part * per, pe);
            pe = min(b + per, pe);
            pb = b;
        }
        bool moved = false;
        for (int k = threadIdx.x; k < pe - pb; k += kAdjThreads) {
            const float4 q = a.cpos[pb + k], p0 = a.cpos[a.comp_off[A.comp_of[pb + k]]], wj = A.wc[pb + k];
            float qx = q.x, qy = q.y, qz = q.z;
            hyperpos(p0.x, p0.y, p0.z, qx, qy, qz, box);
            moved = moved || qx != q.x || qy != q.y || qz != q.z;
            const float4 pa = a.tab_sc[r * kMaxTypes + ftype(q)], pg = a.tab_cs[r * kMaxTypes + ftype(q)];
            rows[k] = make_float4(q.x, q.y, q.z, pa.y);
            roww[k] = make_float4(-wj.x * pg.y, -wj.y * pg.y, -wj.z * pg.y, pg.y);
            rowab[k] = lj_ab(pa.x, 1.f);
        }
        moved = __syncthreads_or(moved) != 0;
        for (int c = c0; c < c1; c++) {
            const int lb = max(a.comp_off[c], pb) - pb, le = min(a.comp_off[c + 1], pe) - pb;
            if (lb >= le) continue;
            const float4 p0 = a.cpos[a.comp_off[c]];
            float ix = me.x, iy = me.y, iz = me.z;
            hyperpos(p0.x, p0.y, p0.z, ix, iy, iz, box);
            const bool listed = (A.cs_mask[A.mask_off[c] + (sl >> 5)] >> (sl & 31)) & 1u;
            const float on = listed ? 1.f : 0.f;
            if (__ballot(listed) == 0ull) {
#pragma unroll 2
                for (int j = lb; j < le; j++) {
                    const float4 q = rows[j];
                    const float2 ab = rowab[j];
                    const float3 d = make_float3(q.x - ix, q.y - iy, q.z - iz);
                    site(powers(d), d, w, dot3(w, d), gh, q.w * ab.x, q.w * ab.y, acc);
                }
            } else if (!moved) {
#pragma unroll 2
                for (int j = lb; j < le; j++) {
                    const float4 q = rows[j], v = roww[j];
                    const float2 ab = rowab[j];
                    const float3 d = make_float3(q.x - ix, q.y - iy, q.z - iz);
                    const float3 u = make_float3(__builtin_fmaf(q.w, w.x, on * v.x), __builtin_fmaf(q.w, w.y, on * v.y),
                                                 __builtin_fmaf(q.w, w.z, on * v.z));
                    site(powers(d), d, u, dot3(u, d), gh * __builtin_fmaf(on, v.w, q.w), ab.x, ab.y, acc);
                }
            } else {
                for (int j = lb; j < le; j++) {
                    const float4 q = rows[j], v = roww[j];
                    const float2 ab = rowab[j];
                    float3 d = make_float3(q.x - ix, q.y - iy, q.z - iz);
                    site(powers(d), d, w, dot3(w, d), gh, q.w * ab.x, q.w * ab.y, acc);
                    float qx = q.x, qy = q.y, qz = q.z;
                    hyperpos(p0.x, p0.y, p0.z, qx, qy, qz, box);
                    d = make_float3(qx - ix, qy - iy, qz - iz);
                    const float3 u = make_float3(on * v.x, on * v.y, on * v.z);
                    site(powers(d), d, u, dot3(u, d), gh * on * v.w, ab.x, ab.y, acc);
                }
            }
        }
    }
    if (active) A.gxs[(size_t)y * a.n_solv + s] = make_float4((float)acc.x, (float)acc.y, (float)acc.z, 0.f);
}

// ---------------------------------------------------------------------------
// Chain side of the same sites.  Block = (compound, slice of solv_slice solvents): the transpose
// of "solvent <- j" with the solvent imaged against the compound's particle 0 and j's stored
// position, as the forward pass pairs them, and "j <- solvent" for the solvents that the compound
// lists.  A thread's pairs are all of one pair of types, so it sums each site's derivative by its
// own 24 eps, and dB of 24 eps = 1 over both sites; dA follows from the three.  The geometric
// derivative is later divided by 2 eps, so it has a sum of its own: as what the arithmetic one left
// of both sites' it carried that one's rounding (1,219 solvents, eps_t = eps_0 / 1000: the gradient
// by eps_t was 4.1e-5 off, 3.1e-6 now).  The credits go to both types.
// ---------------------------------------------------------------------------
LIMA_DEV void adj_chain_role(const AdjArgs& A, int blk, double* bins, char* lds) {
    const StepArgs& a = A.s;
    float4* sp = reinterpret_cast<float4*>(lds);   // x, y, z, listed
    float4* sw = sp + kAdjRows;                    // -w
    const int c = blk / A.n_sslices, y = blk % A.n_sslices;
    const int r = a.comp_rep[c];
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
    const Targets t = targets(n);
    const int gi = base + (t.active ? t.p : 0);
    const float4 me = a.cpos[gi];
    const float4 p0 = a.cpos[base];
    float ix = me.x, iy = me.y, iz = me.z;
    hyperpos(p0.x, p0.y, p0.z, ix, iy, iz, box);
    const bool moved = __syncthreads_or(ix != me.x || iy != me.y || iz != me.z) != 0;
    const float3 w = xyz(A.wc[gi]);
    const int tp = ftype(me);
    const float4 pa = a.tab_sc[r * kMaxTypes + tp], pg = a.tab_cs[r * kMaxTypes + tp];
    const float2 ab = lj_ab(pa.x, 1.f);
    const float gh = 0.5f * A.gE[r], ga = gh * pa.y, gg = gh * pg.y;
    const float3 wg = make_float3(pg.y * w.x, pg.y * w.y, pg.y * w.z);
    D3 acc{0.0, 0.0, 0.0};
    double dBs = 0.0, dEa = 0.0, dEg = 0.0;
    const int s0 = rp.solv_begin + y * A.solv_slice;
    const int s1 = min(s0 + A.solv_slice, rp.solv_end);
    for (int t0 = s0; t0 < s1; t0 += kAdjRows) {
        const int ns = min(kAdjRows, s1 - t0), k = threadIdx.x;
        __syncthreads();
        if (k < ns) {
            float4 q = a.spos[t0 + k];
            hyperpos(p0.x, p0.y, p0.z, q.x, q.y, q.z, box);
            const int sl = t0 + k - rp.solv_begin;
            q.w = (A.cs_mask[A.mask_off[c] + (sl >> 5)] >> (sl & 31)) & 1u ? 1.f : 0.f;
            sp[k] = q;
            const float4 v = A.ws[t0 + k];
            sw[k] = make_float4(-v.x, -v.y, -v.z, 0.f);
        }
        __syncthreads();
        // the sites of row j at distance d: the arithmetic one of weight `arith` (0 or 1), the geometric one of `on`
        auto sites = [&](float3 d, float3 v, float arith, float on) {
            const Powers p = powers(d);
            const float vd = dot3(v, d), wd = dot3(w, d), ea = arith * pa.y;
            const float3 u = make_float3(__builtin_fmaf(ea, v.x, on * wg.x), __builtin_fmaf(ea, v.y, on * wg.y),
                                         __builtin_fmaf(ea, v.z, on * wg.z));
            const float ud = __builtin_fmaf(ea, vd, on * pg.y * wd), gU = __builtin_fmaf(on, gg, arith * ga);
            float phi, psi;
            phi_psi(p, ab.x, ab.y, phi, psi);
            const float c = __builtin_fmaf(gU, phi, -2.f * ud * psi);
            gather(acc, __builtin_fmaf(phi, u.x, c * d.x), __builtin_fmaf(phi, u.y, c * d.y), __builtin_fmaf(phi, u.z, c * d.z));
            dBs += (double)(p.i6 * __builtin_fmaf(ud, p.inv, gU * (-1.f / 12.f)));
            // of 24 eps = 1: (receiver's weight . d) phi + g/2 U
            const float energy = gh * (-1.f / 6.f) * p.i3 * __builtin_fmaf(0.5f * ab.y, p.i3, ab.x);
            dEa += (double)(arith * __builtin_fmaf(vd, phi, energy));
            dEg += (double)(on * __builtin_fmaf(wd, phi, energy));
        };
        if (!moved) {
#pragma unroll 2
            for (int j = t.group; j < ns; j += t.groups) {
                const float4 q = sp[j];
                sites(make_float3(q.x - me.x, q.y - me.y, q.z - me.z), xyz(sw[j]), 1.f, q.w);
            }
        } else {
            for (int j = t.group; j < ns; j += t.groups) {
                const float4 q = sp[j];
                const float3 v = xyz(sw[j]);
                sites(make_float3(q.x - me.x, q.y - me.y, q.z - me.z), v, 1.f, 0.f);
                sites(make_float3(q.x - ix, q.y - iy, q.z - iz), v, 0.f, q.w);
            }
        }
    }
    double v[6] = {acc.x, acc.y, acc.z, dBs, dEa, dEg};
    group_reduce(t, reinterpret_cast<double*>(lds), v);
    if (t.group == 0 && t.active) {
        A.gxc[(size_t)(kAdjChainSlots + y) * A.n_chain + gi] = make_float4((float)v[0], (float)v[1], (float)v[2], 0.f);
        // both sites' sum s6 (dA - 2 s6 dB) of 24 eps = 1 gives dA for the chain rule to sigma
        const double s2 = pa.x, v6 = v[3] * s2 * s2 * s2, eg = pg.y * v[5], both = pa.y * v[4] + eg;
        const double ds = s2 > 0.0 ? 3.0 * (double)pa.w / s2 * (both - 2.0 * s2 * s2 * s2 * v6) : 0.0;
        bins_credit(bins, tp, ds, v[4], eg);
        bins_credit(bins, 0, ds, v[4], eg);
    }
    bins_flush(bins, A.gpar + (size_t)r * kAdjStride);
}

// ---------------------------------------------------------------------------
// Solvent-solvent pairs, both directions of each symmetric pair (Engine.cu:1119-1128): 16 lanes a
// solvent, each on every 16th entry of its list, so that a row is read in whole segments and 16
// gathers are in flight where one lane had one.
// ---------------------------------------------------------------------------
LIMA_DEV void adj_pairs_role(const AdjArgs& A, int blk, double* bins) {
    const StepArgs& a = A.s;
    constexpr int PER = kAdjThreads / kAdjPairLanes;   // solvents of a block
    const int4 tile = a.stiles[blk / (256 / PER)];
    const int first = tile.y + blk % (256 / PER) * PER;
    if (first >= tile.z) return;   // the same for the block
    const int r = tile.x;
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const int s = first + (int)threadIdx.x / kAdjPairLanes, sub = threadIdx.x % kAdjPairLanes;
    const bool active = s < tile.z;
    const int si = active ? s : first;
    const float4 me = a.spos[si];
    const float3 w = xyz(A.ws[si]);
    const float g = A.gE[r];
    const float4 pss = a.tab_ss[r];
    const float2 ab = lj_ab(pss.x, pss.y);
    D3 acc{0.0, 0.0, 0.0};
    double sA = 0.0, sB = 0.0;
    const int cnt = active ? a.ss_cnt[si] : 0;
    const int* row = a.ss_ids + (size_t)si * a.ss_ld;
#pragma unroll 4
    for (int k = sub; k < cnt; k += kAdjPairLanes) {
        const int j = row[k];
        float4 q = a.spos[j];
        const float4 wj = A.ws[j];
        hyperpos(me.x, me.y, me.z, q.x, q.y, q.z, box);
        const float3 d = make_float3(q.x - me.x, q.y - me.y, q.z - me.z), u = make_float3(w.x - wj.x, w.y - wj.y, w.z - wj.z);
        const Powers p = powers(d);
        const float ud = dot3(u, d);
        site(p, d, u, ud, g, ab.x, ab.y, acc);
        float dA, dB;
        pair_dab(p, ud, g, dA, dB);
        sA += (double)dA;
        sB += (double)dB;
    }
    acc.x = group_sum<kAdjPairLanes>(acc.x);
    acc.y = group_sum<kAdjPairLanes>(acc.y);
    acc.z = group_sum<kAdjPairLanes>(acc.z);
    if (active && sub == 0)
        A.gxs[(size_t)A.n_cchunks * a.n_solv + s] = make_float4((float)acc.x, (float)acc.y, (float)acc.z, 0.f);
    sA = wave_sum(sA);
    sB = wave_sum(sB);
    if ((threadIdx.x & 63) == 0) {
        double ds, de;
        chain_rule(sA, sB, pss, pss.y, ds, de);
        bins_credit(bins, 0, ds, de, 0.0);
    }
    bins_flush(bins, A.gpar + (size_t)r * kAdjStride);
}

// ---------------------------------------------------------------------------
// Pairs of a compound's particles with those of a neighbour compound (arithmetic eps,
// Engine.cu:653-676) or of itself (INTRA: geometric eps, Engine.cu:678-700), both directions of
// each pair: the pair enters p's force unless p excludes j and j's force unless j excludes p.
// Returns the position gradient and the credits of target t in `v` (complete in the first group).
// ---------------------------------------------------------------------------
struct AdjPairStage {
    float4 sp[kCompoundBlock], sw[kCompoundBlock];
    uint32_t mask[kCompoundBlock * 4];   // the sources' exclusions of this compound's particles
};
template <bool INTRA>
LIMA_DEV void adj_compound_pairs(const AdjArgs& A, int r, int c, int nb, const Targets& t, char* lds, double (&v)[5]) {
    const StepArgs& a = A.s;
    AdjPairStage& st = *reinterpret_cast<AdjPairStage*>(lds);
    const ReplicaInfo rp = a.reps[r];
    const Box box = make_box(rp.L, rp.half);
    const int base = a.comp_off[c];
    const int gi = base + (t.active ? t.p : 0);
    const float4 p0 = a.cpos[base];
    float4 me = a.cpos[gi];
    hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, box);
    const float3 w = xyz(A.wc[gi]);
    const float gh = 0.5f * A.gE[r];
    const int tp = ftype(me);
    const int nbase = a.comp_off[nb], nn = a.comp_off[nb + 1] - nbase;
    uint32_t m0 = 0u, m1 = 0u, m2 = 0u, m3 = 0u, any = 0u;
    __syncthreads();   // the stage is free
    if ((int)threadIdx.x < nn) {
        const int j = threadIdx.x, gj = nbase + j;
        float4 q = a.cpos[gj];
        hyperpos(p0.x, p0.y, p0.z, q.x, q.y, q.z, box);
        st.sp[j] = q;
        st.sw[j] = A.wc[gj];
        uint32_t b0 = 0u, b1 = 0u, b2 = 0u, b3 = 0u;
        if (INTRA) {
            b0 = a.intra_mask[(size_t)gj * 4]; b1 = a.intra_mask[(size_t)gj * 4 + 1];
            b2 = a.intra_mask[(size_t)gj * 4 + 2]; b3 = a.intra_mask[(size_t)gj * 4 + 3];
        } else {
            for (int e = a.xoff[gj]; e < a.xoff[gj + 1]; e++) {
                const int2 x = a.xent[e];
                const uint32_t bit = x.x == c ? 1u << (x.y & 31) : 0u;
                const int ws = x.y >> 5;
                b0 |= ws == 0 ? bit : 0u; b1 |= ws == 1 ? bit : 0u; b2 |= ws == 2 ? bit : 0u; b3 |= ws == 3 ? bit : 0u;
            }
        }
        any = b0 | b1 | b2 | b3;
        st.mask[j * 4] = b0; st.mask[j * 4 + 1] = b1; st.mask[j * 4 + 2] = b2; st.mask[j * 4 + 3] = b3;
    }
    if (INTRA) {
        m0 = a.intra_mask[(size_t)gi * 4]; m1 = a.intra_mask[(size_t)gi * 4 + 1];
        m2 = a.intra_mask[(size_t)gi * 4 + 2]; m3 = a.intra_mask[(size_t)gi * 4 + 3];
    } else if (t.active) {
        for (int e = a.xoff[gi]; e < a.xoff[gi + 1]; e++) {
            const int2 x = a.xent[e];
            const uint32_t bit = x.x == nb ? 1u << (x.y & 31) : 0u;
            const int ws = x.y >> 5;
            m0 |= ws == 0 ? bit : 0u; m1 |= ws == 1 ? bit : 0u; m2 |= ws == 2 ? bit : 0u; m3 |= ws == 3 ? bit : 0u;
        }
    }
    D3 acc{0.0, 0.0, 0.0};
    double bs = 0.0, be = 0.0;
    const float4* tab = (INTRA ? a.tab_intra : a.tab_inter) + (size_t)r * kMaxTypes * kMaxTypes + tp;
    auto pair = [&](float3 u, float gU, float4 q) {
        const float4 pr = tab[ftype(q) * kMaxTypes];
        const float3 d = make_float3(q.x - me.x, q.y - me.y, q.z - me.z);
        const Powers p = powers(d);
        const float ud = dot3(u, d);
        const float s4 = pr.x * pr.x, s6 = s4 * pr.x, ea = pr.y * s6;
        site(p, d, u, ud, gU, ea, -2.0f * ea * s6, acc);
        float dA, dB;
        pair_dab(p, ud, gU, dA, dB);
        const float v6 = dB * s6;
        bs += (double)(pr.y * s4 * pr.w * __builtin_fmaf(-12.f, v6, 3.f * dA));
        be += (double)((INTRA ? ea : s6) * __builtin_fmaf(-2.f, v6, dA));   // geometric: times 24 eps
    };
    if (!INTRA && !__syncthreads_or((int)(any | m0 | m1 | m2 | m3))) {
        // no exclusions between the two (they exist only where a bridge joins them): both directions of every pair
        const float g = A.gE[r];
#pragma unroll 2
        for (int j = t.group; j < nn; j += t.groups) {
            const float4 wj = st.sw[j];
            pair(make_float3(w.x - wj.x, w.y - wj.y, w.z - wj.z), g, st.sp[j]);
        }
    } else {
        if (INTRA) __syncthreads();
#pragma unroll 2
        for (int j = t.group; j < nn; j += t.groups) {
            const int jw = j >> 5;
            const uint32_t mw = jw == 0 ? m0 : jw == 1 ? m1 : jw == 2 ? m2 : m3;
            const float4 wj = st.sw[j];
            const float fp = (mw >> (j & 31)) & 1u ? 0.f : 1.f, fj = (st.mask[j * 4 + (t.p >> 5)] >> (t.p & 31)) & 1u ? 0.f : 1.f;
            if (fp + fj == 0.f || (INTRA && j == t.p)) continue;
            pair(make_float3(fp * w.x - fj * wj.x, fp * w.y - fj * wj.y, fp * w.z - fj * wj.z), gh * (fp + fj), st.sp[j]);
        }
    }
    v[0] = acc.x; v[1] = acc.y; v[2] = acc.z; v[3] = bs; v[4] = be;
    group_reduce(t, reinterpret_cast<double*>(lds), v);
}

LIMA_DEV void adj_intra_role(const AdjArgs& A, int c, double* bins, char* lds) {
    const StepArgs& a = A.s;
    const int r = a.comp_rep[c], base = a.comp_off[c];
    const Targets t = targets(a.comp_off[c + 1] - base);
    double v[5];
    adj_compound_pairs<true>(A, r, c, c, t, lds, v);
    if (t.group == 0 && t.active) {
        A.gxc[(size_t)2 * A.n_chain + base + t.p] = make_float4((float)v[0], (float)v[1], (float)v[2], 0.f);
        bins_credit(bins, ftype(a.cpos[base + t.p]), v[3], 0.0, v[4]);
    }
    bins_flush(bins, A.gpar + (size_t)r * kAdjStride);
}

// the neighbour-compound items of the step's work list, one part per item
LIMA_DEV void adj_listed_role(const AdjArgs& A, int blk, int nblk, double* bins, char* lds) {
    const StepArgs& a = A.s;
    const int total = *a.cw_total;
    for (int wi = blk; wi < total; wi += nblk) {
        const int c = a.item_comp[wi], k = wi - a.cw_off[c];
        if (k >= a.cc_cnt[c]) continue;   // a solvent chunk: adj_chain_role's
        const int r = a.comp_rep[c], base = a.comp_off[c];
        const Targets t = targets(a.comp_off[c + 1] - base);
        double v[5];
        adj_compound_pairs<false>(A, r, c, a.cc_ids[(size_t)c * a.cap_cc + k], t, lds, v);
        if (t.group == 0 && t.active) {
            A.gpart[(size_t)wi * kCompoundBlock + t.p] = make_float4((float)v[0], (float)v[1], (float)v[2], 0.f);
            bins_credit(bins, ftype(a.cpos[base + t.p]), v[3], v[4], 0.0);
        }
        bins_flush(bins, A.gpar + (size_t)r * kAdjStride);
    }
}

// ---------------------------------------------------------------------------
// A compound's bonded terms: a lane per (term, direction), the derivatives kept in LDS and
// gathered per particle in term order.  Derivatives by the bonded constants are summed over terms.
// ---------------------------------------------------------------------------
inline size_t adj_bonded_lds(int nb, int na, int nd) {
    return 2 * kCompoundBlock * sizeof(float4) + (size_t)(6 * nb + 9 * na + 12 * nd) * sizeof(float);
}
LIMA_DEV void adj_bonded_role(const AdjArgs& A, int c, double* bins, char* lds) {
    const StepArgs& a = A.s;
    float4* pos = reinterpret_cast<float4*>(lds);
    float4* wv = pos + kCompoundBlock;
    float* gb = reinterpret_cast<float*>(wv + kCompoundBlock);
    float* ga = gb + 6 * A.nb;
    float* gd = ga + 9 * A.na;
    const int tid = threadIdx.x, r = a.comp_rep[c];
    const ReplicaInfo rp = a.reps[r];
    const int base = a.comp_off[c], n = a.comp_off[c + 1] - base;
    const float g = A.gE[r];
    if (tid < n) {
        const float4 p0 = a.cpos[base];
        float4 me = a.cpos[base + tid];
        hyperpos(p0.x, p0.y, p0.z, me.x, me.y, me.z, make_box(rp.L, rp.half));
        pos[tid] = me;
        wv[tid] = A.wc[base + tid];
    }
    __syncthreads();
    const int b0 = a.bond_off[c], nbd = a.bond_off[c + 1] - b0;
    const int a0 = a.angle_off[c], nan_ = a.angle_off[c + 1] - a0;
    const int d0 = a.dih_off[c], ndh = a.enable_dihedrals ? a.dih_off[c + 1] - d0 : 0;
    double kb_g = 0.0, b0_g = 0.0, kt_g = 0.0, t0_g = 0.0;
    for (int u = tid; u < ndh * kDihedralDirs; u += kAdjThreads) {
        const int t = u / kDihedralDirs, dir = u % kDihedralDirs;
        const DihD dd = a.dihs[d0 + t];
        gd[t * 12 + dir] = dihedral_vjp(pos[dd.a0], pos[dd.a1], pos[dd.a2], pos[dd.a3], dd.p0, dd.k, dd.n, wv[dd.a0], wv[dd.a1],
                                        wv[dd.a2], wv[dd.a3], g, dir);
    }
    for (int u = tid; u < nan_ * kAngleDirs; u += kAdjThreads) {
        const int t = u / kAngleDirs, dir = u % kAngleDirs;
        const AngleD ad = a.angles[a0 + t];
        const float o = angle_vjp(pos[ad.a0], pos[ad.a1], pos[ad.a2], ad.t0, ad.k, wv[ad.a0], wv[ad.a1], wv[ad.a2], g, dir);
        if (dir < 9) ga[t * 9 + dir] = o;
        t0_g += dir == 9 ? (double)o : 0.0;
        kt_g += dir == 10 ? (double)o : 0.0;
    }
    for (int u = tid; u < nbd * kBondDirs; u += kAdjThreads) {
        const int t = u / kBondDirs, dir = u % kBondDirs;
        const BondD bd = a.bonds[b0 + t];
        const float o = bond_vjp(pos[bd.a0], pos[bd.a1], bd.b0, bd.kb, wv[bd.a0], wv[bd.a1], g, dir);
        if (dir < 6) gb[t * 6 + dir] = o;
        b0_g += dir == 6 ? (double)o : 0.0;
        kb_g += dir == 7 ? (double)o : 0.0;
    }
    auto credit = [&](int k, double x) {
        x = wave_sum(x);
        if ((tid & 63) == 0 && x != 0.0) atomicAdd(&bins[kAdjTypeBins + k], x);
    };
    credit(0, kb_g);
    credit(1, b0_g);
    credit(2, kt_g);
    credit(3, t0_g);
    __syncthreads();
    if (tid < n) {
        const int gi = base + tid;
        D3 acc{0.0, 0.0, 0.0};
        for (int e = a.inc_off[gi]; e < a.inc_off[gi + 1]; e++) {
            const uint32_t v = a.inc[e];
            const uint32_t kind = v >> 30, slot = v & 3u, term = (v >> 2) & 0xFFFFFFFu;
            if (kind == 2 && !a.enable_dihedrals) continue;
            const float* x = kind == 0 ? gb + term * 6 + slot * 3 : kind == 1 ? ga + term * 9 + slot * 3 : gd + term * 12 + slot * 3;
            acc.x += x[0];
            acc.y += x[1];
            acc.z += x[2];
        }
        A.gxc[gi] = make_float4((float)acc.x, (float)acc.y, (float)acc.z, 0.f);
    }
    bins_flush(bins, A.gpar + (size_t)r * kAdjStride);
}

// ---------------------------------------------------------------------------
// Bridges (Engine.cu:897-916): one wavefront per bridge, a lane per (term, direction) of
// kAdjBridgeTerms terms at a time, each particle's lane then adding its own in term order.  The
// sums go to slot 1 of the chain parts (a particle belongs to at most one bridge; particles of
// none keep the zero that the slot was filled with).
// ---------------------------------------------------------------------------
struct AdjBridgeStage {
    float4 pos[kBridgeParticles], wv[kBridgeParticles];
    float out[kAdjBridgeTerms * 12];
    int who[kAdjBridgeTerms * 4];
};
LIMA_DEV void adj_bridge_role(const AdjArgs& A, int b, AdjBridgeStage& st) {
    const StepArgs& a = A.s;
    if (b >= a.n_bridges) return;
    const int lane = threadIdx.x & 63, r = a.br_rep[b];
    const ReplicaInfo rp = a.reps[r];
    const float g = A.gE[r];
    const int q0 = a.br_off[b], np = min(a.br_off[b + 1] - q0, kBridgeParticles);
    if (lane < np) {
        const int gi = a.br_glob[q0 + lane];
        const float4 first = a.cpos[a.br_glob[q0]];
        float4 q = a.cpos[gi];
        if (lane > 0) hyperpos(first.x, first.y, first.z, q.x, q.y, q.z, make_box(rp.L, rp.half));
        st.pos[lane] = q;
        st.wv[lane] = A.wc[gi];
    }
    wave_sync();
    D3 acc{0.0, 0.0, 0.0};
    double par[2] = {0.0, 0.0};   // the kind's two constants, in direction order
    auto sweep = [&](int nterms, int atoms, int dirs, auto&& eval) {
        for (int c0 = 0; c0 < nterms; c0 += kAdjBridgeTerms) {
            const int nt = min(kAdjBridgeTerms, nterms - c0);
            for (int u = lane; u < nt * dirs; u += 64) {
                const int t = u / dirs, dir = u % dirs;
                const float o = eval(c0 + t, dir, &st.who[t * 4]);
                if (dir < 3 * atoms) st.out[t * 12 + dir] = o;
                else par[dir - 3 * atoms] += (double)o;
            }
            wave_sync();
            if (lane < np)
                for (int t = 0; t < nt; t++)
                    for (int k = 0; k < atoms; k++)
                        if (st.who[t * 4 + k] == lane) {
                            const float* x = st.out + t * 12 + k * 3;
                            acc.x += x[0];
                            acc.y += x[1];
                            acc.z += x[2];
                        }
            wave_sync();
        }
    };
    double* gr = A.gpar + (size_t)r * kAdjStride + kAdjTypeBins;
    auto credit = [&](int first, int second) {
        const double x = wave_sum(par[0]), y = wave_sum(par[1]);
        if (lane == 0 && x != 0.0) atomicAdd(gr + first, x);
        if (lane == 0 && y != 0.0) atomicAdd(gr + second, y);
        par[0] = par[1] = 0.0;
    };
    const float4 *pos = st.pos, *wv = st.wv;
    const int tb = a.brb_off[b], ta = a.bra_off[b], td = a.brd_off[b];
    sweep(a.brb_off[b + 1] - tb, 2, kBondDirs, [&](int t, int dir, int* who) {
        const BondD bd = a.brb[tb + t];
        who[0] = bd.a0; who[1] = bd.a1;
        return bond_vjp(pos[bd.a0], pos[bd.a1], bd.b0, bd.kb, wv[bd.a0], wv[bd.a1], g, dir);
    });
    credit(1, 0);
    sweep(a.bra_off[b + 1] - ta, 3, kAngleDirs, [&](int t, int dir, int* who) {
        const AngleD ad = a.bra[ta + t];
        who[0] = ad.a0; who[1] = ad.a1; who[2] = ad.a2;
        return angle_vjp(pos[ad.a0], pos[ad.a1], pos[ad.a2], ad.t0, ad.k, wv[ad.a0], wv[ad.a1], wv[ad.a2], g, dir);
    });
    credit(3, 2);
    sweep(a.enable_dihedrals ? a.brd_off[b + 1] - td : 0, 4, kDihedralDirs, [&](int t, int dir, int* who) {
        const DihD dd = a.brd[td + t];
        who[0] = dd.a0; who[1] = dd.a1; who[2] = dd.a2; who[3] = dd.a3;
        return dihedral_vjp(pos[dd.a0], pos[dd.a1], pos[dd.a2], pos[dd.a3], dd.p0, dd.k, dd.n, wv[dd.a0], wv[dd.a1], wv[dd.a2],
                            wv[dd.a3], g, dir);
    });
    if (lane < np) A.gxc[(size_t)A.n_chain + a.br_glob[q0 + lane]] = make_float4((float)acc.x, (float)acc.y, (float)acc.z, 0.f);
}

__global__ __launch_bounds__(kAdjThreads, 4) void adj_frame_kernel(AdjArgs A, AdjBlocks f) {
    extern __shared__ float4 dyn_lds[];
    double* bins = reinterpret_cast<double*>(dyn_lds);
    char* lds = reinterpret_cast<char*>(dyn_lds) + kAdjHead;
    int b = blockIdx.y * f.width + blockIdx.x;
    if (b < f.bridges) {
        const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        adj_bridge_role(A, 4 * b + wid, reinterpret_cast<AdjBridgeStage*>(lds)[wid]);
        return;
    }
    b -= f.bridges;
    if (b < f.bonded + f.intra + f.listed + f.chain + f.pairs + f.solvent) bins_zero(bins);
    if (b < f.bonded) return adj_bonded_role(A, b, bins, lds);
    b -= f.bonded;
    if (b < f.intra) return adj_intra_role(A, b, bins, lds);
    b -= f.intra;
    if (b < f.pairs) return adj_pairs_role(A, b, bins);
    b -= f.pairs;
    if (b < f.solvent) return adj_solvent_role(A, b, lds);
    b -= f.solvent;
    if (b < f.chain) return adj_chain_role(A, b, bins, lds);
    b -= f.chain;
    if (b < f.listed) adj_listed_role(A, b, f.listed, bins, lds);
}

// bitmask of each compound's solvent list over its replica's solvents
__global__ void adj_mask_zero_kernel(uint32_t* m, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) m[i] = 0u;
}
__global__ __launch_bounds__(256) void adj_mask_set_kernel(StepArgs a, uint32_t* mask, const int* mask_off) {
    const int c = blockIdx.x;
    const ReplicaInfo rp = a.reps[a.comp_rep[c]];
    const int cnt = a.cs_cnt[c];
    for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
        const int sl = a.cs_ids[(size_t)c * a.cap_cs + k] - rp.solv_begin;
        atomicOr(&mask[mask_off[c] + (sl >> 5)], 1u << (sl & 31));
    }
}

// Before a forward frame: its positions kept in X (chain first; or not, X null) and the energy sums cleared.
__global__ __launch_bounds__(256) void adj_begin_kernel(const float4* cpos, const float4* spos, float4* X, double* energy, int nch,
                                                       int ns, int n_energy) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_energy) energy[i] = 0.0;
    if (X && i < nch + ns) X[i] = i < nch ? cpos[i] : spos[i - nch];
}

// After it, per particle: the force residual r = 2 beta (F - F*) of the frame (targets as
// x, y, z triples, or none) and, when `lacc` is given, beta |F - F*|^2 added to the
// particle's own FP64 loss accumulator (one owner per entry: no atomics); the frame's energies kept.
__global__ __launch_bounds__(256) void adj_residual_kernel(const float4* fc, const float4* fs, const float* tc, const float* ts,
                                                           const int* prep, const double* beta, float4* rout, double* lacc,
                                                           const double* energy, double* kept, int nch, int ns, int n_energy) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_energy) kept[i] = energy[i];
    if (i >= nch + ns) return;
    const bool chain = i < nch;
    if (!chain && !fs) {   // solvents disabled
        rout[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const double b = beta[prep[i]];
    const size_t e = chain ? i : i - nch;
    const float4 F = chain ? fc[e] : fs[e];
    const float* t = chain ? tc : ts;
    const float3 T = t ? make_float3(t[3 * e], t[3 * e + 1], t[3 * e + 2]) : make_float3(0.f, 0.f, 0.f);
    const float dx = F.x - T.x, dy = F.y - T.y, dz = F.z - T.z;
    const float tb = (float)(2.0 * b);
    rout[i] = make_float4(tb * dx, tb * dy, tb * dz, 0.f);
    if (lacc) lacc[i] += b * ((double)dx * dx + (double)dy * dy + (double)dz * dz);
}

// per system: the sum of its particles' loss accumulators (chain range, then solvent range)
__global__ __launch_bounds__(256) void adj_loss_reduce_kernel(const ReplicaInfo* reps, const double* lacc, int nch,
                                                              double* loss) {
    __shared__ double red[4];
    const ReplicaInfo rp = reps[blockIdx.x];
    double s = 0.0;
    for (int i = rp.chain_begin + threadIdx.x; i < rp.chain_end; i += blockDim.x) s += lacc[i];
    for (int i = rp.solv_begin + threadIdx.x; i < rp.solv_end; i += blockDim.x) s += lacc[nch + i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) loss[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// w_k = (dt^2/m) a_{k+1} + r_k
LIMA_DEV float4 adj_weight(float4 r, double4 an, double c) {
    return make_float4((float)(an.x * c + r.x), (float)(an.y * c + r.y), (float)(an.z * c + r.z), 0.f);
}
__global__ __launch_bounds__(256) void adj_weight_kernel(const float4* resid, const double4* a_next, const float* cfac,
                                                         float4* w, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w[i] = adj_weight(resid[i], a_next[i], cfac[i]);
}

// a_k = G_x + 2 a_{k+1} - a_{k+2} in FP64 (the recurrence runs over the whole
// trajectory), G_x summed over its parts in slot order; with `resid` (of frame k - 1) also w_{k-1}
__global__ __launch_bounds__(256) void adj_update_kernel(AdjArgs A, int chain_slots, int solv_slots, const double4* a1,
                                                         const double4* a2, double4* out, const float4* resid,
                                                         const float* cfac, float4* w) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int nch = A.n_chain, ns = A.s.n_solv;
    if (i >= nch + ns) return;
    double gx = 0.0, gy = 0.0, gz = 0.0;
    auto add = [&](float4 v) { gx += v.x; gy += v.y; gz += v.z; };
    if (i < nch) {
#pragma unroll 4
        for (int k = 0; k < chain_slots; k++) add(A.gxc[(size_t)k * nch + i]);
        const int c = A.comp_of[i], p = i - A.s.comp_off[c], w0 = A.s.cw_off[c], n = A.s.cc_cnt[c];
#pragma unroll 4
        for (int k = 0; k < n; k++) add(A.gpart[(size_t)(w0 + k) * kCompoundBlock + p]);
    } else {
#pragma unroll 4
        for (int k = 0; k < solv_slots; k++) add(A.gxs[(size_t)k * ns + (i - nch)]);
    }
    const double4 x = a1[i], y = a2[i];
    const double4 a = make_double4(gx + 2.0 * x.x - y.x, gy + 2.0 * x.y - y.y, gz + 2.0 * x.z - y.z, 0.0);
    out[i] = a;
    if (resid) w[i] = adj_weight(resid[i], a, cfac[i]);
}

}  // namespace lima
