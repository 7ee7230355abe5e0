// Fused FP64 FCT path for gfx950: two edge passes and three node-column passes.
//
// Mapping: one 64-lane wavefront per task (a node or an edge, times a tracer); lane l of
// slot s holds level k = 64*s + l of the task's column, so every load of a node or edge
// column is one coalesced row segment, and vertical neighbours move between lanes with
// DPP wavefront shifts. For nl > 64 the node passes run as two launches over a node list
// (kl_*): columns whose wet layers fit 64 lanes in a one-slot kernel, which needs fewer
// registers, the others in the two-slot kernel. With two tracers on a 6-slot mesh the
// one-slot launches take one wavefront per node for both tracers (kl_pass*_all), so the
// tracer-independent loads are made once; a column of at most 32 levels holds one tracer in
// each half of that wavefront. Task indices are wave-uniform (scalar
// registers); each node reads its stencil (incident edges in the reference's summation
// order with the layer ranges of their triangles, incident triangles with their
// vertices) from a per-node table with scalar loads, and then issues the loads of all
// its neighbours' columns back to back. Only wet lanes are computed; T_new is written
// on every lane (dry lanes: T + 0, as the reference's ale_reconstruct does). The kernels
// are bound by the vector memory path (address and data units, L1), so the design
// removes 64-lane loads wherever it can: tables through scalar loads, k-1/k+1 values by
// lane shifts, the node gradient only where an edge reads it, adf_v handed from pass 2
// to pass 3.
//
//   kf_vflux  (edge) : vflux on the edge's wet levels (edge_vflux, tracer_adv.py:69-93)
//   kf_pass1  (node) : LO and the node-averaged gradient gnode (kl_pass1 over a node list)
//                      (compute_fct_lo :298-313, tracer_gradient_elements :316-326,
//                       _node_avg_grad :329-341)
//   k_vimpl   (column): with the implicit split w_i, LO solved for the implicit vertical
//                      advection (:487-529, fct_column.hip)
//   kf_adfh   (edge) : adf_h = MFCT high order - upwind low order, once per edge-level
//                      (:96-105, :196-225, fill_up_dn_grad :344-368)
//   kf_pass2  (node) : cluster bounds, P+/P-, limiter factors (zalesak_limit :389-451),
//                      and adf_v (adv_flux_ver_ho :241-295) stored for pass 3
//   kf_pass3  (node) : limited fluxes, flux2dtracer_fct, ale_reconstruct
//                      (:453-466, :469-484, :142-151)
//
// Operation order and per-node summation order are those of fct_phased.hip (and of the
// reference's jnp expressions). Terms the reference adds as exact zeros (edges or
// elements dry at level k, where the reference multiplies a finite value by 0) are
// skipped, which leaves every sum bit-identical while the inputs are finite on the
// lanes the reference multiplies by zero. The cluster bounds use the fact that the
// vertices of the triangles around a node are the node and the far ends of its edges
// (checked on the host when the plan is built): a maximum over the triangles' vertex
// maxima equals the maximum over that vertex set, whatever the grouping.

#include <cstring>

#include "fct_wave.h"

namespace fct {

struct FusedArgs {
    DevMesh m;
    NodeTab tab;
    double* vflux;         // [D][L]
    const int2* ekr;       // [D] wet level range of the edge [lo, hi)
    const double* uv;
    const double* helem;
    const double* w_e;
    const double* w_i;     // optional implicit part: adf_v takes w_e + w_i
    const double* hnode;
    const double* hnn;
    const double* Z3d;     // optional
    const double* zbar3;   // optional
    double dt;
    int remap;             // block -> task remap, XCD count | chunk << 8 (1 = identity)
    int K;                 // tracers in this launch (<= FCT_KCHUNK)
    const double* T[FCT_KCHUNK];
    const double* Told[FCT_KCHUNK];
    double* Tnew[FCT_KCHUNK];
    double* LO;            // [K][N][L]
    double2* gnode;        // [K][N][L]
    double* adfh;          // [K][D][L]
    double* pf;            // [K][N][L]
    double* adfv;          // [K][N][L] adf_v at each node interface, from pass 2 for pass 3
};

// Batched launches look up (instance, first wavefront) per workgroup.
__device__ __forceinline__ int batch_wave(const int2* __restrict__ blk, int remap, int& inst) {
    const int2 bi = blk[block_tile(remap)];
    inst = __builtin_amdgcn_readfirstlane(bi.x);
    return __builtin_amdgcn_readfirstlane(bi.y + (int)(threadIdx.x >> 6));
}

// ---------------------------------------------------------------------------
// vflux on [kmin_e, kmax_e) for EPW consecutive edges, loads issued together
// ---------------------------------------------------------------------------
template <int NS, int EPW>
__device__ __forceinline__ void vflux_group(const FusedArgs& a, int g) {
    const DevMesh& m = a.m;
    const int L = m.L;
    int e[EPW], tr[EPW];
    int2 et[EPW], kr[EPW];
    double4 c[EPW];
    int kmax = 0;
#pragma unroll
    for (int q = 0; q < EPW; ++q) {
        const int eq = g * EPW + q;
        e[q] = eq < m.D ? (a.tab.vorder ? ldc(a.tab.vorder, eq) : eq) : m.D - 1;
        et[q] = ldc(m.edge_tri, e[q]);
        kr[q] = eq < m.D ? ldc(a.ekr, e[q]) : make_int2(0, 0);
        c[q] = ldc(m.cross, e[q]);
        tr[q] = ldc(m.etr, e[q]);
        kmax = kr[q].y > kmax ? kr[q].y : kmax;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (64 * s >= kmax) break;
        const int k = 64 * s + lane_id();
        double2 u1[EPW], u2[EPW];
        double h1[EPW], h2[EPW];
        if (k < kmax) {
#pragma unroll
            for (int q = 0; q < EPW; ++q) {
                const size_t i1 = (size_t)(et[q].x >= 0 ? et[q].x : 0) * L + k;
                const size_t i2 = (size_t)(et[q].y >= 0 ? et[q].y : 0) * L + k;
                u1[q] = ldv(reinterpret_cast<const double2*>(a.uv), i1);
                u2[q] = ldv(reinterpret_cast<const double2*>(a.uv), i2);
                h1[q] = G(a.helem)[i1];
                h2[q] = G(a.helem)[i2];
            }
        }
#pragma unroll
        for (int q = 0; q < EPW; ++q) {
            if (k < kr[q].x || k >= kr[q].y) continue;
            double t1 = 0.0, t2 = 0.0;
            if (in_bytes(tr[q], 0, k))
                t1 = (u1[q].x * c[q].y - u1[q].y * c[q].x) * h1[q];
            if (in_bytes(tr[q], 16, k))
                t2 = (u2[q].y * c[q].z - u2[q].x * c[q].w) * h2[q];
            G(a.vflux)[(size_t)e[q] * L + k] = t1 + t2;
        }
    }
}

// ---------------------------------------------------------------------------
// pass 1 of node n, tracer j: LO and gnode
// ---------------------------------------------------------------------------
// One node's loops run over DM slots of its ST-slot table row. On an 8-slot mesh most nodes
// have 5 or 6 neighbours: those take the 6-slot loops (a wave-uniform branch), which leaves
// out the loads of two repeated slots (icosa-7 x 70 with 1 % of nodes at 8, two tracers:
// pass 1 293 -> 268 us, pass 2 364 -> 333, pass 3 262 -> 260).
template <int NS, int DM, int ST>
__device__ __forceinline__ void pass1_slots(const FusedArgs& a, int n, int j, int4 hd,
                                            double (*s_nb)[ST + 1][64]) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);   // levels, counts
    // levels at which the adf_h pass reads this node's gnode, as a range [glo, ghi)
    const int ghz = hd.z;
    const int glo = (ghz >> 8) & 0xff, ghi = (ghz >> 16) & 0xff;
    const auto T = G(a.T[j]);
    const size_t b0 = (size_t)n * L;
    const size_t jo = (size_t)j * m.N * L;
    const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
    int4 es[DM];
    int4 el[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
        el[q] = ldc(a.tab.elem, (size_t)n * ST + q);
    }
    // per wavefront: the neighbour columns at the lane's level, then the node's own
    double* nb = &s_nb[threadIdx.x >> 6][0][lane_id()];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (64 * s > nr.y) break;
        const int k = 64 * s + lane_id();
        const bool rd = k < kneed;
        const bool wet = in_layer(nr, k);
        const bool gslot = glo < ghi && glo < 64 * s + 64 && ghi > 64 * s;
        // own column, k-1 and k+1 of T for the vertical fluxes (the one-slot body takes
        // k-1 and k+1 from the neighbouring lanes below)
        const double Tk = rd ? T[b0 + k] : 0.0;
        double Tm = 0.0, Tp = 0.0;
        if (NS > 1) {
            Tm = (rd && k > 0) ? T[b0 + k - 1] : Tk;
            Tp = (k + 1 < kneed) ? T[b0 + k + 1] : 0.0;
        }
        // all neighbour columns and edge fluxes at once (one basic block: slot indices
        // past the node's count repeat slot 0 and are ignored when summing)
        double To[DM] = {}, vf[DM] = {};
        // the node's own fields at k (and k+1 for the lower interface), with the gathers
        double w0 = 0.0, a0 = 0.0, w1 = 0.0, a1 = 0.0, av = 0.0, hn = 0.0, hnd = 0.0;
        const size_t i = b0 + k, ip = b0 + (k + 1 < L ? k + 1 : k);
        if (wet) {
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                vf[q] = G(a.vflux)[(size_t)(es[q].x >> 1) * L + k];
                To[q] = T[(size_t)es[q].y * L + k];
            }
            const double2 aa = ldv(m.aav, i);
            w0 = G(a.w_e)[i]; a0 = aa.x; av = aa.y;
            if (NS > 1) { w1 = G(a.w_e)[ip]; a1 = G(m.area)[ip]; }
            hn = G(a.hnn)[i]; hnd = G(a.hnode)[i];
            // the element vertices are the node and edge neighbours: the gradient below
            // reads them back from the lane's own LDS row by slot code (bits 16.. of the
            // element-slot word: 4 bits per vertex, ST = the node) instead of loading
            // them again
            if (gslot) {
#pragma unroll
                for (int q = 0; q < DM; ++q) nb[q * 64] = To[q];
                nb[ST * 64] = Tk;
            }
        }
        if (NS == 1) {
            // all lanes active here. Lanes past the loaded range hold 0, which is what
            // the two-slot body reads there; lane 63 is never used for k + 1 in one slot.
            // Tm is read on wet lanes only, where it is T[k-1], or T[0] at k = 0
            Tm = wave_prev(Tk, Tk);
            Tp = wave_next(Tk, 0.0);
            w1 = wave_next(w0, 0.0);
            a1 = wave_next(a0, 0.0);
        }
        if (!wet) continue;
        // LO: edges in reference order. Skipped terms add +0.0, which leaves a sum that
        // starts at +0.0 unchanged, so selects replace branches bit for bit.
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double v = vf[q];
            const bool side = es[q].x & 1;
            const double T1 = side ? To[q] : Tk;
            const double T2 = side ? Tk : To[q];
            const double av = fabs(v);
            const double f = -0.5 * (T1 * (v + av) + T2 * (v - av));
            const bool use = q < cnt.x && v != 0.0;
            acc = acc + (use ? (side ? -f : f) : 0.0);
        }
        double fv0, fv1 = 0.0;
        {
            const double aw = fabs(w0);
            fv0 = (-0.5 * (Tk * (w0 + aw) + Tm * (w0 - aw))) * a0;
        }
        if (in_layer(nr, k + 1)) {
            const double aw = fabs(w1);
            fv1 = (-0.5 * (Tp * (w1 + aw) + Tk * (w1 - aw))) * a1;
        }
        const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
        const double numer = Tk * hnd + (acc + (fv0 - fv1)) * a.dt / safe_a;
        const double lo = numer / safe_hn;
        G(a.LO)[jo + i] = (hn > 0.0 && av > 0.0) ? lo : 0.0;
        // gnode: elements in increasing id, only on the levels the adf_h pass reads
        if (!gslot) continue;
        double nx = 0.0, ny = 0.0, den = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const int e = el[q].x;
            const bool use = q < cnt.y && in_bytes(es[q].w, 0, k);
            const size_t g6 = 6 * (size_t)e;
            const unsigned codes = (unsigned)es[q].w >> 16;
            const double tv0 = nb[(codes & 0xf) * 64], tv1 = nb[((codes >> 4) & 0xf) * 64];
            const double tv2 = nb[((codes >> 8) & 0xf) * 64];
            const double gx = ldc(m.gs, g6) * tv0 + ldc(m.gs, g6 + 1) * tv1 + ldc(m.gs, g6 + 2) * tv2;
            const double gy = ldc(m.gs, g6 + 3) * tv0 + ldc(m.gs, g6 + 4) * tv1 + ldc(m.gs, g6 + 5) * tv2;
            const double ea = ldc(m.earea, e);
            nx = nx + (use ? gx * ea : 0.0);
            ny = ny + (use ? gy * ea : 0.0);
            den = den + (use ? ea : 0.0);
        }
        const double d = den > 0.0 ? den : 1.0;
        if (k >= glo && k < ghi) stv(a.gnode, jo + i, make_double2(nx / d, ny / d));
    }
}

template <int NS, int DM>
__device__ __forceinline__ void pass1_body(const FusedArgs& a, int n, int j, int4 hd) {
    __shared__ double s_nb[4][DM + 1][64];
    if (DM > 6 && (hd.z & 0xff) <= 6 && hd.w <= 6) pass1_slots<NS, 6, DM>(a, n, j, hd, s_nb);
    else pass1_slots<NS, DM, DM>(a, n, j, hd, s_nb);
}

// The pointer of tracer slot j0 + jj; half-wavefront columns: of j0 in lanes 0-31 and of
// j0 + 1 in lanes 32-63. (As a sum: a select became a per-lane index into the kernel's
// arguments, which put all of them into scratch memory.)
template <bool HALF, class T>
__device__ __forceinline__ gptr<T> lane_tracer(T* const* p, int j0, int jj) {
    if constexpr (HALF) {
        const uint64_t p0 = (uint64_t)p[j0], p1 = (uint64_t)p[j0 + 1];
        return (gptr<T>)(p0 + (uint64_t)(lane_id() >> 5) * (p1 - p0));
    }
    return G(p[j0 + jj]);
}

// Pass 1 of a shallow node (wet layers end above level 64, one 64-level slot) for its KT
// tracers in one wavefront: the tracer-independent loads (the edge fluxes, w, area,
// areasvol, hnode, hnode_new) are made once; per tracer the arithmetic is pass1_body's.
// KT is a compile-time count so that the tracer pointers are read at constant offsets.
// HALF: a column of at most 32 levels, interfaces included, with its two tracers in the
// wavefront's halves: half the loads, divisions and stores of a column that leaves half of
// the lanes empty, and the mesh tables stay wave-uniform. The passes cost per wavefront
// instruction more than per byte, so short columns (57 % of the nodes at nl = 47, 20 % at
// 70) gain: icosa-7 x 47, pass 1 217 -> 204 us, pass 2 273 -> 237, pass 3 222 -> 187;
// icosa-9 x 70, 2735 -> 2730, 4277 -> 3998, 3537 -> 3410. Where the wet layers pass 31 one
// tracer does not fit a half.
template <int DM, int KT, int ST, bool HALF>
__device__ __forceinline__ void pass1_shallow(const FusedArgs& a, int n, int4 hd, int j0,
                                              double (*s_nb)[ST + 1][64]) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);
    const int glo = (hd.z >> 8) & 0xff, ghi = (hd.z >> 16) & 0xff;
    const size_t b0 = (size_t)n * L;
    const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
    int4 es[DM];
    int4 el[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
        el[q] = ldc(a.tab.elem, (size_t)n * ST + q);
    }
    double* nb = &s_nb[threadIdx.x >> 6][0][lane_id()];
    const int k = col_lane<HALF>();
    const bool rd = k < kneed;
    const bool wet = in_layer(nr, k);
    const bool gslot = glo < ghi;
    const size_t i = b0 + k;
    double vf[DM] = {};
    double w0 = 0.0, a0 = 0.0, av = 0.0, hn = 0.0, hnd = 0.0;
    if (wet) {
#pragma unroll
        for (int q = 0; q < DM; ++q) vf[q] = G(a.vflux)[(size_t)(es[q].x >> 1) * L + k];
        const double2 aa = ldv(m.aav, i);
        w0 = G(a.w_e)[i]; a0 = aa.x; av = aa.y;
        hn = G(a.hnn)[i]; hnd = G(a.hnode)[i];
    }
    const double w1 = wave_next(w0, 0.0), a1 = wave_next(a0, 0.0);
#pragma unroll
    for (int jj = 0; jj < (HALF ? 1 : KT); ++jj) {
        const int j = j0 + (HALF ? lane_id() >> 5 : jj);   // tracer slot
        const auto T = lane_tracer<HALF>(a.T, j0, jj);
        const size_t jo = (size_t)j * m.N * L;
        const double Tk = rd ? T[b0 + k] : 0.0;
        double To[DM] = {};
        if (wet) {
#pragma unroll
            for (int q = 0; q < DM; ++q) To[q] = T[(size_t)es[q].y * L + k];
            if (gslot) {
#pragma unroll
                for (int q = 0; q < DM; ++q) nb[q * 64] = To[q];
                nb[ST * 64] = Tk;
            }
        }
        const double Tm = HALF ? half_prev(Tk, Tk) : wave_prev(Tk, Tk);
        const double Tp = wave_next(Tk, 0.0);
        if (!wet) continue;
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double v = vf[q];
            const bool side = es[q].x & 1;
            const double T1 = side ? To[q] : Tk;
            const double T2 = side ? Tk : To[q];
            const double aq = fabs(v);
            const double f = -0.5 * (T1 * (v + aq) + T2 * (v - aq));
            const bool use = q < cnt.x && v != 0.0;
            acc = acc + (use ? (side ? -f : f) : 0.0);
        }
        double fv0, fv1 = 0.0;
        {
            const double aw = fabs(w0);
            fv0 = (-0.5 * (Tk * (w0 + aw) + Tm * (w0 - aw))) * a0;
        }
        if (in_layer(nr, k + 1)) {
            const double aw = fabs(w1);
            fv1 = (-0.5 * (Tp * (w1 + aw) + Tk * (w1 - aw))) * a1;
        }
        const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
        const double numer = Tk * hnd + (acc + (fv0 - fv1)) * a.dt / safe_a;
        const double lo = numer / safe_hn;
        G(a.LO)[jo + i] = (hn > 0.0 && av > 0.0) ? lo : 0.0;
        if (!gslot) continue;
        double nx = 0.0, ny = 0.0, den = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const int e = el[q].x;
            const bool use = q < cnt.y && in_bytes(es[q].w, 0, k);
            const size_t g6 = 6 * (size_t)e;
            const unsigned codes = (unsigned)es[q].w >> 16;
            const double tv0 = nb[(codes & 0xf) * 64], tv1 = nb[((codes >> 4) & 0xf) * 64];
            const double tv2 = nb[((codes >> 8) & 0xf) * 64];
            const double gx = ldc(m.gs, g6) * tv0 + ldc(m.gs, g6 + 1) * tv1 + ldc(m.gs, g6 + 2) * tv2;
            const double gy = ldc(m.gs, g6 + 3) * tv0 + ldc(m.gs, g6 + 4) * tv1 + ldc(m.gs, g6 + 5) * tv2;
            const double ea = ldc(m.earea, e);
            nx = nx + (use ? gx * ea : 0.0);
            ny = ny + (use ? gy * ea : 0.0);
            den = den + (use ? ea : 0.0);
        }
        const double d = den > 0.0 ? den : 1.0;
        if (k >= glo && k < ghi) stv(a.gnode, jo + i, make_double2(nx / d, ny / d));
    }
}

template <int DM, int KT, int ST>
__device__ __forceinline__ void pass1_shallow_all(const FusedArgs& a, int n, int4 hd, int j0) {
    __shared__ double s_nb[4][ST + 1][64];
    if (KT == 2 && hd.y < 32) pass1_shallow<DM, KT, ST, true>(a, n, hd, j0, s_nb);
    else pass1_shallow<DM, KT, ST, false>(a, n, hd, j0, s_nb);
}

template <int NS, int DM>
__device__ __forceinline__ void pass1_task(const FusedArgs& a, int n, int j) {
    pass1_body<NS, DM>(a, n, j, ldc(a.tab.hdr, n));
}

// ---------------------------------------------------------------------------
// adf_h(e, k) for EPW consecutive edges, tracer j
// ---------------------------------------------------------------------------
__device__ __forceinline__ double2 grad_of(const double* gs, int el, double t0, double t1,
                                           double t2) {
    const size_t g6 = 6 * (size_t)el;
    double2 g;
    g.x = ldc(gs, g6) * t0 + ldc(gs, g6 + 1) * t1 + ldc(gs, g6 + 2) * t2;
    g.y = ldc(gs, g6 + 3) * t0 + ldc(gs, g6 + 4) * t1 + ldc(gs, g6 + 5) * t2;
    return g;
}

template <int NS, int EPW>
__device__ __forceinline__ void adfh_group(const FusedArgs& a, int g, int j) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const auto T = G(a.T[j]);
    const auto To = G(a.Told[j]);
    const double2* gn = a.gnode + (size_t)j * m.N * L;
    const auto out = G(a.adfh + (size_t)j * m.D * L);
    int e[EPW], u[EPW][2], d[EPW][2], cu[EPW], cd[EPW];
    int2 kr[EPW], nd[EPW], ur[EPW], ud[EPW];
    double2 cc[EPW];
    int kmax = 0;
#pragma unroll
    for (int q = 0; q < EPW; ++q) {
        const int eq = g * EPW + q;
        e[q] = eq < m.D ? eq : m.D - 1;
        kr[q] = eq < m.D ? ldc(a.ekr, e[q]) : make_int2(0, 0);
        nd[q] = ldc(m.edges, e[q]);
        ur[q] = ldc(m.utri_rng, e[q]);
        ud[q] = ldc(m.updn, e[q]);
        cc[q] = ldc(m.edge_c, e[q]);
        const int4 va = ldc(m.udv, 2 * (size_t)e[q]);
        const int vb = ldc(reinterpret_cast<const int*>(m.udv), 8 * (size_t)e[q] + 4);
        u[q][0] = va.x; u[q][1] = va.y; d[q][0] = va.z; d[q][1] = va.w;
        cu[q] = vb & 3; cd[q] = (vb >> 2) & 3;
    }
#pragma unroll
    for (int q = 0; q < EPW; ++q) kmax = kr[q].y > kmax ? kr[q].y : kmax;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (64 * s >= kmax) break;
        const int k = 64 * s + lane_id();
        double vf[EPW] = {}, T1[EPW] = {}, T2[EPW] = {}, O1[EPW] = {}, O2[EPW] = {};
        double tu[EPW][3] = {}, td[EPW][3] = {};
        // per edge: does any wet level of this slot use the up/dn triangle gradients
        // (nt), does any use the node gradients gnode (ng; few edges, so those loads
        // wait until the edge is computed and take no registers before)
        bool nt[EPW], ng[EPW];
#pragma unroll
        for (int q = 0; q < EPW; ++q) {
            const int lo = kr[q].x > 64 * s ? kr[q].x : 64 * s;
            const int hi = kr[q].y < 64 * s + 64 ? kr[q].y : 64 * s + 64;
            const int tl = lo > ur[q].x ? lo : ur[q].x, th = hi < ur[q].y ? hi : ur[q].y;
            nt[q] = tl < th;
            ng[q] = lo < hi && !(tl == lo && th == hi);
        }
        if (k < kmax) {
#pragma unroll
            for (int q = 0; q < EPW; ++q) {
                const size_t i1 = (size_t)nd[q].x * L + k, i2 = (size_t)nd[q].y * L + k;
                vf[q] = G(a.vflux)[(size_t)e[q] * L + k];
                T1[q] = T[i1]; T2[q] = T[i2]; O1[q] = To[i1]; O2[q] = To[i2];
                if (nt[q]) {
                    // the up triangle's vertex at slot cu is the edge's first node, the down
                    // triangle's at slot cd its second: their T is already loaded
                    const double a0 = T[(size_t)u[q][0] * L + k], a1 = T[(size_t)u[q][1] * L + k];
                    const double b0 = T[(size_t)d[q][0] * L + k], b1 = T[(size_t)d[q][1] * L + k];
                    tu[q][0] = cu[q] == 0 ? T1[q] : a0;
                    tu[q][1] = cu[q] == 0 ? a0 : (cu[q] == 1 ? T1[q] : a1);
                    tu[q][2] = cu[q] == 2 ? T1[q] : a1;
                    td[q][0] = cd[q] == 0 ? T2[q] : b0;
                    td[q][1] = cd[q] == 0 ? b0 : (cd[q] == 1 ? T2[q] : b1);
                    td[q][2] = cd[q] == 2 ? T2[q] : b1;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < EPW; ++q) {
            if (k < kr[q].x || k >= kr[q].y) continue;
            const bool tri = k >= ur[q].x && k < ur[q].y;
            const double A1 = ab2(O1[q], T1[q]), A2 = ab2(O2[q], T2[q]);
            double2 gu = make_double2(0.0, 0.0), gd = gu;
            if (nt[q]) {
                gu = grad_of(m.gs, ud[q].x, tu[q][0], tu[q][1], tu[q][2]);
                gd = grad_of(m.gs, ud[q].y, td[q][0], td[q][1], td[q][2]);
            }
            double2 ga = make_double2(0.0, 0.0), gb = ga;
            if (ng[q]) {
                ga = ldv(gn, (size_t)nd[q].x * L + k);
                gb = ldv(gn, (size_t)nd[q].y * L + k);
            }
            const double g0 = tri ? gu.x : ga.x, g1 = tri ? gd.x : gb.x;
            const double g2 = tri ? gu.y : ga.y, g3 = tri ? gd.y : gb.y;
            const double v = vf[q];
            const double av = fabs(v);
            const double flo = -0.5 * (T1[q] * (v + av) + T2[q] * (v - av));
            const double diff = A2 - A1;
            const double Tm1 = A1 + (2.0 * diff + cc[q].x * g0 + cc[q].y * g2) / 6.0;
            const double Tm2 = A2 - (2.0 * diff + cc[q].x * g1 + cc[q].y * g3) / 6.0;
            const double ho = -0.5 * ((v + av) * Tm1 + (v - av) * Tm2);
            const double r = v != 0.0 ? ho - flo : 0.0;
            out[(size_t)e[q] * L + k] = r;
        }
    }
}

// ---------------------------------------------------------------------------
// adf_h over edge patches: KT tracers, KC levels per chunk, TPE threads per edge
// ---------------------------------------------------------------------------
// A workgroup takes one edge patch (the edges a compact node patch owns). For each chunk
// of KC levels it loads (T, ttfAB) of the patch's node list into LDS, KC lanes per node
// column so that every load instruction reads whole 8*KC-byte row segments, and the
// patch's vflux likewise; then each edge's TPE threads compute its chunk levels from
// LDS (the same expressions in the same order as adfh_group, so the same bits) and leave
// adf_h in LDS, from where it is stored as row segments on the edge's wet levels. The
// loads of the next chunk are issued before the current chunk is computed, so their
// latency overlaps the arithmetic. Each node column of the patch is read from memory
// once per chunk instead of once per incident edge; only the node-averaged gradients
// (read on the few levels where an edge does not use its up/down triangles) are still
// gathered per edge.
// Keeps a 32-bit row index from being widened to one 64-bit pointer per array and item for
// the whole chunk loop: with those (and 22 to 75 registers spilled to scratch) the
// one-tracer kernel ran the icosa-7 x 70 step in 973 us, without them in 797.
__device__ __forceinline__ uint32_t opaque32(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

template <int KT, int KC, int TPE>
__device__ __forceinline__ void adfh_patch(const FusedArgs& a, int p, int j0, int seg, int nseg) {
    constexpr int NT = FCT_EP * TPE;              // threads
    constexpr int PS = FCT_PU + 1;                // row pitches padded against bank conflicts
    constexpr int ES = FCT_EP + 1;
    constexpr int NI = (FCT_PU * KC + NT - 1) / NT;   // node-column items per thread
    constexpr int NV = (FCT_EP * KC + NT - 1) / NT;   // edge-column items per thread
    constexpr int LPT = KC / TPE;                 // chunk levels per thread
    __shared__ double2 ta[KT][KC][PS];            // (T, ttfAB) of the node list
    __shared__ double vo[KT][KC][ES];             // vflux in (tracer 0's rows), adf_h out
    __shared__ int2 ekr_s[FCT_EP];
    const DevMesh& m = a.m;
    const int L = m.L;
    const int4 pt = ldc(a.tab.ep.ptab, p);
    const int first = pt.x, noff = pt.y, cnt = pt.z & 0xffff, U = pt.z >> 16;
    int klo = pt.w & 0xff, khi = (pt.w >> 8) & 0xff;
    {   // this workgroup's segment of the patch's level chunks
        const int per = ((khi - klo + KC - 1) / KC + nseg - 1) / nseg * KC;
        klo += seg * per;
        khi = khi < klo + per ? khi : klo + per;
        if (klo >= khi) return;
    }
    const int t = threadIdx.x, q = t % FCT_EP, kq = (t / FCT_EP) * LPT;
    int2 kr = make_int2(0, 0), ur = kr, nd = kr, sl = kr;
    double2 cc = make_double2(0.0, 0.0);
    double gu[6] = {}, gd[6] = {};
    if (q < cnt) {
        const int e = G(a.tab.ep.elist)[first + q];
        kr = ldv(a.ekr, e);
        ur = ldv(m.utri_rng, e);
        nd = ldv(m.edges, e);
        sl = ldv(a.tab.ep.eslot, (size_t)first + q);
        cc = ldv(m.edge_c, e);
        if (ur.x < ur.y) {
            const int2 ud = ldv(m.updn, e);
#pragma unroll
            for (int i = 0; i < 6; ++i) {
                gu[i] = G(m.gs)[6 * (size_t)ud.x + i];
                gd[i] = G(m.gs)[6 * (size_t)ud.y + i];
            }
        }
        if (t < FCT_EP) ekr_s[q] = kr;
    }
    const int s1 = sl.x & 0xff, s2 = (sl.x >> 8) & 0xff;
    const int sua = (sl.x >> 16) & 0xff, sub = (sl.x >> 24) & 0xff;
    const int sda = sl.y & 0xff, sdb = (sl.y >> 8) & 0xff;
    const int cu = (sl.y >> 16) & 3, cd = (sl.y >> 18) & 3;
    // row indices of this thread's items: node columns (slot s, level kk) and edge
    // columns (edge q, level kk), i = t + r * NT, s or q = i / KC, kk = i % KC
    uint32_t nrow[NI], erow[NV];
#pragma unroll
    for (int r = 0; r < NI; ++r) {
        const int i = t + r * NT, s = i / KC;
        nrow[r] = (s < U ? (uint32_t)G(a.tab.ep.pnodes)[noff + s] * (uint32_t)L : 0u) + i % KC;
    }
#pragma unroll
    for (int r = 0; r < NV; ++r) {
        const int i = t + r * NT, qq = i / KC;
        erow[r] = (qq < cnt ? (uint32_t)G(a.tab.ep.elist)[first + qq] * (uint32_t)L : 0u) + i % KC;
    }
    double pT[NI][KT], pO[NI][KT], pv[NV];
#define FCT_PREFETCH(K0)                                                                    \
    do {                                                                                    \
        _Pragma("unroll") for (int r = 0; r < NI; ++r) {                                    \
            const int i = t + r * NT, s = i / KC, k = (K0) + i % KC;                        \
            const bool ok = s < U && k < L;                                                 \
            _Pragma("unroll") for (int jj = 0; jj < KT; ++jj) {                             \
                pT[r][jj] = ok ? (G(a.T[j0 + jj]) + (K0))[opaque32(nrow[r])] : 0.0;              \
                pO[r][jj] = ok ? (G(a.Told[j0 + jj]) + (K0))[opaque32(nrow[r])] : 0.0;           \
            }                                                                               \
        }                                                                                   \
        _Pragma("unroll") for (int r = 0; r < NV; ++r) {                                    \
            const int i = t + r * NT, qq = i / KC, k = (K0) + i % KC;                       \
            pv[r] = (qq < cnt && k < L) ? (G(a.vflux) + (K0))[opaque32(erow[r])] : 0.0;          \
        }                                                                                   \
    } while (0)
    FCT_PREFETCH(klo);
    for (int k0 = klo; k0 < khi; k0 += KC) {
#pragma unroll
        for (int r = 0; r < NI; ++r) {
            const int i = t + r * NT, s = i / KC, kk = i % KC;
            if (s < U) {
#pragma unroll
                for (int jj = 0; jj < KT; ++jj)
                    ta[jj][kk][s] = make_double2(pT[r][jj], ab2(pO[r][jj], pT[r][jj]));
            }
        }
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int i = t + r * NT, qq = i / KC, kk = i % KC;
            if (qq < cnt) vo[0][kk][qq] = pv[r];
        }
        __syncthreads();
        if (k0 + KC < khi) FCT_PREFETCH(k0 + KC);
        if (q < cnt) {
#pragma unroll
            for (int kl = 0; kl < LPT; ++kl) {
                const int kk = kq + kl, k = k0 + kk;
                const double v = vo[0][kk][q];
                const bool wet = k >= kr.x && k < kr.y;
                const bool tri = k >= ur.x && k < ur.y;
#pragma unroll
                for (int jj = 0; jj < KT; ++jj) {
                    double r = 0.0;
                    if (wet) {
                        const double2 e1 = ta[jj][kk][s1], e2 = ta[jj][kk][s2];
                        const double T1 = e1.x, T2 = e2.x, A1 = e1.y, A2 = e2.y;
                        double g0, g1, g2, g3;
                        if (tri) {
                            const double a0 = ta[jj][kk][sua].x, a1 = ta[jj][kk][sub].x;
                            const double b0 = ta[jj][kk][sda].x, b1 = ta[jj][kk][sdb].x;
                            const double u0 = cu == 0 ? T1 : a0;
                            const double u1 = cu == 0 ? a0 : (cu == 1 ? T1 : a1);
                            const double u2 = cu == 2 ? T1 : a1;
                            const double d0 = cd == 0 ? T2 : b0;
                            const double d1 = cd == 0 ? b0 : (cd == 1 ? T2 : b1);
                            const double d2 = cd == 2 ? T2 : b1;
                            g0 = gu[0] * u0 + gu[1] * u1 + gu[2] * u2;
                            g2 = gu[3] * u0 + gu[4] * u1 + gu[5] * u2;
                            g1 = gd[0] * d0 + gd[1] * d1 + gd[2] * d2;
                            g3 = gd[3] * d0 + gd[4] * d1 + gd[5] * d2;
                        } else {
                            const double2* gn = a.gnode + (size_t)(j0 + jj) * m.N * L;
                            const double2 ga = ldv(gn, (size_t)nd.x * L + k);
                            const double2 gb = ldv(gn, (size_t)nd.y * L + k);
                            g0 = ga.x; g1 = gb.x; g2 = ga.y; g3 = gb.y;
                        }
                        const double av = fabs(v);
                        const double flo = -0.5 * (T1 * (v + av) + T2 * (v - av));
                        const double diff = A2 - A1;
                        const double Tm1 = A1 + (2.0 * diff + cc.x * g0 + cc.y * g2) / 6.0;
                        const double Tm2 = A2 - (2.0 * diff + cc.x * g1 + cc.y * g3) / 6.0;
                        const double ho = -0.5 * ((v + av) * Tm1 + (v - av) * Tm2);
                        r = v != 0.0 ? ho - flo : 0.0;
                    }
                    vo[jj][kk][q] = r;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int i = t + r * NT, qq = i / KC, kk = i % KC, k = k0 + kk;
            if (qq < cnt) {
                const int2 rr = ekr_s[qq];
                if (k >= rr.x && k < rr.y) {
#pragma unroll
                    for (int jj = 0; jj < KT; ++jj)
                        (G(a.adfh + (size_t)(j0 + jj) * m.D * L) + k0)[opaque32(erow[r])] = vo[jj][kk][qq];
                }
            }
        }
        __syncthreads();
    }
#undef FCT_PREFETCH
}

// ---------------------------------------------------------------------------
// vertical antidiffusive flux (adv_flux_ver_ho - adv_flux_ver, tracer_adv.py:241-295,
// 108-120) at interface k from the column's ttfAB at k-2..k+1 and T at k-1, k
// ---------------------------------------------------------------------------
// The three QR4C gradients of interface k are one quotient at three levels:
// qc(k) = (ttf[k-1] - ttf[k]) / nz_safe(Z[k-1] - Z[k]), qu(k) = qc(k+1), qd(k) = qc(k-1)
// (the same operands in the same order, so the same bits): the column divides once per
// level and takes qu, qd by lane shifts.
__device__ __forceinline__ double adfv_at(int k, int2 nr, double A1, double A, double Tm,
                                          double Tk, double W, double ar, double Znz,
                                          double Zm1, double qc, double qu, double qd,
                                          double zb) {
    double hi = 0.0;
    if (in_iface(nr, k)) {
        if (k == nr.x) {
            hi = -A * W * ar;
        } else if (k == nr.y) {
            hi = 0.0;
        } else if (k == nr.x + 1 || k == nr.y - 1) {
            hi = -0.5 * (A1 + A) * W * ar;
        } else if (k >= nr.x + 2 && k <= nr.y - 2) {
            const double Tmean1 = A + (2.0 * qc + qu) * (zb - Znz) / 3.0;
            const double Tmean2 = A1 + (2.0 * qc + qd) * (zb - Zm1) / 3.0;
            hi = -0.5 * (Tmean1 + Tmean2) * W * ar;
        }
    }
    double lo = 0.0;
    if (in_layer(nr, k)) {
        const double aw = fabs(W);
        lo = (-0.5 * (Tk * (W + aw) + Tm * (W - aw))) * ar;
    }
    return hi - lo;
}

// Column of adf_v for the node: every lane k <= nzmax (0 elsewhere). All lanes active.
// Also hands back areasvol at every level (loaded with the area, clamped like it).
// The column's w, area, areasvol, depth Z at k and interface depth at every lane
// (clamped below the last level): the tracer-independent inputs of adfv_column.
template <int NS, bool HALF = false>
__device__ __forceinline__ void adfv_inputs(const FusedArgs& a, int n, double (&W)[NS],
                                            double (&ar)[NS], double (&avc)[NS],
                                            double (&Zc)[NS], double (&zb)[NS]) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const size_t b0 = (size_t)n * L;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        const int kc = k < L ? k : L - 1;
        const size_t i = b0 + kc;
        W[s] = G(a.w_e)[i];
        if (a.w_i) W[s] = W[s] + G(a.w_i)[i];
        const double2 aa = ldv(m.aav, i);
        ar[s] = aa.x;
        avc[s] = aa.y;
        if (a.Z3d) {
            Zc[s] = G(a.Z3d)[i];
            zb[s] = G(a.zbar3)[i];
        } else {
            const double2 z = ldv(m.zzb, kc);
            Zc[s] = z.x;
            zb[s] = z.y;
        }
    }
}

template <int NS, bool HALF = false>
__device__ __forceinline__ void adfv_compute(const FusedArgs& a, int2 nr,
                                             const double (&Tc)[NS], const double (&Ac)[NS],
                                             const double (&W)[NS], const double (&ar)[NS],
                                             const double (&Zc)[NS], const double (&zb)[NS],
                                             double (&out)[NS]) {
    const int L = a.m.L;
    double Tm[NS], A1[NS];
    col_prev_own<NS, HALF>(Tc, Tm);
    col_prev_own<NS, HALF>(Ac, A1);
    // The reference's stencil depths (_z_stencil, tracer_adv.py:228-238) clamp Z[k-1] and
    // Z[k-2] at the top and Z[k+1] at the bottom. qc is needed at levels nr.x+1 .. nr.y-1
    // only (qd at nr.x+2 reads nr.x+1, qu at nr.y-2 reads nr.y-1): there 1 <= k <= L-2,
    // no clamp applies, and Z[k-1] is the plain lane shift of Z.
    double Zm1[NS], qc[NS], qu[NS], qd[NS];
    col_prev_own<NS, HALF>(Zc, Zm1);
#pragma unroll
    for (int s = 0; s < NS; ++s)
        qc[s] = 64 * s <= nr.y ? (A1[s] - Ac[s]) / nz_safe(Zm1[s] - Zc[s]) : 0.0;
    col_next<NS>(qc, qu, 0.0);
    col_prev<NS, HALF>(qc, qd, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        out[s] = 0.0;
        if (k <= nr.y && k < L)
            out[s] = adfv_at(k, nr, A1[s], Ac[s], Tm[s], Tc[s], W[s], ar[s], Zc[s], Zm1[s],
                             qc[s], qu[s], qd[s], zb[s]);
    }
}

template <int NS>
__device__ __forceinline__ void adfv_column(const FusedArgs& a, int n, int2 nr,
                                            const double (&Tc)[NS], const double (&Ac)[NS],
                                            double (&out)[NS], double (&avc)[NS]) {
    double W[NS], ar[NS], Zc[NS], zb[NS];
    adfv_inputs<NS>(a, n, W, ar, avc, Zc, zb);
    adfv_compute<NS>(a, nr, Tc, Ac, W, ar, Zc, zb, out);
}

// ---------------------------------------------------------------------------
// pass 2 of node n, tracer j: cluster bounds, P+/P-, limiter factors
// ---------------------------------------------------------------------------
template <int NS, int DM, int ST>
__device__ __forceinline__ void pass2_slots(const FusedArgs& a, int n, int j, int2 nr, int2 cnt) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const size_t jo = (size_t)j * m.N * L;
    const size_t b0 = (size_t)n * L;
    const auto Tb = G(a.T[j]);
    const auto LOb = G(a.LO + jo);
    const auto Tr = G(Tb + b0);
    const auto Or = G(a.Told[j] + b0);
    const auto LOr = G(LOb + b0);
    const auto adfh = G(a.adfh + (size_t)j * m.D * L);
    const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
    int4 es[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
    double Tc[NS], Ac[NS], LOc[NS], tvx[NS], tvn[NS], ap[NS], am[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        Tc[s] = 0.0; Ac[s] = 0.0; LOc[s] = 0.0;
        tvx[s] = -INFINITY; tvn[s] = INFINITY; ap[s] = 0.0; am[s] = 0.0;
        if (64 * s >= kneed) continue;
        const int k = 64 * s + lane_id();
        const bool rd = k < kneed;
        const bool wet = in_layer(nr, k);
        // own column and the neighbours' LO, T and the edges' antidiffusive fluxes,
        // loaded in one basic block
        double lnb[DM] = {}, tnb[DM] = {}, fh[DM] = {};
        double lo_own = 0.0;
        if (rd) {
            Tc[s] = Tr[k];
            Ac[s] = ab2(Or[k], Tc[s]);
            lo_own = LOr[k];
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const size_t r = (size_t)es[q].y * L + k;
                lnb[q] = LOb[r];
                tnb[q] = Tb[r];
                fh[q] = adfh[(size_t)(es[q].x >> 1) * L + k];
            }
        }
        LOc[s] = wet ? lo_own : 0.0;
        // a1-a3: max/min of (LO, T) over the vertices of the node's triangles that are
        // wet at k, and the -+1e3 pad when one of them is dry at k
        bool act = false, inact = false;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool in = in_bytes(es[q].w, 0, k);
            act = act || (q < cnt.y && in);
            inact = inact || (q < cnt.y && !in);
        }
        double mx = act ? fmax(LOc[s], Tc[s]) : -INFINITY;
        double mn = act ? fmin(LOc[s], Tc[s]) : INFINITY;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool inc = q < cnt.x && (in_bytes(es[q].z, 0, k) || in_bytes(es[q].z, 16, k));
            mx = inc ? fmax(mx, fmax(lnb[q], tnb[q])) : mx;
            mn = inc ? fmin(mn, fmin(lnb[q], tnb[q])) : mn;
        }
        mx = inact ? fmax(mx, -FCT_BIG) : mx;
        mn = inact ? fmin(mn, FCT_BIG) : mn;
        tvx[s] = rd ? mx : -INFINITY;
        tvn[s] = rd ? mn : INFINITY;
        // b1: P+/P- from the incident edges in reference order
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double f = (es[q].x & 1) ? -fh[q] : fh[q];
            const bool use = wet && q < cnt.x;
            ap[s] = ap[s] + (use ? fmax(f, 0.0) : 0.0);
            am[s] = am[s] + (use ? fmin(f, 0.0) : 0.0);
        }
    }
    double tvxm[NS], tvxp[NS], tvnm[NS], tvnp[NS];
    col_prev<NS>(tvx, tvxm, col_bcast0<NS>(tvx));
    col_next<NS>(tvx, tvxp, 0.0);
    col_prev<NS>(tvn, tvnm, col_bcast0<NS>(tvn));
    col_next<NS>(tvn, tvnp, 0.0);
    double fvc[NS], fvb[NS], avc[NS];
    adfv_column<NS>(a, n, nr, Tc, Ac, fvc, avc);
    col_next<NS>(fvc, fvb, 0.0);
    // for pass 3, which reads it instead of computing it again
    const auto Fv = G(a.adfv + jo);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        if (k <= nr.y && k < L) Fv[b0 + k] = fvc[s];
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        if (!in_layer(nr, k)) continue;
        const size_t i = b0 + k;
        const bool use_own = (k == nr.x) || (k == nr.y - 1);
        const double cmax = use_own ? tvx[s] : fmax(fmax(tvxm[s], tvx[s]), tvxp[s]);
        const double cmin = use_own ? tvn[s] : fmin(fmin(tvnm[s], tvn[s]), tvnp[s]);
        const double ttf_max = cmax - LOc[s];
        const double ttf_min = cmin - LOc[s];
        const double pos_v = fmax(fvc[s], 0.0) + fmax(-fvb[s], 0.0);
        const double neg_v = fmin(fvc[s], 0.0) + fmin(-fvb[s], 0.0);
        const double fplus = pos_v + ap[s];
        const double fminus = neg_v + am[s];
        const double av = avc[s], hn = G(a.hnn)[i];
        const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
        const double flux_pos = fplus * a.dt / safe_a / safe_hn + FCT_FLUX_EPS;
        const double flux_neg = fminus * a.dt / safe_a / safe_hn - FCT_FLUX_EPS;
        const bool valid = av > 0.0 && hn > 0.0;
        // fmin(1, x / y) is 1 wherever x / y >= 1 (rounding is monotone and 1 is a
        // double), which the signs and one comparison decide: only lanes where the
        // limiter may bind divide, and a wavefront with none skips the divisions
        const bool bp = valid && !(flux_pos > 0.0 && ttf_max >= flux_pos);
        const bool bm = valid && !(flux_neg < 0.0 && ttf_min <= flux_neg);
        double fp = 1.0, fm = 1.0;
        if (bp) fp = fmin(1.0, ttf_max / flux_pos);
        if (bm) fm = fmin(1.0, ttf_min / flux_neg);
        // (plus, minus) factor pairs, interleaved: pass 3 reads both with one load
        stv(reinterpret_cast<double2*>(a.pf), jo + i, make_double2(fp, fm));
    }
}

template <int NS, int DM>
__device__ __forceinline__ void pass2_body(const FusedArgs& a, int n, int j, int2 nr, int2 cnt) {
    // (two copies of the two-slot body in one kernel put its arrays into scratch memory:
    // 221 against 62 us for the deep columns of icosa-7 x 70, one tracer)
    if (NS == 1 && DM > 6 && cnt.x <= 6 && cnt.y <= 6) pass2_slots<NS, 6, DM>(a, n, j, nr, cnt);
    else pass2_slots<NS, DM, DM>(a, n, j, nr, cnt);
}

// Pass 2 of a shallow node (one 64-level slot) for its KT tracers in one wavefront: w,
// area, areasvol, the stencil depths and hnode_new are loaded once; per tracer the
// arithmetic is pass2_body's.
template <int DM, int KT, int ST, bool HALF>
__device__ __forceinline__ void pass2_shallow(const FusedArgs& a, int n, int2 nr, int2 cnt, int j0) {
    constexpr int NS = 1;
    const DevMesh& m = a.m;
    const int L = m.L;
    double Ws[NS], ars[NS], avs[NS], Zcs[NS], zbs[NS];
    adfv_inputs<NS, HALF>(a, n, Ws, ars, avs, Zcs, zbs);
    double hns[NS];
    {
        const int kl = col_lane<HALF>();
        hns[0] = in_layer(nr, kl) ? G(a.hnn)[(size_t)n * L + kl] : 0.0;
    }
#pragma unroll
    for (int jj = 0; jj < (HALF ? 1 : KT); ++jj) {
        const int j = j0 + (HALF ? lane_id() >> 5 : jj);   // tracer slot
        const size_t jo = (size_t)j * m.N * L;
        const size_t b0 = (size_t)n * L;
        const auto Tb = lane_tracer<HALF>(a.T, j0, jj);
        const auto LOb = G(a.LO + jo);
        const auto Tr = Tb + b0;
        const auto Or = lane_tracer<HALF>(a.Told, j0, jj) + b0;
        const auto LOr = LOb + b0;
        const auto adfh = G(a.adfh + (size_t)j * m.D * L);
        const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
        int4 es[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
        double Tc[NS], Ac[NS], LOc[NS], tvx[NS], tvn[NS], ap[NS], am[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            Tc[s] = 0.0; Ac[s] = 0.0; LOc[s] = 0.0;
            tvx[s] = -INFINITY; tvn[s] = INFINITY; ap[s] = 0.0; am[s] = 0.0;
            if (64 * s >= kneed) continue;
            const int k = 64 * s + col_lane<HALF>();
            const bool rd = k < kneed;
            const bool wet = in_layer(nr, k);
            // own column and the neighbours' LO, T and the edges' antidiffusive fluxes,
            // loaded in one basic block
            double lnb[DM] = {}, tnb[DM] = {}, fh[DM] = {};
            double lo_own = 0.0;
            if (rd) {
                Tc[s] = Tr[k];
                Ac[s] = ab2(Or[k], Tc[s]);
                lo_own = LOr[k];
#pragma unroll
                for (int q = 0; q < DM; ++q) {
                    const size_t r = (size_t)es[q].y * L + k;
                    lnb[q] = LOb[r];
                    tnb[q] = Tb[r];
                    fh[q] = adfh[(size_t)(es[q].x >> 1) * L + k];
                }
            }
            LOc[s] = wet ? lo_own : 0.0;
            // a1-a3: max/min of (LO, T) over the vertices of the node's triangles that are
            // wet at k, and the -+1e3 pad when one of them is dry at k
            bool act = false, inact = false;
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const bool in = in_bytes(es[q].w, 0, k);
                act = act || (q < cnt.y && in);
                inact = inact || (q < cnt.y && !in);
            }
            double mx = act ? fmax(LOc[s], Tc[s]) : -INFINITY;
            double mn = act ? fmin(LOc[s], Tc[s]) : INFINITY;
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const bool inc = q < cnt.x && (in_bytes(es[q].z, 0, k) || in_bytes(es[q].z, 16, k));
                mx = inc ? fmax(mx, fmax(lnb[q], tnb[q])) : mx;
                mn = inc ? fmin(mn, fmin(lnb[q], tnb[q])) : mn;
            }
            mx = inact ? fmax(mx, -FCT_BIG) : mx;
            mn = inact ? fmin(mn, FCT_BIG) : mn;
            tvx[s] = rd ? mx : -INFINITY;
            tvn[s] = rd ? mn : INFINITY;
            // b1: P+/P- from the incident edges in reference order
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const double f = (es[q].x & 1) ? -fh[q] : fh[q];
                const bool use = wet && q < cnt.x;
                ap[s] = ap[s] + (use ? fmax(f, 0.0) : 0.0);
                am[s] = am[s] + (use ? fmin(f, 0.0) : 0.0);
            }
        }
        double tvxm[NS], tvxp[NS], tvnm[NS], tvnp[NS];
        col_prev_own<NS, HALF>(tvx, tvxm);
        col_next<NS>(tvx, tvxp, 0.0);
        col_prev_own<NS, HALF>(tvn, tvnm);
        col_next<NS>(tvn, tvnp, 0.0);
        double fvc[NS], fvb[NS];
        adfv_compute<NS, HALF>(a, nr, Tc, Ac, Ws, ars, Zcs, zbs, fvc);
        col_next<NS>(fvc, fvb, 0.0);
        // for pass 3, which reads it instead of computing it again
        const auto Fv = G(a.adfv + jo);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 64 * s + col_lane<HALF>();
            if (k <= nr.y && k < L) Fv[b0 + k] = fvc[s];
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 64 * s + col_lane<HALF>();
            if (!in_layer(nr, k)) continue;
            const size_t i = b0 + k;
            const bool use_own = (k == nr.x) || (k == nr.y - 1);
            const double cmax = use_own ? tvx[s] : fmax(fmax(tvxm[s], tvx[s]), tvxp[s]);
            const double cmin = use_own ? tvn[s] : fmin(fmin(tvnm[s], tvn[s]), tvnp[s]);
            const double ttf_max = cmax - LOc[s];
            const double ttf_min = cmin - LOc[s];
            const double pos_v = fmax(fvc[s], 0.0) + fmax(-fvb[s], 0.0);
            const double neg_v = fmin(fvc[s], 0.0) + fmin(-fvb[s], 0.0);
            const double fplus = pos_v + ap[s];
            const double fminus = neg_v + am[s];
            const double av = avs[s], hn = hns[s];
            const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
            const double flux_pos = fplus * a.dt / safe_a / safe_hn + FCT_FLUX_EPS;
            const double flux_neg = fminus * a.dt / safe_a / safe_hn - FCT_FLUX_EPS;
            const bool valid = av > 0.0 && hn > 0.0;
            // fmin(1, x / y) is 1 wherever x / y >= 1 (rounding is monotone and 1 is a
            // double), which the signs and one comparison decide: only lanes where the
            // limiter may bind divide, and a wavefront with none skips the divisions
            const bool bp = valid && !(flux_pos > 0.0 && ttf_max >= flux_pos);
            const bool bm = valid && !(flux_neg < 0.0 && ttf_min <= flux_neg);
            double fp = 1.0, fm = 1.0;
            if (bp) fp = fmin(1.0, ttf_max / flux_pos);
            if (bm) fm = fmin(1.0, ttf_min / flux_neg);
            // (plus, minus) factor pairs, interleaved: pass 3 reads both with one load
            stv(reinterpret_cast<double2*>(a.pf), jo + i, make_double2(fp, fm));
        }
    }
}

template <int DM, int KT, int ST>
__device__ __forceinline__ void pass2_shallow_all(const FusedArgs& a, int n, int2 nr, int2 cnt, int j0) {
    if (KT == 2 && nr.y < 32) {
        // (keeps the two bodies' common loads from being merged across the branch, which
        // took the kernel's arguments through scratch memory: three times the pass's time)
        asm volatile("" ::: "memory");
        pass2_shallow<DM, KT, ST, true>(a, n, nr, cnt, j0);
        asm volatile("" ::: "memory");
    } else {
        pass2_shallow<DM, KT, ST, false>(a, n, nr, cnt, j0);
    }
}

template <int NS, int DM>
__device__ __forceinline__ void pass2_task(const FusedArgs& a, int n, int j) {
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);
    if (NS == 1 || nr.y < 64) pass2_body<1, DM>(a, n, j, nr, cnt);
    else pass2_body<NS, DM>(a, n, j, nr, cnt);
}

// ---------------------------------------------------------------------------
// pass 3 of node n, tracer j: limited fluxes, divergence, reconstruction
// ---------------------------------------------------------------------------
template <int NS, int DM, int ST>
__device__ __forceinline__ void pass3_slots(const FusedArgs& a, int n, int j, int2 nr, int2 cnt) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const auto T = G(a.T[j]);
    const size_t jo = (size_t)j * m.N * L;
    const double2* pm = reinterpret_cast<const double2*>(a.pf) + jo;   // (plus, minus) pairs
    const auto adfh = G(a.adfh + (size_t)j * m.D * L);
    const size_t b0 = (size_t)n * L;
    const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
    int4 es[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
    // adf_v at the node's interfaces (k <= nzmax) as pass 2 computed it
    const auto Fv = G(a.adfv + jo);
    double Tc[NS], fvc[NS], Pc[NS], Mc[NS], acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        Tc[s] = 0.0; fvc[s] = 0.0; Pc[s] = 1.0; Mc[s] = 1.0; acc[s] = 0.0;
        if (64 * s >= kneed) continue;
        const int k = 64 * s + lane_id();
        const bool wet = in_layer(nr, k);
        // T on every level of the slot (one load for the wet levels and the dry ones
        // below, which are copied)
        if (k < L) Tc[s] = T[b0 + k];
        if (k < kneed) fvc[s] = Fv[b0 + k];
        double fh[DM] = {}, po[DM] = {}, mo[DM] = {};
        if (wet) {
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                fh[q] = adfh[(size_t)(es[q].x >> 1) * L + k];
                const double2 f = ldv(pm, (size_t)es[q].y * L + k);
                po[q] = f.x;
                mo[q] = f.y;
            }
        }
        if (wet) {
            const double2 f = ldv(pm, b0 + k);
            Pc[s] = f.x;
            Mc[s] = f.y;
        }
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double f = fh[q];
            const bool side = es[q].x & 1;
            const double ae = side ? (f >= 0.0 ? fmin(po[q], Mc[s]) : fmin(mo[q], Pc[s]))
                                   : (f >= 0.0 ? fmin(Pc[s], mo[q]) : fmin(Mc[s], po[q]));
            const double fl = ae * f;
            const bool use = wet && q < cnt.x && f != 0.0;
            acc[s] = acc[s] + (use ? (side ? -fl : fl) : 0.0);
        }
    }
    double Pm[NS], Mm[NS];
    col_prev<NS>(Pc, Pm, col_bcast0<NS>(Pc));
    col_prev<NS>(Mc, Mm, col_bcast0<NS>(Mc));
    double vl[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        vl[s] = 0.0;
        if (in_iface(nr, k) && k < L) {
            const double f = fvc[s];
            double ae;
            if (k == nr.x) ae = f >= 0.0 ? Pc[s] : Mc[s];
            else ae = f >= 0.0 ? fmin(Mm[s], Pc[s]) : fmin(Pm[s], Mc[s]);
            vl[s] = ae * f;
        }
    }
    double vl1[NS];
    col_next<NS>(vl, vl1, 0.0);
    const auto LO = G(a.LO + jo);
    const auto Tn = G(a.Tnew[j]);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        if (k >= L) continue;
        const size_t i = b0 + k;
        if (!in_layer(nr, k)) {
            const double Ti = 64 * s < kneed ? Tc[s] : T[i];
            Tn[i] = Ti + 0.0;
            continue;
        }
        const double av = G(m.areasvol)[i], hn = G(a.hnn)[i], hnd = G(a.hnode)[i];
        const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
        const double Ti = Tc[s];
        const double lo_trans = -Ti * hnd + LO[i] * hn;
        const double vdiv = av > 0.0 ? (vl[s] - vl1[s]) * a.dt / safe_a : 0.0;
        const double dttf_v = lo_trans + vdiv;
        const double dttf_h = acc[s] * a.dt / safe_a;
        double del = dttf_h + dttf_v;
        del = del + Ti * (hnd - hn);
        const double dT = hn > 0.0 ? del / safe_hn : 0.0;
        Tn[i] = Ti + dT;
    }
    // levels past the slots (a shallow column taking the one-slot body): dry copies
    for (int k = 64 * NS + lane_id(); k < L; k += 64) Tn[b0 + k] = T[b0 + k] + 0.0;
}

template <int NS, int DM>
__device__ __forceinline__ void pass3_body(const FusedArgs& a, int n, int j, int2 nr, int2 cnt) {
    if (DM > 6 && cnt.x <= 6 && cnt.y <= 6) pass3_slots<NS, 6, DM>(a, n, j, nr, cnt);
    else pass3_slots<NS, DM, DM>(a, n, j, nr, cnt);
}

// Pass 3 of a shallow node (one 64-level slot) for its KT tracers in one wavefront:
// areasvol, hnode_new and hnode are loaded once; per tracer the arithmetic is
// pass3_body's.
template <int DM, int KT, int ST, bool HALF>
__device__ __forceinline__ void pass3_shallow(const FusedArgs& a, int n, int2 nr, int2 cnt, int j0) {
    constexpr int NS = 1;
    const DevMesh& m = a.m;
    const int L = m.L;
    int4 es[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
    const int kl = col_lane<HALF>();
    const bool wetl = in_layer(nr, kl);
    double av_s = 0.0, hn_s = 0.0, hnd_s = 0.0;
    if (wetl) {
        av_s = G(m.areasvol)[(size_t)n * L + kl];
        hn_s = G(a.hnn)[(size_t)n * L + kl];
        hnd_s = G(a.hnode)[(size_t)n * L + kl];
    }
#pragma unroll
    for (int jj = 0; jj < (HALF ? 1 : KT); ++jj) {
        const int j = j0 + (HALF ? lane_id() >> 5 : jj);   // tracer slot
        const auto T = lane_tracer<HALF>(a.T, j0, jj);
        const size_t jo = (size_t)j * m.N * L;
        const double2* pm = reinterpret_cast<const double2*>(a.pf) + jo;   // (plus, minus) pairs
        const auto adfh = G(a.adfh + (size_t)j * m.D * L);
        const size_t b0 = (size_t)n * L;
        const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
        // adf_v at the node's interfaces (k <= nzmax) as pass 2 computed it
        const auto Fv = G(a.adfv + jo);
        double Tc[NS], fvc[NS], Pc[NS], Mc[NS], acc[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            Tc[s] = 0.0; fvc[s] = 0.0; Pc[s] = 1.0; Mc[s] = 1.0; acc[s] = 0.0;
            if (64 * s >= kneed) continue;
            const int k = 64 * s + col_lane<HALF>();
            const bool wet = in_layer(nr, k);
            // T on every level of the slot (one load for the wet levels and the dry ones
            // below, which are copied)
            if (k < L) Tc[s] = T[b0 + k];
            if (k < kneed) fvc[s] = Fv[b0 + k];
            double fh[DM] = {}, po[DM] = {}, mo[DM] = {};
            if (wet) {
#pragma unroll
                for (int q = 0; q < DM; ++q) {
                    fh[q] = adfh[(size_t)(es[q].x >> 1) * L + k];
                    const double2 f = ldv(pm, (size_t)es[q].y * L + k);
                    po[q] = f.x;
                    mo[q] = f.y;
                }
            }
            if (wet) {
                const double2 f = ldv(pm, b0 + k);
                Pc[s] = f.x;
                Mc[s] = f.y;
            }
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const double f = fh[q];
                const bool side = es[q].x & 1;
                const double ae = side ? (f >= 0.0 ? fmin(po[q], Mc[s]) : fmin(mo[q], Pc[s]))
                                       : (f >= 0.0 ? fmin(Pc[s], mo[q]) : fmin(Mc[s], po[q]));
                const double fl = ae * f;
                const bool use = wet && q < cnt.x && f != 0.0;
                acc[s] = acc[s] + (use ? (side ? -fl : fl) : 0.0);
            }
        }
        double Pm[NS], Mm[NS];
        col_prev_own<NS, HALF>(Pc, Pm);
        col_prev_own<NS, HALF>(Mc, Mm);
        double vl[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 64 * s + col_lane<HALF>();
            vl[s] = 0.0;
            if (in_iface(nr, k) && k < L) {
                const double f = fvc[s];
                double ae;
                if (k == nr.x) ae = f >= 0.0 ? Pc[s] : Mc[s];
                else ae = f >= 0.0 ? fmin(Mm[s], Pc[s]) : fmin(Pm[s], Mc[s]);
                vl[s] = ae * f;
            }
        }
        double vl1[NS];
        col_next<NS>(vl, vl1, 0.0);
        const auto LO = G(a.LO + jo);
        const auto Tn = lane_tracer<HALF>(a.Tnew, j0, jj);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 64 * s + col_lane<HALF>();
            if (k >= L) continue;
            const size_t i = b0 + k;
            if (!in_layer(nr, k)) {
                const double Ti = 64 * s < kneed ? Tc[s] : T[i];
                Tn[i] = Ti + 0.0;
                continue;
            }
            const double av = av_s, hn = hn_s, hnd = hnd_s;
            const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
            const double Ti = Tc[s];
            const double lo_trans = -Ti * hnd + LO[i] * hn;
            const double vdiv = av > 0.0 ? (vl[s] - vl1[s]) * a.dt / safe_a : 0.0;
            const double dttf_v = lo_trans + vdiv;
            const double dttf_h = acc[s] * a.dt / safe_a;
            double del = dttf_h + dttf_v;
            del = del + Ti * (hnd - hn);
            const double dT = hn > 0.0 ? del / safe_hn : 0.0;
            Tn[i] = Ti + dT;
        }
        // levels past the slots (a shallow column taking the one-slot body): dry copies
        for (int k = (HALF ? 32 : 64) + col_lane<HALF>(); k < L; k += HALF ? 32 : 64) Tn[b0 + k] = T[b0 + k] + 0.0;
    }
}

template <int DM, int KT, int ST>
__device__ __forceinline__ void pass3_shallow_all(const FusedArgs& a, int n, int2 nr, int2 cnt, int j0) {
    if (KT == 2 && nr.y < 32) pass3_shallow<DM, KT, ST, true>(a, n, nr, cnt, j0);
    else pass3_shallow<DM, KT, ST, false>(a, n, nr, cnt, j0);
}

template <int NS, int DM>
__device__ __forceinline__ void pass3_task(const FusedArgs& a, int n, int j) {
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);
    if (NS == 1 || nr.y < 64) pass3_body<1, DM>(a, n, j, nr, cnt);
    else pass3_body<NS, DM>(a, n, j, nr, cnt);
}

// ---------------------------------------------------------------------------
// upwind-only step of node n, tracer j (advect_one, tracer_adv.py:154-165): upwind
// fluxes of ttfAB (adv_flux_hor :96-105, adv_flux_ver :108-120), flux2dtracer
// (:123-139) and ale_reconstruct (:142-151); every lane of T_new is written
// ---------------------------------------------------------------------------
template <int NS, int DM, int ST>
__device__ __forceinline__ void upwind_slots(const FusedArgs& a, int n, int j, int4 hd) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);
    const auto T = G(a.T[j]);
    const auto To = G(a.Told[j]);
    const auto Tn = G(a.Tnew[j]);
    const size_t b0 = (size_t)n * L;
    int4 es[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) es[q] = ldc(a.tab.edge, (size_t)n * ST + q);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        if (64 * s >= L) break;
        const bool wet = in_layer(nr, k);
        const size_t i = b0 + k;
        double Ti = 0.0;
        if (k < L) Ti = T[i];
        if (!wet) {
            if (k < L) Tn[i] = Ti + 0.0;
            continue;
        }
        const double A = ab2(To[i], Ti);
        const size_t im = k > 0 ? i - 1 : i;
        const double Am = ab2(To[im], T[im]);
        const bool below = in_layer(nr, k + 1);
        const double Ap = below ? ab2(To[i + 1], T[i + 1]) : 0.0;
        double vf[DM], A2[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            vf[q] = G(a.vflux)[(size_t)(es[q].x >> 1) * L + k];
            const size_t r = (size_t)es[q].y * L + k;
            A2[q] = ab2(To[r], T[r]);
        }
        double raw = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double v = vf[q];
            const bool side = es[q].x & 1;
            const double T1 = side ? A2[q] : A;
            const double T2 = side ? A : A2[q];
            const double av = fabs(v);
            const double f = -0.5 * (T1 * (v + av) + T2 * (v - av));
            const bool use = q < cnt.x && v != 0.0;
            raw = raw + (use ? (side ? -f : f) : 0.0);
        }
        double fv0, fv1 = 0.0;
        {
            const double wk = G(a.w_e)[i], aw = fabs(wk);
            fv0 = (-0.5 * (A * (wk + aw) + Am * (wk - aw))) * G(m.area)[i];
        }
        if (below) {
            const double wk = G(a.w_e)[i + 1], aw = fabs(wk);
            fv1 = (-0.5 * (Ap * (wk + aw) + A * (wk - aw))) * G(m.area)[i + 1];
        }
        const double av = G(m.areasvol)[i], hn = G(a.hnn)[i], hnd = G(a.hnode)[i];
        const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
        const double dttf_v = (fv0 - fv1) * a.dt / safe_a;
        const double dttf_h = raw * a.dt / safe_a;
        double del = dttf_h + dttf_v;
        del = del + Ti * (hnd - hn);
        const double dT = hn > 0.0 ? del / safe_hn : 0.0;
        Tn[i] = Ti + dT;
    }
}

// The same over the node's ring (NodeTab::ring), one 64-level slot s: each triangle of the
// node loaded once and its edges' volume fluxes formed here, for all K tracers, so that no
// edge flux pass runs and no flux crosses memory; the levels above and below come from the
// neighbouring lanes (and one uniform load where the slot ends). The first tracer's columns
// are in flight with the triangles. The terms go through the lane's LDS column into the
// table's 2e+side order. Bound by the vector memory path (six triangles of 24 B and twelve
// tracer columns a node) at four wavefronts per SIMD: icosa-7 x 47 187 us, 251 with
// the edge flux pass (158 + 100); 219 with the tracer's loads behind the fluxes, 258 at five
// wavefronts (spills). icosa-7 x 70 289 -> 234 us; with both slots of a column in registers
// 339.
template <bool HALO, int DM, int ST>
__device__ __forceinline__ void upwind_ring(const FusedArgs& a, int n, int4 hd, int s, double* term) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 nr = make_int2(hd.x, hd.y);
    const int k = 64 * s + lane_id();
    const size_t i = (size_t)n * L + k;
    const size_t up = (size_t)n * L + 64 * s - 1, dn = (size_t)n * L + 64 * s + 64;
    const bool has_up = HALO && s > 0, has_dn = HALO && 64 * s + 64 < nr.y;
    int4 r[DM];
    double4 cr[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) r[q] = ldc(a.tab.ring, (size_t)n * ST + q);
#pragma unroll
    for (int q = 0; q < DM; ++q) cr[q] = ldc(m.cross, r[q].z < 0 ? 0 : r[q].z >> 1);
    double Ti, Ai, T2[DM], A2[DM], Tu, Td;
    auto load = [&](int j) {
        const auto T = G(a.T[j]);
        const auto To = G(a.Told[j]);
        Ti = Ai = Tu = Td = 0.0;
        if (k < L) {
            Ti = T[i];
            Ai = To[i];
        }
        if (has_up) Tu = ab2(To[up], T[up]);
        if (has_dn) Td = ab2(To[dn], T[dn]);
        if (k < nr.y) {
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const size_t c = (size_t)r[q].x * L + k;
                T2[q] = T[c];
                A2[q] = To[c];
            }
        }
    };
    load(0);
    double vf[DM];
    {
        double2 w[DM];
        double h[DM];
        bool in[DM];
        if (k < nr.y) {
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const size_t c = (size_t)r[q].y * L + k;
                w[q] = ldv(reinterpret_cast<const double2*>(a.uv), c);
                h[q] = G(a.helem)[c];
            }
        }
#pragma unroll
        for (int q = 0; q < DM; ++q)
            in[q] = q > 0 && (r[q].w & FCT_RING_DUP) ? in[q > 0 ? q - 1 : 0] : in_bytes(r[q].w, 0, k);
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const int b = (q + DM - 1) % DM;
            const bool prev = r[q].w & FCT_RING_PREV;   // the edge's triangles: (b, q) or (q, b)
            const double xb = prev ? cr[q].x : cr[q].z, yb = prev ? cr[q].y : cr[q].w;
            const double xq = prev ? cr[q].z : cr[q].x, yq = prev ? cr[q].w : cr[q].y;
            const double tb = in[b] ? (w[b].y * xb - w[b].x * yb) * h[b] : 0.0;
            const double tq = in[q] ? (w[q].y * xq - w[q].x * yq) * h[q] : 0.0;
            vf[q] = prev ? tq - tb : tb - tq;           // (the first triangle's term is negated)
        }
    }
    // the node's own fields
    double w0 = 0.0, a0 = 0.0, av = 0.0, hn = 0.0, hnd = 0.0;
    const bool wet = in_layer(nr, k);
    if (wet) {
        const double2 aa = ldv(m.aav, i);
        w0 = G(a.w_e)[i]; a0 = aa.x; av = aa.y;
        hn = G(a.hnn)[i]; hnd = G(a.hnode)[i];
    }
    const double w1 = wave_next(w0, has_dn ? G(a.w_e)[dn] : 0.0);
    const double a1 = wave_next(a0, has_dn ? G(m.area)[dn] : 0.0);
#pragma unroll 1
    for (int j = 0;;) {
        const auto Tn = G(a.Tnew[j]);
        const double A = ab2(Ai, Ti);
        const double Am = wave_prev(A, has_up ? Tu : A);   // (level 0 takes itself)
        const double Ap = wave_next(A, Td);
        if (wet) {
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                if (r[q].z < 0) continue;
                const double v = vf[q], far = ab2(A2[q], T2[q]);
                const bool side = r[q].z & 1;
                const double x1 = side ? far : A, x2 = side ? A : far;
                const double aq = fabs(v);
                const double f = -0.5 * (x1 * (v + aq) + x2 * (v - aq));
                term[((r[q].w >> 16) & 0xf) * 64] = v != 0.0 ? (side ? -f : f) : 0.0;
            }
            double raw = 0.0;
#pragma unroll
            for (int q = 0; q < DM; ++q)
                if (q < (hd.z & 0xff)) raw = raw + term[q * 64];
            double fv0, fv1 = 0.0;
            {
                const double aw = fabs(w0);
                fv0 = (-0.5 * (A * (w0 + aw) + Am * (w0 - aw))) * a0;
            }
            if (in_layer(nr, k + 1)) {
                const double aw = fabs(w1);
                fv1 = (-0.5 * (Ap * (w1 + aw) + A * (w1 - aw))) * a1;
            }
            const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
            const double dttf_v = (fv0 - fv1) * a.dt / safe_a;
            const double dttf_h = raw * a.dt / safe_a;
            double del = dttf_h + dttf_v;
            del = del + Ti * (hnd - hn);
            const double dT = hn > 0.0 ? del / safe_hn : 0.0;
            Tn[i] = Ti + dT;
        } else if (k < L) {
            Tn[i] = Ti + 0.0;
        }
        if (++j == a.K) break;
        load(j);
    }
}

template <int NS, int DM>
__device__ __forceinline__ void upwind_task(const FusedArgs& a, int n, int j) {
    const int4 hd = ldc(a.tab.hdr, n);
    if (DM > 6 && (hd.z & 0xff) <= 6) upwind_slots<NS, 6, DM>(a, n, j, hd);
    else upwind_slots<NS, DM, DM>(a, n, j, hd);
}

// ---------------------------------------------------------------------------
// kernels: single instance (descriptor by value) and batched (descriptor array)
// ---------------------------------------------------------------------------
// Occupancy targets (wavefronts per SIMD) per kernel: the most the compiler reaches
// without spilling to scratch (node degree 8 tables need more registers); the passes
// are latency-bound, so more resident wavefronts hide more of each one's memory waits.
#define FCT_OCC(n) __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(n)))

template <int NS, int EPW>
__global__ void FCT_OCC(8) kf_vflux(FusedArgs a) {
    int w;
    if (single_wave((a.m.D + EPW - 1) / EPW, a.remap, w)) vflux_group<NS, EPW>(a, w);
}
template <int NS, int EPW>
__global__ void FCT_OCC(8) kb_vflux(const FusedArgs* __restrict__ d,
                                                const int2* __restrict__ blk, int remap) {
    int inst;
    const int w = batch_wave(blk, remap, inst);
    const FusedArgs& a = d[inst];
    if (w < (a.m.D + EPW - 1) / EPW) vflux_group<NS, EPW>(a, w);
}

template <int NS, int EPW>
__global__ void FCT_OCC(8) kf_adfh(FusedArgs a) {
    int w;
    if (!single_wave((int64_t)((a.m.D + EPW - 1) / EPW) * a.K, a.remap, w)) return;
    const int g = w / a.K;
    adfh_group<NS, EPW>(a, g, w - g * a.K);
}
template <int NS, int EPW>
__global__ void FCT_OCC(8) kb_adfh(const FusedArgs* __restrict__ d,
                                               const int2* __restrict__ blk, int remap) {
    int inst;
    const int w = batch_wave(blk, remap, inst);
    const FusedArgs& a = d[inst];
    if (w >= ((a.m.D + EPW - 1) / EPW) * a.K) return;
    const int g = w / a.K;
    adfh_group<NS, EPW>(a, g, w - g * a.K);
}

// adf_h over edge patches; KT tracers from slot j0 of the launch's tracer chunk. At most
// 128 registers per thread, 168 in the one-tracer kernel with a thread per edge: its 40 KB
// of LDS allow four workgroups per CU, but at 128 registers it spills 22 of them.
template <int KT, int KC, int TPE>
__global__ void __launch_bounds__(FCT_EP * TPE) __attribute__((amdgpu_waves_per_eu(KT == 1 && KC == 8 && TPE == 1 ? 3 : 4)))
ke_adfh(FusedArgs a, int j0, int nseg) {
    const int b = (int)block_tile(a.remap), p = b / nseg;
    adfh_patch<KT, KC, TPE>(a, p, j0, b - p * nseg, nseg);
}
// batched form: per workgroup (instance, patch | first tracer << 24 | segment << 27)
template <int KT, int KC, int TPE>
__global__ void __launch_bounds__(FCT_EP * TPE) __attribute__((amdgpu_waves_per_eu(4)))
kbe_adfh(const FusedArgs* __restrict__ d, const int2* __restrict__ blk, int remap, int nseg) {
    const int2 e = blk[block_tile(remap)];
    const int inst = __builtin_amdgcn_readfirstlane(e.x);
    const unsigned pj = (unsigned)__builtin_amdgcn_readfirstlane(e.y);
    adfh_patch<KT, KC, TPE>(d[inst], (int)(pj & 0xffffffu), (int)(pj >> 24) & 7, (int)(pj >> 27), nseg);
}

#define FCT_NODE_KERNELS(PASS, OCC)                                                     \
    template <int NS, int DM>                                                           \
    __global__ void FCT_OCC(DM == 6 ? OCC : 4) kf_##PASS(FusedArgs a) {                 \
        int w;                                                                          \
        if (!single_wave((int64_t)a.m.N * a.K, a.remap, w)) return;                       \
        const int n = w / a.K;                                                          \
        PASS##_task<NS, DM>(a, n, w - n * a.K);                                         \
    }                                                                                   \
    template <int NS, int DM>                                                           \
    __global__ void FCT_OCC(DM == 6 ? OCC : 4) kb_##PASS(const FusedArgs* __restrict__ d, \
                                                     const int2* __restrict__ blk,      \
                                                     int remap) {                         \
        int inst;                                                                       \
        const int w = batch_wave(blk, remap, inst);                                       \
        const FusedArgs& a = d[inst];                                                   \
        if (w >= a.m.N * a.K) return;                                                   \
        const int n = w / a.K;                                                          \
        PASS##_task<NS, DM>(a, n, w - n * a.K);                                         \
    }

FCT_NODE_KERNELS(upwind, 5)
FCT_NODE_KERNELS(pass1, 5)
FCT_NODE_KERNELS(pass2, 5)
FCT_NODE_KERNELS(pass3, 6)
#undef FCT_NODE_KERNELS

// The upwind step over the rings, one wavefront per node for all tracers, a 64-level slot at
// a time (occupancy on 8-slot tables, 1 % of the nodes at 8: one slot 225 us at three wavefronts,
// 235 at four, with spills; two slots 324 and 270)
template <int NS, int DM>
__global__ void FCT_OCC(DM == 8 && NS == 1 ? 3 : 4) kf_upwind_ring(FusedArgs a) {
    __shared__ double s_term[4][DM][64];
    int n;
    if (!single_wave(a.m.N, a.remap, n)) return;
    const int4 hd = ldc(a.tab.hdr, n);
    double* term = &s_term[threadIdx.x >> 6][0][lane_id()];
#pragma unroll 1
    for (int s = 0; s < NS; ++s) {
        if (NS > 1 && 64 * s >= hd.y) {       // nothing wet from here on
            for (int j = 0; j < a.K; ++j)
                for (int k = 64 * s + lane_id(); k < a.m.L; k += 64)
                    G(a.Tnew[j])[(size_t)n * a.m.L + k] = G(a.T[j])[(size_t)n * a.m.L + k] + 0.0;
            break;
        }
        if (DM > 6 && (hd.z & 0xff) <= 6) upwind_ring<(NS > 1), 6, DM>(a, n, hd, s, term);
        else upwind_ring<(NS > 1), DM, DM>(a, n, hd, s, term);
    }
}

// Passes 2 and 3 over `count` nodes of the node list from `first`, all of whose wet
// layers fit NSB slots: shallow columns (NSB = 1) run with fewer registers per
// wavefront and so more wavefronts per SIMD than the two-slot body needs.
#define FCT_LIST_KERNELS(PASS, OCC1, OCC2)                                                  template <int NSB, int DM>                                                              __global__ void FCT_OCC(DM == 6 ? (NSB == 1 ? OCC1 : OCC2) : 4)                              kl_##PASS(FusedArgs a, int first, int count) {                                          int w;                                                                                  if (!single_wave((int64_t)count * a.K, a.remap, w)) return;                              const int t = w / a.K;                                                                  const int n = ldc(a.tab.nlist, (size_t)first + t);                                      const int4 hd = ldc(a.tab.hdr, n);                                                      PASS##_body<NSB, DM>(a, n, w - t * a.K, make_int2(hd.x, hd.y),                                               make_int2(hd.z & 0xff, hd.w));                                 }

FCT_LIST_KERNELS(pass2, 7, 4)
FCT_LIST_KERNELS(pass3, 8, 6)
#undef FCT_LIST_KERNELS

// batched form: the block table maps each workgroup to (instance, first wavefront of the
// instance's shallow (deep = 0) or deep (deep = 1) node list)
#define FCT_BATCH_LIST_KERNEL(PASS, OCC1, OCC2, CALL)                                      \
    template <int NSB, int DM>                                                            \
    __global__ void FCT_OCC(DM == 6 ? (NSB == 1 ? OCC1 : OCC2) : 4)                        \
        kbl_##PASS(const FusedArgs* __restrict__ d, const int2* __restrict__ blk, int remap, \
                   int deep) {                                                            \
        int inst;                                                                         \
        const int w = batch_wave(blk, remap, inst);                                       \
        const FusedArgs& a = d[inst];                                                     \
        const int ns = a.tab.nshallow;                                                    \
        const int first = deep ? ns : 0, count = deep ? a.m.N - ns : ns;                  \
        if (w >= count * a.K) return;                                                     \
        const int t = w / a.K;                                                            \
        const int n = ldc(a.tab.nlist, (size_t)first + t);                                \
        const int4 hd = ldc(a.tab.hdr, n);                                                \
        CALL;                                                                             \
    }

FCT_BATCH_LIST_KERNEL(pass1, 5, 5, (pass1_body<NSB, DM>(a, n, w - t * a.K, hd)))
FCT_BATCH_LIST_KERNEL(pass2, 7, 4, (pass2_body<NSB, DM>(a, n, w - t * a.K, make_int2(hd.x, hd.y),
                                                        make_int2(hd.z & 0xff, hd.w))))
FCT_BATCH_LIST_KERNEL(pass3, 8, 6, (pass3_body<NSB, DM>(a, n, w - t * a.K, make_int2(hd.x, hd.y),
                                                        make_int2(hd.z & 0xff, hd.w))))
#undef FCT_BATCH_LIST_KERNEL

// one wavefront per shallow node for KT tracers from slot j0
template <int DM, int KT, int ST = DM>
__global__ void FCT_OCC(DM == 6 ? 6 : 4) kl_pass2_all(FusedArgs a, int count, int j0) {
    int w;
    if (!single_wave((int64_t)count, a.remap, w)) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    const int4 hd = ldc(a.tab.hdr, n);
    pass2_shallow_all<DM, KT, ST>(a, n, make_int2(hd.x, hd.y), make_int2(hd.z & 0xff, hd.w), j0);
}

template <int DM, int KT, int ST = DM>
__global__ void FCT_OCC(DM == 6 ? 7 : 4) kl_pass3_all(FusedArgs a, int count, int j0) {
    int w;
    if (!single_wave((int64_t)count, a.remap, w)) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    const int4 hd = ldc(a.tab.hdr, n);
    pass3_shallow_all<DM, KT, ST>(a, n, make_int2(hd.x, hd.y), make_int2(hd.z & 0xff, hd.w), j0);
}

template <int DM, int KT, int ST = DM>
__global__ void FCT_OCC(DM == 6 ? 5 : 4) kl_pass1_all(FusedArgs a, int count, int j0) {
    int w;
    if (!single_wave((int64_t)count, a.remap, w)) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    pass1_shallow_all<DM, KT, ST>(a, n, ldc(a.tab.hdr, n), j0);
}

// batched multi-tracer passes: waves over each instance's shallow node list; the block
// table's instance field carries the first tracer slot in its high 16 bits
template <int DM, int KT>
__global__ void FCT_OCC(DM == 6 ? 5 : 4) kbp_pass1(const FusedArgs* __restrict__ d,
                                                     const int2* __restrict__ blk, int remap) {
    int ij;
    const int w = batch_wave(blk, remap, ij);
    const FusedArgs& a = d[ij & 0xffff];
    if (w >= a.tab.nshallow) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    pass1_shallow_all<DM, KT, DM>(a, n, ldc(a.tab.hdr, n), ij >> 16);
}
template <int DM, int KT>
__global__ void FCT_OCC(DM == 6 ? 6 : 4) kbp_pass2(const FusedArgs* __restrict__ d,
                                                     const int2* __restrict__ blk, int remap) {
    int ij;
    const int w = batch_wave(blk, remap, ij);
    const FusedArgs& a = d[ij & 0xffff];
    if (w >= a.tab.nshallow) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    const int4 hd = ldc(a.tab.hdr, n);
    pass2_shallow_all<DM, KT, DM>(a, n, make_int2(hd.x, hd.y), make_int2(hd.z & 0xff, hd.w), ij >> 16);
}
template <int DM, int KT>
__global__ void FCT_OCC(DM == 6 ? 7 : 4) kbp_pass3(const FusedArgs* __restrict__ d,
                                                     const int2* __restrict__ blk, int remap) {
    int ij;
    const int w = batch_wave(blk, remap, ij);
    const FusedArgs& a = d[ij & 0xffff];
    if (w >= a.tab.nshallow) return;
    const int n = ldc(a.tab.nlist, (size_t)w);
    const int4 hd = ldc(a.tab.hdr, n);
    pass3_shallow_all<DM, KT, DM>(a, n, make_int2(hd.x, hd.y), make_int2(hd.z & 0xff, hd.w), ij >> 16);
}

template <int NSB, int DM>
__global__ void FCT_OCC(DM == 6 ? 8 : 4) kl_pass1(FusedArgs a, int first,
                                                                   int count) {
    int w;
    if (!single_wave((int64_t)count * a.K, a.remap, w)) return;
    const int t = w / a.K;
    const int n = ldc(a.tab.nlist, (size_t)first + t);
    pass1_body<NSB, DM>(a, n, w - t * a.K, ldc(a.tab.hdr, n));
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
// A patch's level chunks are dealt to several workgroups until a launch has about 2048 of
// them (two to three are resident per CU, so four rounds of the chip): on the pi mesh 35
// workgroups walking six chunks each took 95 us of a 108 us step, one chunk per
// workgroup 12 us; at icosa-7 (1350 patches) two segments give 1044 us per step against
// 1059 with one, and with 2048 patches or more the segments only repeat the patch's table
// loads. A launch that has fewer chunks than the chip has CUs goes to the wavefront-per-
// edge kernel instead (0 segments): icosa-4 x 48 33.8 against 38.7 us per step with one
// tracer, pi 45 against 50; icosa-5 (510 chunks) 60 against 62 with one tracer and 89
// against 88 with two, where the lines cross.
int adfh_segments(int64_t patches, int L, int kc) {
    const int chunks = (L + kc - 1) / kc;
    if (patches <= 0 || patches * chunks < 256) return 0;
    const int64_t n = (2048 + patches - 1) / patches;
    return (int)(n > chunks ? chunks : n);
}

// node pass `stage` (1, 3 or 4) over the first `count` nodes of the node list with the
// tracers taken two per wavefront (and a last one alone when K is odd)
template <int DM, int ST>
static void launch_shallow_multi(const FusedArgs& fa, const FusedTuning& t, hipStream_t s,
                                 int stage, int count) {
    const dim3 blk(64 * t.wpb), g(blocks_for(count, t.wpb));
    for (int j0 = 0; j0 < fa.K; j0 += 2) {
        const bool two = fa.K - j0 >= 2;
        if (stage == 1) {
            if (two) hipLaunchKernelGGL((kl_pass1_all<DM, 2, ST>), g, blk, 0, s, fa, count, j0);
            else hipLaunchKernelGGL((kl_pass1_all<DM, 1, ST>), g, blk, 0, s, fa, count, j0);
        } else if (stage == 3) {
            if (two) hipLaunchKernelGGL((kl_pass2_all<DM, 2, ST>), g, blk, 0, s, fa, count, j0);
            else hipLaunchKernelGGL((kl_pass2_all<DM, 1, ST>), g, blk, 0, s, fa, count, j0);
        } else {
            if (two) hipLaunchKernelGGL((kl_pass3_all<DM, 2, ST>), g, blk, 0, s, fa, count, j0);
            else hipLaunchKernelGGL((kl_pass3_all<DM, 1, ST>), g, blk, 0, s, fa, count, j0);
        }
    }
}

// node pass `stage` over the nodes [first, first + count) of the node list, every tracer
// in a wavefront of its own
template <int NSB, int DM>
static void launch_list(const FusedArgs& fa, const FusedTuning& t, hipStream_t s, int stage,
                        int first, int count) {
    if (!count) return;
    const dim3 blk(64 * t.wpb), g(blocks_for(node_waves(count, fa.K), t.wpb));
    if (stage == 1) hipLaunchKernelGGL((kl_pass1<NSB, DM>), g, blk, 0, s, fa, first, count);
    else if (stage == 3) hipLaunchKernelGGL((kl_pass2<NSB, DM>), g, blk, 0, s, fa, first, count);
    else hipLaunchKernelGGL((kl_pass3<NSB, DM>), g, blk, 0, s, fa, first, count);
}

// node pass `stage` (1, 3 or 4): over the node list where there is one (shallow columns in
// one-slot kernels, several tracers sharing a wavefront on the leading nodes of at most
// six slots; then the deep columns), else over all nodes in id order
template <int NS, int DM>
static void launch_nodes(const FusedArgs& fa, const FusedTuning& t, hipStream_t s, int stage) {
    const NodeTab& tb = fa.tab;
    if constexpr (NS == 1) {      // every plan with nl > 64 has a list
        if (!tb.nlist) {
            const dim3 blk(64 * t.wpb), g(blocks_for(node_waves(fa.m.N, fa.K), t.wpb));
            if (stage == 1) hipLaunchKernelGGL((kf_pass1<1, DM>), g, blk, 0, s, fa);
            else if (stage == 3) hipLaunchKernelGGL((kf_pass2<1, DM>), g, blk, 0, s, fa);
            else hipLaunchKernelGGL((kf_pass3<1, DM>), g, blk, 0, s, fa);
            return;
        }
    }
    const int n6 = fa.K >= 2 && t.pair ? tb.nsix : 0;
    if (n6) launch_shallow_multi<6, DM>(fa, t, s, stage, n6);
    launch_list<1, DM>(fa, t, s, stage, n6, tb.nshallow - n6);
    if (NS == 2) launch_list<2, DM>(fa, t, s, stage, tb.nshallow, fa.m.N - tb.nshallow);
}

template <int NS, int DM>
static void launch_single(const FusedArgs& fa, const FusedTuning& t, hipStream_t s, int stage) {
    const DevMesh& m = fa.m;
    const dim3 blk(64 * t.wpb);
    switch (stage) {
        case 0:
            if (t.vflux_epw == 2)
                hipLaunchKernelGGL((kf_vflux<NS, 2>), dim3(blocks_for(vflux_waves(m.D, t), t.wpb)), blk, 0, s, fa);
            else
                hipLaunchKernelGGL((kf_vflux<NS, 4>), dim3(blocks_for(vflux_waves(m.D, t), t.wpb)), blk, 0, s, fa);
            break;
        case 2:
            if (const int nseg = t.adfh_kc ? adfh_segments(fa.tab.ep.np, m.L, t.adfh_kc) : 0) {
                const dim3 g((unsigned)(fa.tab.ep.np * nseg));
                for (int j = 0; j < fa.K; j += 2) {
                    const bool two = fa.K - j >= 2;
#define FCT_KE(KC, TPE)                                                                         \
    do {                                                                                        \
        if (two) hipLaunchKernelGGL((ke_adfh<2, KC, TPE>), g, dim3(FCT_EP * TPE), 0, s, fa, j, nseg); \
        else hipLaunchKernelGGL((ke_adfh<1, KC, TPE>), g, dim3(FCT_EP * TPE), 0, s, fa, j, nseg);     \
    } while (0)
                    if (t.adfh_kc == 4) {
                        if (t.adfh_tpe == 1) FCT_KE(4, 1);
                        else if (t.adfh_tpe == 2) FCT_KE(4, 2);
                        else FCT_KE(4, 4);
                    } else {
                        if (t.adfh_tpe == 1) FCT_KE(8, 1);
                        else if (t.adfh_tpe == 2) FCT_KE(8, 2);
                        else FCT_KE(8, 4);
                    }
#undef FCT_KE
                }
            } else if (t.adfh_epw == 1)
                hipLaunchKernelGGL((kf_adfh<NS, 1>), dim3(blocks_for(adfh_waves(m.D, fa.K, t), t.wpb)), blk, 0, s, fa);
            else
                hipLaunchKernelGGL((kf_adfh<NS, 2>), dim3(blocks_for(adfh_waves(m.D, fa.K, t), t.wpb)), blk, 0, s, fa);
            break;
        default:
            launch_nodes<NS, DM>(fa, t, s, stage);
            break;
    }
}

template <int NS, int DM>
static int launch_fused_t(FusedArgs& fa, const fct_step_args* a, int kw, const FusedTuning& t,
                          hipStream_t s) {
    fa.K = 1;
    if (fa.m.D) launch_single<NS, DM>(fa, t, s, 0);
    int rc = check_launch("kf_vflux");
    if (rc) return rc;
    for (int j0 = 0; j0 < a->ntracers; j0 += kw) {
        const int K = (a->ntracers - j0) < kw ? (a->ntracers - j0) : kw;
        fa.K = K;
        for (int j = 0; j < FCT_KCHUNK; ++j) {
            const int jj = j0 + (j < K ? j : 0);
            fa.T[j] = a->T[jj]; fa.Told[j] = a->T_old[jj]; fa.Tnew[j] = a->T_new[jj];
        }
        launch_single<NS, DM>(fa, t, s, 1);
        if (a->w_i && (rc = launch_vimpl_wet(fa.m, a->w_i, a->hnode_new, a->dt, fa.LO, fa.LO, K, s)))
            return rc;
        for (int stage = 2; stage <= 4; ++stage) launch_single<NS, DM>(fa, t, s, stage);
        if ((rc = check_launch("fused passes"))) return rc;
    }
    return FCT_OK;
}

static bool tuning_ok(const FusedTuning& t) {
    return (t.wpb == 1 || t.wpb == 2 || t.wpb == 4) && (t.vflux_epw == 2 || t.vflux_epw == 4) &&
           (t.adfh_epw == 1 || t.adfh_epw == 2) && t.xcd >= 1 &&
           (t.adfh_kc == 0 || t.adfh_kc == 4 || t.adfh_kc == 8) &&
           (t.adfh_tpe == 1 || t.adfh_tpe == 2 || t.adfh_tpe == 4);
}

static void base_args(FusedArgs& fa, const DevMesh& m, const NodeTab& tab, const int2* ekr,
                      const fct_step_args* a, const FusedTuning& tune, double* vflux, double* LO,
                      double* gnode, double* adfh, double* pf, double* adfv) {
    fa.m = m; fa.tab = tab; fa.vflux = vflux; fa.ekr = ekr; fa.uv = a->uv; fa.helem = a->helem;
    fa.w_e = a->w_e; fa.w_i = a->w_i; fa.hnode = a->hnode; fa.hnn = a->hnode_new; fa.Z3d = a->Z3d;
    fa.zbar3 = a->zbar3; fa.dt = a->dt; fa.remap = tune.remap(); fa.K = 0;
    fa.LO = LO; fa.gnode = (double2*)gnode; fa.adfh = adfh; fa.pf = pf; fa.adfv = adfv;
}

int launch_fused(const DevMesh& m, const NodeTab& tab, const int2* ekr, const fct_step_args* a,
                 int kw, const FusedTuning& tune, double* vflux, double* LO, double* gnode,
                 double* adfh, double* pf, double* adfv, hipStream_t s) {
    if (!tuning_ok(tune)) return set_error(FCT_E_INVALID, "bad launch-shape knobs");
    FusedArgs fa;
    base_args(fa, m, tab, ekr, a, tune, vflux, LO, gnode, adfh, pf, adfv);
    if (kw > FCT_KCHUNK) kw = FCT_KCHUNK;
    if (tab.dm == 6 && m.L <= 64) return launch_fused_t<1, 6>(fa, a, kw, tune, s);
    if (tab.dm == 6 && m.L <= 128) return launch_fused_t<2, 6>(fa, a, kw, tune, s);
    if (tab.dm == 8 && m.L <= 64) return launch_fused_t<1, 8>(fa, a, kw, tune, s);
    if (tab.dm == 8 && m.L <= 128) return launch_fused_t<2, 8>(fa, a, kw, tune, s);
    return set_error(FCT_E_UNSUPPORTED, "fused path supports node degree <= 8 and nl <= 128");
}

template <int NS, int DM>
static int launch_tape_t(FusedArgs& fa, const fct_step_args* a, int j0, int K, const FusedTuning& t,
                         const FusedTape& tp, hipStream_t s) {
    fa.K = 1;
    if (j0 == 0 && fa.m.D) launch_single<NS, DM>(fa, t, s, 0);
    fa.K = K;
    for (int j = 0; j < FCT_KCHUNK; ++j) {
        const int jj = j0 + (j < K ? j : 0);
        fa.T[j] = a->T[jj]; fa.Told[j] = a->T_old[jj]; fa.Tnew[j] = nullptr;
    }
    if (a->w_i) fa.LO = tp.LOx;
    launch_single<NS, DM>(fa, t, s, 1);
    if (a->w_i) {
        const int rc = launch_vimpl_wet(fa.m, a->w_i, a->hnode_new, a->dt, tp.LOx, tp.LO, K, s);
        if (rc) return rc;
        fa.LO = tp.LO;
    }
    for (int stage = 2; stage <= 3; ++stage) launch_single<NS, DM>(fa, t, s, stage);
    return check_launch("adjoint tape");
}

int launch_tape(const DevMesh& m, const NodeTab& tab, const int2* ekr, const fct_step_args* a,
                int j0, int K, const FusedTuning& tune, const FusedTape& tp, hipStream_t s) {
    if (!tuning_ok(tune)) return set_error(FCT_E_INVALID, "bad launch-shape knobs");
    FusedArgs fa;
    base_args(fa, m, tab, ekr, a, tune, tp.vflux, tp.LO, tp.gnode, tp.adfh, tp.pf, tp.adfv);
    if (tab.dm == 6) return m.L <= 64 ? launch_tape_t<1, 6>(fa, a, j0, K, tune, tp, s)
                                      : launch_tape_t<2, 6>(fa, a, j0, K, tune, tp, s);
    return m.L <= 64 ? launch_tape_t<1, 8>(fa, a, j0, K, tune, tp, s)
                     : launch_tape_t<2, 8>(fa, a, j0, K, tune, tp, s);
}

int launch_vflux_fused(const DevMesh& m, const NodeTab& tab, const int2* ekr, const double* uv,
                       const double* helem, const FusedTuning& tune, double* vflux,
                       hipStream_t s) {
    if (!tuning_ok(tune)) return set_error(FCT_E_INVALID, "bad launch-shape knobs");
    if (!m.D) return FCT_OK;
    FusedArgs fa{};
    fa.m = m; fa.tab = tab; fa.ekr = ekr; fa.uv = uv; fa.helem = helem; fa.vflux = vflux;
    fa.remap = tune.remap(); fa.K = 1;
    if (m.L <= 64) launch_single<1, 8>(fa, tune, s, 0);      // (the edge pass reads no node table)
    else launch_single<2, 8>(fa, tune, s, 0);
    return check_launch("kf_vflux");
}

template <int NS, int DM>
static int launch_upwind_t(FusedArgs& fa, const fct_step_args* a, const FusedTuning& t,
                           hipStream_t s) {
    const DevMesh& m = fa.m;
    fa.K = 1;
    // (meshes with a node whose triangles make no ring: fluxes once per edge into memory)
    if (m.D && !fa.tab.ring_flux) launch_single<NS, DM>(fa, t, s, 0);
    int rc = check_launch("kf_vflux");
    if (rc) return rc;
    for (int j0 = 0; j0 < a->ntracers; j0 += FCT_KCHUNK) {
        const int K = (a->ntracers - j0) < FCT_KCHUNK ? (a->ntracers - j0) : FCT_KCHUNK;
        fa.K = K;
        for (int j = 0; j < FCT_KCHUNK; ++j) {
            const int jj = j0 + (j < K ? j : 0);
            fa.T[j] = a->T[jj]; fa.Told[j] = a->T_old[jj]; fa.Tnew[j] = a->T_new[jj];
        }
        if (fa.tab.ring_flux)
            hipLaunchKernelGGL((kf_upwind_ring<NS, DM>), dim3(blocks_for(m.N, t.wpb)), dim3(64 * t.wpb), 0, s, fa);
        else
            hipLaunchKernelGGL((kf_upwind<NS, DM>), dim3(blocks_for(node_waves(m.N, K), t.wpb)), dim3(64 * t.wpb), 0, s, fa);
        if ((rc = check_launch("kf_upwind"))) return rc;
    }
    return FCT_OK;
}

int launch_upwind(const DevMesh& m, const NodeTab& tab, const int2* ekr, const fct_step_args* a,
                  const FusedTuning& tune, double* vflux, hipStream_t s) {
    if (!tuning_ok(tune)) return set_error(FCT_E_INVALID, "bad launch-shape knobs");
    FusedArgs fa;
    base_args(fa, m, tab, ekr, a, tune, vflux, nullptr, nullptr, nullptr, nullptr, nullptr);
    if (tab.dm == 6 && m.L <= 64) return launch_upwind_t<1, 6>(fa, a, tune, s);
    if (tab.dm == 6 && m.L <= 128) return launch_upwind_t<2, 6>(fa, a, tune, s);
    if (tab.dm == 8 && m.L <= 64) return launch_upwind_t<1, 8>(fa, a, tune, s);
    if (tab.dm == 8 && m.L <= 128) return launch_upwind_t<2, 8>(fa, a, tune, s);
    return set_error(FCT_E_UNSUPPORTED, "upwind path supports node degree <= 8 and nl <= 128");
}

size_t fused_args_size() { return sizeof(FusedArgs); }

int fill_fused_args(void* out, const DevMesh& m, const NodeTab& tab, const int2* ekr,
                    const fct_step_args* a, const FusedTuning& tune, double* vflux, double* LO,
                    double* gnode, double* adfh, double* pf, double* adfv) {
    if (a->ntracers > FCT_KCHUNK)
        return set_error(FCT_E_UNSUPPORTED, "batched instances take at most %d tracers", FCT_KCHUNK);
    FusedArgs fa;
    base_args(fa, m, tab, ekr, a, tune, vflux, LO, gnode, adfh, pf, adfv);
    fa.K = a->ntracers;
    for (int j = 0; j < FCT_KCHUNK; ++j) {
        const int jj = j < fa.K ? j : 0;
        fa.T[j] = a->T[jj]; fa.Told[j] = a->T_old[jj]; fa.Tnew[j] = a->T_new[jj];
    }
    memcpy(out, &fa, sizeof(fa));
    return FCT_OK;
}

template <int NS, int DM>
static void launch_batch_t(const BatchGroup& g, const FusedTuning& t, hipStream_t s) {
    const dim3 blk(64 * t.wpb);
    if (g.nb_v) {
        if (t.vflux_epw == 2)
            hipLaunchKernelGGL((kb_vflux<NS, 2>), dim3(g.nb_v), blk, 0, s, g.desc, g.blk_v, t.remap());
        else
            hipLaunchKernelGGL((kb_vflux<NS, 4>), dim3(g.nb_v), blk, 0, s, g.desc, g.blk_v, t.remap());
    }
    const bool split = NS == 2 && g.blk_ns;
    if (g.nb_pa) hipLaunchKernelGGL((kbp_pass1<DM, 2>), dim3(g.nb_pa), blk, 0, s, g.desc, g.blk_pa, t.remap());
    if (g.nb_p1) hipLaunchKernelGGL((kbp_pass1<DM, 1>), dim3(g.nb_p1), blk, 0, s, g.desc, g.blk_p1, t.remap());
    if (split) {
        if (g.nb_ns) hipLaunchKernelGGL((kbl_pass1<1, DM>), dim3(g.nb_ns), blk, 0, s, g.desc, g.blk_ns, t.remap(), 0);
        if (g.nb_nd) hipLaunchKernelGGL((kbl_pass1<2, DM>), dim3(g.nb_nd), blk, 0, s, g.desc, g.blk_nd, t.remap(), 1);
    } else if (g.nb_n) {
        hipLaunchKernelGGL((kb_pass1<NS, DM>), dim3(g.nb_n), blk, 0, s, g.desc, g.blk_n, t.remap());
    }
    if (g.nb_e2 || g.nb_e1) {
#define FCT_KBE(KC, TPE)                                                                            \
    do {                                                                                            \
        if (g.nb_e2) hipLaunchKernelGGL((kbe_adfh<2, KC, TPE>), dim3(g.nb_e2), dim3(FCT_EP * TPE), 0, s, \
                                        g.desc, g.blk_e2, t.remap(), g.nseg2);                               \
        if (g.nb_e1) hipLaunchKernelGGL((kbe_adfh<1, KC, TPE>), dim3(g.nb_e1), dim3(FCT_EP * TPE), 0, s, \
                                        g.desc, g.blk_e1, t.remap(), g.nseg1);                               \
    } while (0)
        if (t.adfh_kc == 4) {
            if (t.adfh_tpe == 1) FCT_KBE(4, 1);
            else if (t.adfh_tpe == 2) FCT_KBE(4, 2);
            else FCT_KBE(4, 4);
        } else {
            if (t.adfh_tpe == 1) FCT_KBE(8, 1);
            else if (t.adfh_tpe == 2) FCT_KBE(8, 2);
            else FCT_KBE(8, 4);
        }
#undef FCT_KBE
    }
    if (g.nb_a) {
        if (t.adfh_epw == 1)
            hipLaunchKernelGGL((kb_adfh<NS, 1>), dim3(g.nb_a), blk, 0, s, g.desc, g.blk_a, t.remap());
        else
            hipLaunchKernelGGL((kb_adfh<NS, 2>), dim3(g.nb_a), blk, 0, s, g.desc, g.blk_a, t.remap());
    }
    if (g.nb_pa) hipLaunchKernelGGL((kbp_pass2<DM, 2>), dim3(g.nb_pa), blk, 0, s, g.desc, g.blk_pa, t.remap());
    if (g.nb_p1) hipLaunchKernelGGL((kbp_pass2<DM, 1>), dim3(g.nb_p1), blk, 0, s, g.desc, g.blk_p1, t.remap());
    if (split) {
        if (g.nb_ns) hipLaunchKernelGGL((kbl_pass2<1, DM>), dim3(g.nb_ns), blk, 0, s, g.desc, g.blk_ns, t.remap(), 0);
        if (g.nb_nd) hipLaunchKernelGGL((kbl_pass2<2, DM>), dim3(g.nb_nd), blk, 0, s, g.desc, g.blk_nd, t.remap(), 1);
    } else if (g.nb_n) {
        hipLaunchKernelGGL((kb_pass2<NS, DM>), dim3(g.nb_n), blk, 0, s, g.desc, g.blk_n, t.remap());
    }
    if (g.nb_pa) hipLaunchKernelGGL((kbp_pass3<DM, 2>), dim3(g.nb_pa), blk, 0, s, g.desc, g.blk_pa, t.remap());
    if (g.nb_p1) hipLaunchKernelGGL((kbp_pass3<DM, 1>), dim3(g.nb_p1), blk, 0, s, g.desc, g.blk_p1, t.remap());
    if (split) {
        if (g.nb_ns) hipLaunchKernelGGL((kbl_pass3<1, DM>), dim3(g.nb_ns), blk, 0, s, g.desc, g.blk_ns, t.remap(), 0);
        if (g.nb_nd) hipLaunchKernelGGL((kbl_pass3<2, DM>), dim3(g.nb_nd), blk, 0, s, g.desc, g.blk_nd, t.remap(), 1);
    } else if (g.nb_n) {
        hipLaunchKernelGGL((kb_pass3<NS, DM>), dim3(g.nb_n), blk, 0, s, g.desc, g.blk_n, t.remap());
    }
}

int launch_batch_group(const BatchGroup& g, const FusedTuning& t, hipStream_t s) {
    if (!tuning_ok(t)) return set_error(FCT_E_INVALID, "bad launch-shape knobs");
    if (g.dm == 6 && g.ns == 1) launch_batch_t<1, 6>(g, t, s);
    else if (g.dm == 6 && g.ns == 2) launch_batch_t<2, 6>(g, t, s);
    else if (g.dm == 8 && g.ns == 1) launch_batch_t<1, 8>(g, t, s);
    else if (g.dm == 8 && g.ns == 2) launch_batch_t<2, 8>(g, t, s);
    else return set_error(FCT_E_UNSUPPORTED, "batch group (%d slots, degree %d)", g.ns, g.dm);
    return check_launch("batched fused passes");
}

}  // namespace fct
