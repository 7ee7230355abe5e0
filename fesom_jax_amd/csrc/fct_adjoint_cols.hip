// Reverse mode of one FCT step for meshes with the fused node tables: the chain rule of
// fct_adjoint.hip (same conventions, same formulas) on the fused path's tape, one
// wavefront per node, edge or triangle column with lane = level.
//
// The flat form (one thread per entity and level, a kernel per stage) ran 26 kernels per
// tracer, each dividing 64-bit indices, walking the CSR lists per thread and storing every
// intermediate cotangent. Here the column is a wavefront: tables come through scalar loads,
// a node's neighbour columns are loaded together, terms that couple levels move between
// lanes, and everything a node owns stays in registers between the stages. The elements
// around a node are taken from a ring of its neighbours (a triangle joins two consecutive
// slots), so that their vertices are registers at fixed indices; through LDS rows indexed by
// slot codes kc_vertex took 376 us per tracer of icosa-7 x 47 instead of 259. An edge hands
// on two numbers and the sign of its flux (a bit per level) instead of eight: kc_edge 395
// -> 301 us. icosa-7 x 47, two tracers: 7.60 -> 3.39 ms (tape 0.79; two tracers per launch and
// short columns in halves, below, included); with the split at icosa-6 x 70: 5.38 -> 1.54 ms.
//
//   kc_ghsc   (node)  cotangent of the horizontal divergence, read by edges and neighbours
//   kc_limit  (node)  limited fluxes, limiter factors, P+/P-, cluster bounds, QR4C, and the
//                     shares of the tied elements: ka_final, ka_vlim, ka_hlim, ka_fac,
//                     ka_adfv, ka_qr, ka_share in one pass
//   kc_vertex (node)  vertex cotangents of the bounds, then LO and its vertical flux:
//                     ka_vertex, ka_lo, ka_fv (under the implicit split the last two are
//                     kc_split, after the column solve's transpose)
//   kc_edge   (edge)  ka_adfh and ka_edge; triangle gradients recomputed from T
//   kc_gnum   (node)  the node-averaged gradients' cotangents, on their few levels
//   kc_tr     (triangle) ka_tr
//   kc_gather (node)  ka_node_edges and ka_node_final
//   kc_uv     (triangle) ka_uv, once for all tracers
//   kc_add    (flat)  small meshes, where a launch takes two tracers (grid.y): the odd
//                     tracers' w cotangents onto the even ones'
//
// Like the forward passes the kernels are bound by the vector memory path (a 64-lane load
// costs 25 to 36 clocks of a CU, hit or not): kc_limit makes 30 neighbour loads per node,
// kc_vertex 24, kc_edge 16 loads per edge. The tape's values and decisions are the forward
// path's bits (recomputed in the same order), so the branches of the chain rule are too;
// sums run in table order and agree with the flat form to rounding.

#include <type_traits>

#include "fct_wave.h"

namespace fct {

namespace {

__device__ __forceinline__ double gmax_x(double g, double x, double y) {
    return x > y ? g : (x == y ? 0.5 * g : 0.0);
}
__device__ __forceinline__ double gmin_x(double g, double x, double y) {
    return x < y ? g : (x == y ? 0.5 * g : 0.0);
}
__device__ __forceinline__ double gabs(double g, double x) { return x >= 0.0 ? g : -g; }

struct ColArgs {
    DevMesh m;
    NodeTab tab;
    const int2* ekr;
    int remap, first;             // first: gw, gwi, g_vf are written, not added to
    double dt;
    const double *helem, *w_e, *w_i, *Z3d, *zbar3, *hnode, *hnn;
    const double *T, *Told, *g_out;
    double *gT, *gTold;
    // the tape of this tracer (fused path): wet lanes only, adf_v on k <= nzmax
    const double *vflux, *LO, *adfh, *adfv;
    const double2 *pm, *gnode;
    // cotangents: node columns (wet lanes unless said otherwise)
    double* ghsc;                 // [N][L]
    double2 *gpm;                 // of P+/P-
    double2 *tv, *sh;             // node bounds (max, min) and their shares per tied element
    double2 *gd;                  // (ghsc, LO divergence)
    double *gA, *gadfv, *gLO;
    double2 *gnum;
    // edge columns: what the upwind end's A and T take (one of the two ends has none, so
    // that and the sign of vflux are all an edge hands on), vflux; bit l of edge_up[e][s]
    // says that vflux >= 0 at level 64 * s + l
    double2* eg;
    double* g_vf;
    uint64_t* edge_up;
    double2* g_tr;                // [E][L]
    double *gw, *gwi;             // every lane; may be null
    const int *ud_off, *ud_ent, *et_off, *et_ent;
    // a launch over two tracers (gridDim.y = 2): the second one's fields, its w cotangents
    // (added to the first's at the end), its edge cotangent as kc_uv reads it, and the
    // distance to its workspace (doubles)
    const double *T1, *Told1, *g_out1, *g_vf1;
    double *gT1, *gTold1, *gw1, *gwi1;
    size_t node_stride, edge_stride, elem_stride;
};

// the arguments of this workgroup's tracer
__device__ __forceinline__ ColArgs of_tracer(ColArgs a) {
    if (blockIdx.y == 0) return a;
    const size_t NL = (size_t)a.m.N * a.m.L, DL = (size_t)a.m.D * a.m.L;
    a.T = a.T1; a.Told = a.Told1; a.g_out = a.g_out1;
    a.gT = a.gT1; a.gTold = a.gTold1; a.gw = a.gw1; a.gwi = a.gwi1;
    a.LO += NL; a.adfh += DL; a.adfv += NL; a.pm += NL; a.gnode += NL;
    const size_t d = a.node_stride, d2 = d / 2;
    a.ghsc += d; a.gA += d; a.gadfv += d; a.gLO += d;
    a.gpm += d2; a.tv += d2; a.sh += d2; a.gd += d2; a.gnum += d2;
    a.eg += a.edge_stride / 2;
    a.g_vf += a.edge_stride;
    a.edge_up += (size_t)a.m.D * (a.m.L <= 64 ? 1 : 2);
    a.g_tr += a.elem_stride / 2;
    return a;
}

// the arguments of this lane's tracer, where a short column's two tracers share a wavefront
// (lane = 32 * tracer + level)
__device__ __forceinline__ ColArgs of_half(ColArgs a) {
    const size_t h = lane_id() >> 5;
    const auto to = [&](auto& p, auto q) {
        p = (std::decay_t<decltype(p)>)((uint64_t)p + h * ((uint64_t)q - (uint64_t)p));
    };
    to(a.T, a.T1); to(a.Told, a.Told1); to(a.g_out, a.g_out1);
    to(a.gT, a.gT1); to(a.gTold, a.gTold1); to(a.gw, a.gw1); to(a.gwi, a.gwi1);
    const size_t NL = h * a.m.N * a.m.L, DL = h * a.m.D * a.m.L;
    a.LO += NL; a.adfh += DL; a.adfv += NL; a.pm += NL; a.gnode += NL;
    const size_t d = h * a.node_stride, d2 = d / 2;
    a.ghsc += d; a.gA += d; a.gadfv += d; a.gLO += d;
    a.gpm += d2; a.tv += d2; a.sh += d2; a.gd += d2; a.gnum += d2;
    a.eg += h * a.edge_stride / 2;
    a.g_vf += h * a.edge_stride;
    a.edge_up += h * a.m.D * (a.m.L <= 64 ? 1 : 2);
    a.g_tr += h * a.elem_stride / 2;
    return a;
}

// the wavefront's node: of the node list from `first` where there is one
__device__ __forceinline__ bool node_task(const ColArgs& a, int first, int count, int& n) {
    int w;
    if (!single_wave(count, a.remap, w)) return false;
    n = a.tab.nlist ? ldc(a.tab.nlist, (size_t)first + w) : w;
    return true;
}

// ---- R1: cotangent of the horizontal divergence (tracer_adv.py:469-484) ----------
// four nodes per wavefront, their loads together
constexpr int GH_NODES = 4;
__device__ __forceinline__ void ghsc_body(const ColArgs& a, int w) {
    const DevMesh& m = a.m;
    const int L = m.L;
    for (int k = lane_id(); k < L; k += 64) {
        double g[GH_NODES], hn[GH_NODES], av[GH_NODES];
        bool wet[GH_NODES];
#pragma unroll
        for (int q = 0; q < GH_NODES; ++q) {
            const int n = w * GH_NODES + q;
            wet[q] = n < m.N && in_layer(ldc(m.nlev, n < m.N ? n : 0), k);
            const size_t i = (size_t)n * L + k;
            g[q] = wet[q] ? G(a.g_out)[i] : 0.0;
            hn[q] = wet[q] ? G(a.hnn)[i] : 0.0;
            av[q] = wet[q] ? G(m.areasvol)[i] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < GH_NODES; ++q) {
            const int n = w * GH_NODES + q;
            const double r = (hn[q] > 0.0 ? g[q] / hn[q] : 0.0) / (av[q] > 0.0 ? av[q] : 1.0) * a.dt;
            if (wet[q]) G(a.ghsc)[(size_t)n * L + k] = r;
        }
    }
}

// ---- R2: everything of the limiter that a node owns ------------------------------
template <int NS, int DM, bool HALF>
__device__ __forceinline__ void limit_body(const ColArgs& a, int n) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y);
    const int ne = hd.z & 0xff;     // incident edges
    const size_t b0 = (size_t)n * L;
    const int kneed = nr.y + 1 < L ? nr.y + 1 : L;
    int4 es[DM];
    int2 rg[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        es[q] = ldc(a.tab.edge, (size_t)n * DM + q);
        const int4 r = ldc(a.tab.ring, (size_t)n * DM + q);
        rg[q] = make_int2(r.x, r.w & 0xffff);
    }
    double Tc[NS], Ac[NS], LOc[NS], tvx[NS], tvn[NS], ap[NS], am[NS], hp[NS], hm[NS];
    double P[NS], M[NS], fv[NS], gx[NS], cx[NS], cn[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        Tc[s] = Ac[s] = LOc[s] = ap[s] = am[s] = hp[s] = hm[s] = fv[s] = gx[s] = 0.0;
        tvx[s] = -INFINITY; tvn[s] = INFINITY;
        P[s] = M[s] = cx[s] = cn[s] = 1.0;
        if (64 * s >= kneed) continue;
        const int k = 64 * s + col_lane<HALF>();
        const bool wet = in_layer(nr, k);
        const size_t i = b0 + k;
        if (k < kneed) {
            Tc[s] = G(a.T)[i];
            Ac[s] = ab2(G(a.Told)[i], Tc[s]);
            fv[s] = G(a.adfv)[i];
        }
        double lo[DM] = {}, t[DM] = {}, fh[DM] = {}, gs[DM] = {};
        double2 pq[DM] = {};
        double g_own = 0.0, av = 0.0;
        if (wet) {
            LOc[s] = G(a.LO)[i];
            const double2 f = ldv(a.pm, i);
            P[s] = f.x; M[s] = f.y;
            g_own = G(a.ghsc)[i];
            av = G(m.areasvol)[i];
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const size_t r = (size_t)es[q].y * L + k;
                fh[q] = G(a.adfh)[(size_t)(es[q].x >> 1) * L + k];
                gs[q] = G(a.ghsc)[r];
                pq[q] = ldv(a.pm, r);
                const size_t p = (size_t)rg[q].x * L + k;
                lo[q] = G(a.LO)[p];
                t[q] = G(a.T)[p];
            }
            const double wxo = fmax(LOc[s], Tc[s]), wno = fmin(LOc[s], Tc[s]);
            // a2, a3: node bounds over the elements, and how many attain them
            double ex[DM], en[DM];
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const int q1 = (q + 1) % DM;
                const bool in = in_bytes(rg[q].y, 0, k);
                ex[q] = fmax(fmax(wxo, fmax(lo[q], t[q])), fmax(lo[q1], t[q1]));
                en[q] = fmin(fmin(wno, fmin(lo[q], t[q])), fmin(lo[q1], t[q1]));
                // triangles that are dry here pad the bounds
                ex[q] = in ? ex[q] : -FCT_BIG;
                en[q] = in ? en[q] : FCT_BIG;
                if (rg[q].y) {
                    tvx[s] = fmax(tvx[s], ex[q]);
                    tvn[s] = fmin(tvn[s], en[q]);
                }
            }
            cx[s] = cn[s] = 0.0;
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                cx[s] += rg[q].y && ex[q] == tvx[s] ? 1.0 : 0.0;
                cn[s] += rg[q].y && en[q] == tvn[s] ? 1.0 : 0.0;
            }
            // b1 sums (the forward pass's order), and the factors' cotangents of the
            // horizontal fluxes
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const bool use = q < ne, side = es[q].x & 1;
                const double f = side ? -fh[q] : fh[q];
                ap[s] = ap[s] + (use ? fmax(f, 0.0) : 0.0);
                am[s] = am[s] + (use ? fmin(f, 0.0) : 0.0);
                const bool pos = fh[q] >= 0.0;
                // (a neighbour that is dry here holds no values)
                const bool wet_e = in_bytes(es[q].z, 0, k) || in_bytes(es[q].z, 16, k);
                const double g = use && wet_e ? (side ? gs[q] - g_own : g_own - gs[q]) * fh[q] : 0.0;
                // the node's own factor is P where the flux enters it
                const bool own_p = pos != side;
                const double mine = own_p ? P[s] : M[s];
                const double theirs = own_p ? pq[q].y : pq[q].x;
                const double ga = gmin_x(g, mine, theirs);
                hp[s] += own_p ? ga : 0.0;
                hm[s] += own_p ? 0.0 : ga;
            }
        }
        // dry vertices never meet a wet element; at interface nzmax the column's own bounds
        // are not read
        gx[s] = wet && av > 0.0 ? g_own : 0.0;
    }
    // limited vertical fluxes (:453-459): interface k's cotangent goes to the factors of
    // levels k and k-1
    double gxm[NS], Pm[NS], Mm[NS], gva[NS], gp[NS], gm[NS], gpp[NS], gmp[NS], nx[NS];
    col_prev<NS, HALF>(gx, gxm, 0.0);
    col_prev<NS, HALF>(P, Pm, 1.0);
    col_prev<NS, HALF>(M, Mm, 1.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        const double gvl = in_iface(nr, k) ? gx[s] - gxm[s] : 0.0;
        const bool pv = fv[s] >= 0.0;
        const double g = gvl * fv[s];
        gp[s] = gm[s] = gpp[s] = gmp[s] = 0.0;
        double ae;
        if (k == nr.x) {
            ae = pv ? P[s] : M[s];
            if (pv) gp[s] = g; else gm[s] = g;
        } else if (pv) {
            ae = fmin(Mm[s], P[s]);
            gp[s] = gmin_x(g, P[s], Mm[s]);
            gmp[s] = gmin_x(g, Mm[s], P[s]);
        } else {
            ae = fmin(Pm[s], M[s]);
            gm[s] = gmin_x(g, M[s], Pm[s]);
            gpp[s] = gmin_x(g, Pm[s], M[s]);
        }
        gva[s] = gvl * ae;
    }
    col_next<NS>(gpp, nx, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) gp[s] += nx[s] + hp[s];
    col_next<NS>(gmp, nx, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) gm[s] += nx[s] + hm[s];
    // limiter factors (:441-451)
    double tvxm[NS], tvxp[NS], tvnm[NS], tvnp[NS], fvb[NS];
    col_prev_own<NS, HALF>(tvx, tvxm);
    col_next<NS>(tvx, tvxp, 0.0);
    col_prev_own<NS, HALF>(tvn, tvnm);
    col_next<NS>(tvn, tvnp, 0.0);
    col_next<NS>(fv, fvb, 0.0);
    double gfp[NS], gfn[NS], mx[NS], mn[NS], W[NS], ar[NS], Zc[NS], zb[NS], A1[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        const int kc = k < L ? k : L - 1;
        const size_t i = b0 + kc;
        const bool wet = in_layer(nr, k);
        W[s] = G(a.w_e)[i];
        if (a.w_i) W[s] = W[s] + G(a.w_i)[i];
        const double2 aa = ldv(m.aav, i);
        ar[s] = aa.x;
        if (a.Z3d) { Zc[s] = G(a.Z3d)[i]; zb[s] = G(a.zbar3)[i]; }
        else { const double2 z = ldv(m.zzb, kc); Zc[s] = z.x; zb[s] = z.y; }
        gfp[s] = gfn[s] = mx[s] = mn[s] = 0.0;
        if (wet) {
            const double av = aa.y, hn = G(a.hnn)[i];
            const double safe_a = av > 0.0 ? av : 1.0, safe_hn = hn > 0.0 ? hn : 1.0;
            const bool own = (k == nr.x) || (k == nr.y - 1), valid = av > 0.0 && hn > 0.0;
            const double cmax = own ? tvx[s] : fmax(fmax(tvxm[s], tvx[s]), tvxp[s]);
            const double cmin = own ? tvn[s] : fmin(fmin(tvnm[s], tvn[s]), tvnp[s]);
            const double up = cmax - LOc[s], dn = cmin - LOc[s];
            const double fplus = (fmax(fv[s], 0.0) + fmax(-fvb[s], 0.0)) + ap[s];
            const double fminus = (fmin(fv[s], 0.0) + fmin(-fvb[s], 0.0)) + am[s];
            const double fpos = fplus * a.dt / safe_a / safe_hn + FCT_FLUX_EPS;
            const double fneg = fminus * a.dt / safe_a / safe_hn - FCT_FLUX_EPS;
            // the factor is min(1, up / fpos): no cotangent where the quotient exceeds 1,
            // which a factor of two decides without dividing
            if (valid && !(fpos > 0.0 && up >= 2.0 * fpos)) {
                const double g = gmin_x(gp[s], up / fpos, 1.0);
                mx[s] = g / fpos;
                gfp[s] = (-g * up) * (1.0 / (fpos * fpos)) / safe_hn / safe_a * a.dt;
            }
            if (valid && !(fneg < 0.0 && dn <= 2.0 * fneg)) {
                const double g = gmin_x(gm[s], dn / fneg, 1.0);
                mn[s] = g / fneg;
                gfn[s] = (-g * dn) * (1.0 / (fneg * fneg)) / safe_hn / safe_a * a.dt;
            }
            // T_new depends on LO through LO * hnode_new / hnode_new
            const double g_lo = hn > 0.0 ? G(a.g_out)[i] : 0.0;
            stv(a.gpm, i, make_double2(gfp[s], gfn[s]));
            stv(a.tv, i, make_double2(tvx[s], tvn[s]));
            G(a.gLO)[i] = g_lo - (mx[s] + mn[s]);
        }
    }
    // cotangent of adf_v: limited flux, P+/P- of this level and of the one above
    double gfpm[NS], gfnm[NS], gav[NS];
    col_prev<NS, HALF>(gfp, gfpm, 0.0);
    col_prev<NS, HALF>(gfn, gfnm, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        gav[s] = gva[s] + (gmax_x(gfp[s], fv[s], 0.0) + gmin_x(gfn[s], fv[s], 0.0));
        if (k > 0) gav[s] += -gmax_x(gfpm[s], -fv[s], 0.0) - gmin_x(gfnm[s], -fv[s], 0.0);
    }
    // cluster bounds (a4) and the tied elements' shares: level j's cotangent goes to the
    // bounds of j-1, j, j+1
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        double ga[NS], gb[NS], gc[NS], o1[NS], o2[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 64 * s + col_lane<HALF>();
            const double g = w ? mn[s] : mx[s];
            const double x = w ? tvnm[s] : tvxm[s], y = w ? tvn[s] : tvx[s], z = w ? tvnp[s] : tvxp[s];
            ga[s] = gc[s] = 0.0;
            gb[s] = g;
            if (k != nr.x && k != nr.y - 1) {
                const double m1 = w ? fmin(x, y) : fmax(x, y);
                const double g1 = w ? gmin_x(g, m1, z) : gmax_x(g, m1, z);
                gc[s] = w ? gmin_x(g, z, m1) : gmax_x(g, z, m1);
                ga[s] = w ? gmin_x(g1, x, y) : gmax_x(g1, x, y);
                gb[s] = w ? gmin_x(g1, y, x) : gmax_x(g1, y, x);
                if (k == 0) gb[s] += ga[s];
            }
        }
        col_next<NS>(ga, o1, 0.0);
        col_prev<NS, HALF>(gc, o2, 0.0);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const double v = (gb[s] + o1[s]) + o2[s], c = w ? cn[s] : cx[s];
            if (w) mn[s] = c > 0.0 ? v / c : 0.0;
            else mx[s] = c > 0.0 ? v / c : 0.0;
        }
    }
    // QR4C (:241-295): interface j's cotangent goes to A[j], A[j-1], A[j-2], A[j+1], w[j]
    col_prev_own<NS, HALF>(Ac, A1);
    double Zm1[NS], dz[NS], qc[NS], qu[NS], qd[NS], dzu[NS], dzd[NS];
    col_prev_own<NS, HALF>(Zc, Zm1);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        dz[s] = nz_safe(Zm1[s] - Zc[s]);
        qc[s] = 64 * s <= nr.y ? (A1[s] - Ac[s]) / dz[s] : 0.0;
    }
    col_next<NS>(qc, qu, 0.0);
    col_prev<NS, HALF>(qc, qd, 0.0);
    col_next<NS>(dz, dzu, 1.0);
    col_prev<NS, HALF>(dz, dzd, 1.0);
    double t0[NS], tm1[NS], tm2[NS], tp1[NS], tw[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        t0[s] = tm1[s] = tm2[s] = tp1[s] = tw[s] = 0.0;
        if (!in_layer(nr, k)) continue;      // interface nzmax has no high-order flux
        const double g = gav[s] * ar[s];
        if (k == nr.x) {
            t0[s] = -(g * W[s]);
            tw[s] = -(g * Ac[s]);
        } else if (k == nr.x + 1 || k == nr.y - 1) {
            t0[s] = tm1[s] = -0.5 * (g * W[s]);
            tw[s] = g * (-0.5 * (A1[s] + Ac[s]));
        } else {
            const double h1 = zb[s] - Zc[s], h2 = zb[s] - Zm1[s];
            const double q1 = Ac[s] + (2.0 * qc[s] + qu[s]) * h1 / 3.0;
            const double q2 = A1[s] + (2.0 * qc[s] + qd[s]) * h2 / 3.0;
            tw[s] = g * (-0.5 * (q1 + q2));
            const double gt = -0.5 * (g * W[s]);
            const double g1 = gt / 3.0 * h1, g2 = gt / 3.0 * h2;
            const double gc = (2.0 * g1 + 2.0 * g2) / dz[s];
            tp1[s] = -(g1 / dzu[s]);
            tm2[s] = g2 / dzd[s];
            t0[s] = (gt - gc) - tp1[s];
            tm1[s] = (gt + gc) - tm2[s];
        }
    }
    double x1[NS], x2[NS], x3[NS], x4[NS];
    col_next<NS>(tm2, x1, 0.0);
    col_next<NS>(tm1, x2, 0.0);
    col_next<NS>(x1, x3, 0.0);
    col_prev<NS, HALF>(tp1, x4, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        if (k >= L) continue;
        const size_t i = b0 + k;
        if (in_layer(nr, k)) {
            stv(a.sh, i, make_double2(mx[s], mn[s]));
            G(a.gadfv)[i] = gav[s];
            G(a.gA)[i] = (t0[s] + x2[s]) + (x3[s] + x4[s]);
        }
        if (a.gw) G(a.gw)[i] = a.first ? tw[s] : G(a.gw)[i] + tw[s];
        if (a.gwi) G(a.gwi)[i] = a.first ? tw[s] : G(a.gwi)[i] + tw[s];
    }
    if (a.first)      // levels past the slots (a shallow column in the one-slot body)
        for (int k = (HALF ? 32 : 64 * NS) + col_lane<HALF>(); k < L; k += HALF ? 32 : 64) {
            if (a.gw) G(a.gw)[b0 + k] = 0.0;
            if (a.gwi) G(a.gwi)[b0 + k] = 0.0;
        }
}

// LO's vertical upwind flux and adf_v's (:108-120): cotangents gl, gh of the two at
// this lane's interface (equal without the split) and w_e, w_e + w_i; returns T's
// contribution of this interface to its own level, hands back the one to the level
// above in `up`
__device__ __forceinline__ double upwind_v(double g, double W, int k, double& up) {
    const double aw = fabs(W);
    up = g * (W - aw);
    return k == 0 ? g * (W + aw) + up : g * (W + aw);
}

// ---- LO (:298-313) and its vertical flux, from the column's gLO -------------------
// gT receives what the column's T takes from LO, the vertical fluxes and the bounds (gt)
template <int NS, bool SPLIT, bool HALF>
__device__ __forceinline__ void lo_column(const ColArgs& a, int n, int2 nr, const double (&gLO)[NS],
                                          const double (&gt)[NS], const double (&Tc)[NS]) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const size_t b0 = (size_t)n * L;
    double gdv[NS], gdm[NS], acc[NS], av[NS], We[NS], Wf[NS], ar[NS], gq[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        gdv[s] = acc[s] = We[s] = Wf[s] = ar[s] = gq[s] = 0.0;
        if (!in_layer(nr, k)) continue;
        const size_t i = b0 + k;
        const double2 aa = ldv(m.aav, i);
        ar[s] = aa.x; av[s] = aa.y;
        const double hn = G(a.hnn)[i];
        We[s] = G(a.w_e)[i];
        Wf[s] = SPLIT ? We[s] + G(a.w_i)[i] : We[s];
        gq[s] = -G(a.gadfv)[i];
        const bool valid = hn > 0.0 && av[s] > 0.0;
        const double gnum = (valid ? gLO[s] : 0.0) / (hn > 0.0 ? hn : 1.0);
        gdv[s] = gnum / (av[s] > 0.0 ? av[s] : 1.0) * a.dt;
        acc[s] = gt[s] + gnum * G(a.hnode)[i];
        // T_new's direct dependence on T cancels where the layer is updated
        if (!(hn > 0.0)) acc[s] += G(a.g_out)[i];
        stv(a.gd, i, make_double2(G(a.ghsc)[i], gdv[s]));
    }
    col_prev<NS, HALF>(gdv, gdm, 0.0);
    double up[NS], upn[NS], Tm[NS];
    col_prev_own<NS, HALF>(Tc, Tm);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        up[s] = 0.0;
        if (!in_layer(nr, k)) continue;
        const double gl0 = gdv[s] - (k > 0 ? gdm[s] : 0.0);
        double u1 = 0.0, u2 = 0.0, gw, gwi = 0.0;
        if (SPLIT) {
            const double gl = -0.5 * (gl0 * ar[s]), gh = -0.5 * (gq[s] * ar[s]);
            acc[s] += upwind_v(gl, We[s], k, u1) + upwind_v(gh, Wf[s], k, u2);
            const double lp = gl * Tc[s], lm = gl * Tm[s], hp = gh * Tc[s], hm = gh * Tm[s];
            gwi = hp + hm + gabs(hp - hm, Wf[s]);
            gw = (lp + lm + gabs(lp - lm, We[s])) + gwi;
        } else {
            const double g = -0.5 * ((gq[s] + gl0) * ar[s]);
            acc[s] += upwind_v(g, We[s], k, u1);
            const double p = g * Tc[s], q = g * Tm[s];
            gw = p + q + gabs(p - q, We[s]);
        }
        up[s] = u1 + u2;
        if (a.gw) G(a.gw)[b0 + k] += gw;
        if (SPLIT && a.gwi) G(a.gwi)[b0 + k] += gwi;
    }
    col_next<NS>(up, upn, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + col_lane<HALF>();
        if (in_layer(nr, k)) G(a.gT)[b0 + k] = acc[s] + upn[s];
        // the surface interface's flux reads the dry level above it
        if (k + 1 == nr.x) G(a.gT)[b0 + k] = G(a.g_out)[b0 + k] + upn[s];
    }
}

// ---- R3: vertex cotangents of the bounds; without the split also LO ---------------
template <int NS, int DM, bool SPLIT, bool HALF>
__device__ __forceinline__ void vertex_body(const ColArgs& a, int n) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y);
    const size_t b0 = (size_t)n * L;
    int2 rg[DM];      // ring: neighbour, layer range of the triangle to the next slot
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        const int4 r = ldc(a.tab.ring, (size_t)n * DM + q);
        rg[q] = make_int2(r.x, r.w & 0xffff);
    }
    double gLO[NS], gt[NS], Tc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        gLO[s] = gt[s] = Tc[s] = 0.0;
        if (64 * s >= nr.y) continue;
        const int k = 64 * s + col_lane<HALF>();
        const size_t i = b0 + k;
        if (k < nr.y) Tc[s] = G(a.T)[i];      // the level above the surface too
        if (!in_layer(nr, k)) continue;
        double lo[DM], t[DM];
        double2 tv[DM], sh[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const size_t r = (size_t)rg[q].x * L + k;
            lo[q] = G(a.LO)[r];
            t[q] = G(a.T)[r];
            tv[q] = ldv(a.tv, r);
            sh[q] = ldv(a.sh, r);
        }
        const double lo0 = G(a.LO)[i], tc = Tc[s];
        const double2 tv0 = ldv(a.tv, i), sh0 = ldv(a.sh, i);
        gLO[s] = G(a.gLO)[i];
#pragma unroll
        for (int w = 0; w < 2; ++w) {      // the maximum, then the minimum
            const double x0 = w ? fmin(lo0, tc) : fmax(lo0, tc);
            const double v0 = w ? tv0.y : tv0.x, s0 = w ? sh0.y : sh0.x;
            double gm = 0.0;
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const int q1 = (q + 1) % DM;
                const double x1 = w ? fmin(lo[q], t[q]) : fmax(lo[q], t[q]);
                const double x2 = w ? fmin(lo[q1], t[q1]) : fmax(lo[q1], t[q1]);
                const double e = w ? fmin(fmin(x0, x1), x2) : fmax(fmax(x0, x1), x2);
                // the extremum's cotangent: the shares of the vertices whose bound it
                // attains, split between the vertices that attain it
                double g = v0 == e ? s0 : 0.0;
                g = g + ((w ? tv[q].y : tv[q].x) == e ? (w ? sh[q].y : sh[q].x) : 0.0);
                g = g + ((w ? tv[q1].y : tv[q1].x) == e ? (w ? sh[q1].y : sh[q1].x) : 0.0);
                const int h = 1 + (x1 == e) + (x2 == e);      // where x0 attains it
                g = h == 1 ? g : (h == 2 ? 0.5 * g : g / 3.0);
                gm = gm + (in_bytes(rg[q].y, 0, k) && x0 == e ? g : 0.0);
            }
            gLO[s] = gLO[s] + (w ? gmin_x(gm, lo0, tc) : gmax_x(gm, lo0, tc));
            gt[s] = gt[s] + (w ? gmin_x(gm, tc, lo0) : gmax_x(gm, tc, lo0));
        }
        if (SPLIT) {
            G(a.gLO)[i] = gLO[s];
            G(a.gT)[i] = gt[s];
        }
    }
    if (!SPLIT) lo_column<NS, false, HALF>(a, n, nr, gLO, gt, Tc);
}

// ---- R3 under the split, after the column solve's transpose -----------------------
template <int NS>
__device__ __forceinline__ void split_body(const ColArgs& a, int n) {
    const int L = a.m.L;
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y);
    const size_t b0 = (size_t)n * L;
    double gLO[NS], gt[NS], Tc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        const bool wet = in_layer(nr, k);
        gLO[s] = wet ? G(a.gLO)[b0 + k] : 0.0;
        gt[s] = wet ? G(a.gT)[b0 + k] : 0.0;
        Tc[s] = k < nr.y ? G(a.T)[b0 + k] : 0.0;
    }
    lo_column<NS, true, false>(a, n, nr, gLO, gt, Tc);
}

// ---- R4: edges (:196-225, :344-368, :426-435, :460-466, :96-105) -------------------
template <int NS, bool HALF>
__device__ __forceinline__ void edge_body(const ColArgs& a, int e) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 kr = ldc(a.ekr, e), nd = ldc(m.edges, e), ur = ldc(m.utri_rng, e), ud = ldc(m.updn, e);
    const double2 cc = ldc(m.edge_c, e);
    const int4 va = ldc(m.udv, 2 * (size_t)e);
    const int vb = ldc(reinterpret_cast<const int*>(m.udv), 8 * (size_t)e + 4);
    const int cu = vb & 3, cd = (vb >> 2) & 3;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (64 * s >= kr.y) break;
        const int k = 64 * s + col_lane<HALF>();
        if (k < kr.x || k >= kr.y) continue;
        const int lo = kr.x > 64 * s ? kr.x : 64 * s, hi = kr.y < 64 * s + 64 ? kr.y : 64 * s + 64;
        const int tl = lo > ur.x ? lo : ur.x, th = hi < ur.y ? hi : ur.y;
        const bool any_tri = tl < th, any_avg = !(tl == lo && th == hi);
        const size_t t = (size_t)e * L + k;
        const size_t i1 = (size_t)nd.x * L + k, i2 = (size_t)nd.y * L + k;
        const double vf = G(a.vflux)[t], adf = G(a.adfh)[t];
        const double T1 = G(a.T)[i1], T2 = G(a.T)[i2];
        const double O1 = G(a.Told)[i1], O2 = G(a.Told)[i2];
        const double2 p1 = ldv(a.pm, i1), p2 = ldv(a.pm, i2);
        const double2 q1 = ldv(a.gpm, i1), q2 = ldv(a.gpm, i2);
        const double2 d1 = ldv(a.gd, i1), d2 = ldv(a.gd, i2);
        double gv0 = 0.0;
        if (!a.first) gv0 = G(a.g_vf)[t];
        double a0 = 0.0, a1 = 0.0, b0 = 0.0, b1 = 0.0;
        if (any_tri) {
            a0 = G(a.T)[(size_t)va.x * L + k]; a1 = G(a.T)[(size_t)va.y * L + k];
            b0 = G(a.T)[(size_t)va.z * L + k]; b1 = G(a.T)[(size_t)va.w * L + k];
        }
        double2 ga = make_double2(0.0, 0.0), gb = ga;
        if (any_avg) {
            ga = ldv(a.gnode, i1);
            gb = ldv(a.gnode, i2);
        }
        const bool tri = k >= ur.x && k < ur.y;
        if (any_tri) {
            const size_t gu = 6 * (size_t)ud.x, gw = 6 * (size_t)ud.y;
            const double u0 = cu == 0 ? T1 : a0, u1 = cu == 0 ? a0 : (cu == 1 ? T1 : a1);
            const double u2 = cu == 2 ? T1 : a1;
            const double v0 = cd == 0 ? T2 : b0, v1 = cd == 0 ? b0 : (cd == 1 ? T2 : b1);
            const double v2 = cd == 2 ? T2 : b1;
            const double ux = ldc(m.gs, gu) * u0 + ldc(m.gs, gu + 1) * u1 + ldc(m.gs, gu + 2) * u2;
            const double uy = ldc(m.gs, gu + 3) * u0 + ldc(m.gs, gu + 4) * u1 + ldc(m.gs, gu + 5) * u2;
            const double wx = ldc(m.gs, gw) * v0 + ldc(m.gs, gw + 1) * v1 + ldc(m.gs, gw + 2) * v2;
            const double wy = ldc(m.gs, gw + 3) * v0 + ldc(m.gs, gw + 4) * v1 + ldc(m.gs, gw + 5) * v2;
            if (tri) { ga = make_double2(ux, uy); gb = make_double2(wx, wy); }
        }
        // adf_h: limited flux and P+/P-
        const bool pos = adf >= 0.0;
        const double ae = fmin(pos ? p1.x : p1.y, pos ? p2.y : p2.x);
        double gh = (d1.x - d2.x) * ae;
        gh = gh + (((gmax_x(q1.x, adf, 0.0) - gmax_x(q2.x, -adf, 0.0)) + gmin_x(q1.y, adf, 0.0)) -
                   gmin_x(q2.y, -adf, 0.0));
        // high order (A, gradients), then upwind (T)
        const double av = fabs(vf);
        const double A1 = ab2(O1, T1), A2 = ab2(O2, T2);
        const double diff = A2 - A1;
        const double Tm1 = A1 + (2.0 * diff + cc.x * ga.x + cc.y * ga.y) / 6.0;
        const double Tm2 = A2 - (2.0 * diff + cc.x * gb.x + cc.y * gb.y) / 6.0;
        // (vf + |vf|, vf - |vf|) is (2 vf, 0) or (0, 2 vf): only the upwind end's mean and T
        // take a cotangent, besides vflux
        const double gs2 = -0.5 * gh, gs1 = -0.5 * (-gh + (d1.y - d2.y));
        const double v2 = vf >= 0.0 ? vf + av : vf - av;
        double gp = gs2 * Tm1, gm = gs2 * Tm2;
        double gv = gp + gm + gabs(gp - gm, vf);
        gp = gs1 * T1;
        gm = gs1 * T2;
        gv = gv + (gp + gm + gabs(gp - gm, vf));
        stv(a.eg, t, make_double2(gs2 * v2, gs1 * v2));
        G(a.g_vf)[t] = gv0 + gv;
        uint64_t up = __ballot(vf >= 0.0);             // lanes of wet levels
        if (HALF) up &= 0xffffffffu;                   // the same in both halves
        if (k == lo) ((gptr<uint64_t>)a.edge_up)[(size_t)e * NS + s] = up;
    }
}

// whether edge e's vflux is >= 0 at this lane's level of slot s
template <int NS>
__device__ __forceinline__ bool edge_up(const ColArgs& a, int e, int s) {
    const uint64_t b = ((cptr<uint64_t>)a.edge_up)[(size_t)e * NS + s];
    return (b >> lane_id()) & 1;
}

// ---- node-averaged gradients (:329-341), on the levels [glo, ghi) that edges read ----
template <int NS, int DM>
__device__ __forceinline__ void gnum_body(const ColArgs& a, int n) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int4 hd = ldc(a.tab.hdr, n);
    const int glo = (hd.z >> 8) & 0xff, ghi = (hd.z >> 16) & 0xff;
    if (glo >= ghi) return;
    const int ne = hd.z & 0xff;
    int ent[DM], ew[DM];
    int2 ur[DM], kr[DM];
    double2 cc[DM];
    double ea[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        const int4 es = ldc(a.tab.edge, (size_t)n * DM + q);
        ent[q] = es.x;
        ew[q] = es.w;
        ea[q] = ldc(m.earea, ldc(reinterpret_cast<const int*>(a.tab.elem), 4 * ((size_t)n * DM + q)));
    }
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        ur[q] = ldc(m.utri_rng, ent[q] >> 1);
        kr[q] = ldc(a.ekr, ent[q] >> 1);
        cc[q] = ldc(m.edge_c, ent[q] >> 1);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (glo >= 64 * s + 64 || ghi <= 64 * s) continue;
        const int k = 64 * s + lane_id();
        if (k < glo || k >= ghi) continue;
        double g[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool on = q < ne && k >= kr[q].x && k < kr[q].y && !(k >= ur[q].x && k < ur[q].y);
            g[q] = on ? G(reinterpret_cast<double*>(a.eg))[2 * ((size_t)(ent[q] >> 1) * L + k)] : 0.0;
        }
        double gx = 0.0, gy = 0.0, den = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool side = ent[q] & 1;
            // the upwind end's gradient only, with the sign of its mean's edge vector
            double h = edge_up<NS>(a, ent[q] >> 1, s) != side ? g[q] / 6.0 : 0.0;
            if (side) h = -h;
            gx = gx + h * cc[q].x;
            gy = gy + h * cc[q].y;
            den = den + (q < hd.w && in_bytes(ew[q], 0, k) ? ea[q] : 0.0);
        }
        const double d = den > 0.0 ? den : 1.0;
        stv(a.gnum, (size_t)n * L + k, make_double2(gx / d, gy / d));
    }
}

// ---- element gradient cotangents (:316-368) -------------------------------------------
// Two triangles per wavefront, four of each one's edges (those that have it as their up or
// down triangle) at a time, so that the chain list entry -> edge tables -> column is paid
// once for eight columns.
constexpr int TR_EL = 2, TR_ED = 4;
template <int NS>
__device__ __forceinline__ void tr_body(const ColArgs& a, int w) {
    const DevMesh& m = a.m;
    const int L = m.L;
    int e[TR_EL], p0[TR_EL], p1[TR_EL], v[TR_EL][3], z[TR_EL][3];
    int2 er[TR_EL];
    double ea[TR_EL];
    int top = 0, deg = 0;
#pragma unroll
    for (int i = 0; i < TR_EL; ++i) {
        const bool on = w * TR_EL + i < m.E;
        e[i] = on ? w * TR_EL + i : m.E - 1;
        er[i] = on ? ldc(m.elev, e[i]) : make_int2(0, 0);
        p0[i] = ldc(a.ud_off, e[i]);
        p1[i] = ldc(a.ud_off, e[i] + 1);
        ea[i] = ldc(m.earea, e[i]);
#pragma unroll
        for (int j = 0; j < 3; ++j) v[i][j] = ldc(m.en, 3 * (size_t)e[i] + j);
        top = er[i].y > top ? er[i].y : top;
        deg = p1[i] - p0[i] > deg ? p1[i] - p0[i] : deg;
    }
#pragma unroll
    for (int i = 0; i < TR_EL; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            z[i][j] = ldc(reinterpret_cast<const int*>(a.tab.hdr), 4 * (size_t)v[i][j] + 2);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (64 * s >= top) break;
        const int k = 64 * s + lane_id();
        double gx[TR_EL] = {}, gy[TR_EL] = {};
        for (int b = 0; b < deg; b += TR_ED) {
            int d[TR_EL][TR_ED];
            int2 ur[TR_EL][TR_ED];
            double2 cc[TR_EL][TR_ED];
            double g[TR_EL][TR_ED];
#pragma unroll
            for (int i = 0; i < TR_EL; ++i)
#pragma unroll
                for (int j = 0; j < TR_ED; ++j) {
                    const int p = p0[i] + b + j;
                    d[i][j] = p < p1[i] ? ldc(a.ud_ent, p) : -1;
                }
#pragma unroll
            for (int i = 0; i < TR_EL; ++i)
#pragma unroll
                for (int j = 0; j < TR_ED; ++j) {
                    const int x = d[i][j] < 0 ? 0 : d[i][j] >> 1;
                    ur[i][j] = ldc(m.utri_rng, x);
                    cc[i][j] = ldc(m.edge_c, x);
                    const bool role = d[i][j] & 1;
                    const bool on = d[i][j] >= 0 && k >= er[i].x && k < er[i].y &&
                                    k >= ur[i][j].x && k < ur[i][j].y &&
                                    edge_up<NS>(a, x, s) != role;
                    g[i][j] = on ? G(reinterpret_cast<double*>(a.eg))[2 * ((size_t)x * L + k)] : 0.0;
                }
#pragma unroll
            for (int i = 0; i < TR_EL; ++i)
#pragma unroll
                for (int j = 0; j < TR_ED; ++j) {
                    const double h = d[i][j] & 1 ? -(g[i][j] / 6.0) : g[i][j] / 6.0;
                    gx[i] = gx[i] + h * cc[i][j].x;
                    gy[i] = gy[i] + h * cc[i][j].y;
                }
        }
#pragma unroll
        for (int i = 0; i < TR_EL; ++i) {
            const bool wet = k >= er[i].x && k < er[i].y;
            double sx = 0.0, sy = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (wet && in_bytes(z[i][j], 8, k)) {
                    const double2 q = ldv(a.gnum, (size_t)v[i][j] * L + k);
                    sx = sx + q.x;
                    sy = sy + q.y;
                }
            if (wet) stv(a.g_tr, (size_t)e[i] * L + k, make_double2(gx[i] + sx * ea[i], gy[i] + sy * ea[i]));
        }
    }
}

// ---- nodes gather edges and triangles; AB2 (:59-66) ------------------------------------
// (NSL: the mesh's slots, NS the node's)
template <int NS, int DM, int NSL>
__device__ __forceinline__ void gather_body(const ColArgs& a, int n) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int4 hd = ldc(a.tab.hdr, n);
    const int2 nr = make_int2(hd.x, hd.y), cnt = make_int2(hd.z & 0xff, hd.w);
    const size_t b0 = (size_t)n * L;
    int ent[DM], rng[DM], erg[DM];
    int4 el[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        const int4 es = ldc(a.tab.edge, (size_t)n * DM + q);
        ent[q] = es.x; rng[q] = es.z; erg[q] = es.w;
        el[q] = ldc(a.tab.elem, (size_t)n * DM + q);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        const bool wet = in_layer(nr, k);
        const size_t i = b0 + k;
        if (!wet) {
            if (k < L) {
                if (k + 1 != nr.x) G(a.gT)[i] = G(a.g_out)[i];
                G(a.gTold)[i] = 0.0;
            }
            continue;
        }
        double2 at[DM] = {}, tr[DM] = {};
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            at[q] = ldv(a.eg, (size_t)(ent[q] >> 1) * L + k);
            tr[q] = ldv(a.g_tr, (size_t)el[q].x * L + k);
        }
        double ga = G(a.gA)[i], gt = G(a.gT)[i];
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool ein = q < cnt.x && (in_bytes(rng[q], 0, k) || in_bytes(rng[q], 16, k));
            // the upwind mean is A + (2 (A2 - A1) + ...) / 6
            const double g3 = 2.0 * (at[q].x / 6.0);
            const bool mine = edge_up<NSL>(a, ent[q] >> 1, s) != (bool)(ent[q] & 1);
            ga = ga + (ein ? (mine ? at[q].x - g3 : g3) : 0.0);
            gt = gt + (ein && mine ? at[q].y : 0.0);
            const int v = el[q].y == n ? 0 : (el[q].z == n ? 1 : 2);
            const size_t g6 = 6 * (size_t)el[q].x + v;
            const double c = tr[q].x * ldc(m.gs, g6) + tr[q].y * ldc(m.gs, g6 + 3);
            gt = gt + (q < cnt.y && in_bytes(erg[q], 0, k) ? c : 0.0);
        }
        G(a.gT)[i] = gt + AB_NEW * ga;
        G(a.gTold)[i] = AB_OLD * ga;
    }
    for (int k = 64 * NS + lane_id(); k < L; k += 64) {
        G(a.gT)[b0 + k] = G(a.g_out)[b0 + k];
        G(a.gTold)[b0 + k] = 0.0;
    }
}

// ---- uv from the vflux cotangent (:69-93) ----------------------------------------------
template <int NS>
__device__ __forceinline__ void uv_body(const ColArgs& a, double2* g_uv, int e) {
    const DevMesh& m = a.m;
    const int L = m.L;
    const int2 er = ldc(m.elev, e);
    const int p0 = ldc(a.et_off, e), p1 = ldc(a.et_off, e + 1);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = 64 * s + lane_id();
        const bool wet = k >= er.x && k < er.y;
        double gx = 0.0, gy = 0.0;
        const size_t t = (size_t)e * L + k;
        const double h = wet ? G(a.helem)[t] : 0.0;
        for (int p = p0; p < p1; p += 3) {       // a triangle has three edges
            double g[3];
            int en[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                en[i] = ldc(a.et_ent, p + i < p1 ? p + i : p);
                const bool rd = wet && p + i < p1;
                const size_t x = (size_t)(en[i] >> 1) * L + k;
                g[i] = rd ? G(a.g_vf)[x] : 0.0;
                if (a.g_vf1) g[i] = g[i] + (rd ? G(a.g_vf1)[x] : 0.0);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double4 c = ldc(m.cross, en[i] >> 1);
                const double x = g[i] * h;
                const bool second = en[i] & 1;
                gx = gx + (second ? -(x * c.w) : x * c.y);
                gy = gy + (second ? x * c.z : -(x * c.x));
            }
        }
        if (k < L) stv(g_uv, t, make_double2(gx, gy));
    }
}

#define KC_OCC(n) __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(n)))

__global__ void KC_OCC(6) kc_ghsc(ColArgs a0) {
    const ColArgs a = of_tracer(a0);
    int w;
    if (single_wave((a.m.N + GH_NODES - 1) / GH_NODES, a.remap, w)) ghsc_body(a, w);
}
template <int NS, int DM, bool HALVES>
__global__ void KC_OCC(NS == 1 && DM == 6 ? 4 : 3) kc_limit(ColArgs a0, int first, int count) {
    const ColArgs a = of_tracer(a0);
    int n;
    if (!node_task(a, first, count, n)) return;
    if constexpr (HALVES)
        if (ldc(a0.tab.hdr, n).y < 31) {
            if (blockIdx.y) return;
            asm volatile("" ::: "memory");      // no merging of the two bodies' loads
            limit_body<1, DM, true>(of_half(a0), n);
            return;
        }
    limit_body<NS, DM, false>(a, n);
}
template <int NS, int DM, bool SPLIT, bool HALVES>
__global__ void KC_OCC(DM == 6 ? 4 : 3) kc_vertex(ColArgs a0, int first, int count) {
    const ColArgs a = of_tracer(a0);
    int n;
    if (!node_task(a, first, count, n)) return;
    if constexpr (HALVES)
        if (ldc(a0.tab.hdr, n).y < 31) {
            if (blockIdx.y) return;
            asm volatile("" ::: "memory");      // no merging of the two bodies' loads
            vertex_body<1, DM, SPLIT, true>(of_half(a0), n);
            return;
        }
    vertex_body<NS, DM, SPLIT, false>(a, n);
}
template <int NS>
__global__ void KC_OCC(8) kc_split(ColArgs a0, int first, int count) {
    const ColArgs a = of_tracer(a0);
    int n;
    if (node_task(a, first, count, n)) split_body<NS>(a, n);
}
template <int NS, bool HALVES>
__global__ void KC_OCC(6) kc_edge(ColArgs a0) {
    const ColArgs a = of_tracer(a0);
    int e;
    if (!single_wave(a.m.D, a.remap, e)) return;
    if constexpr (HALVES)
        if (ldc(a0.ekr, e).y < 32) {
            if (blockIdx.y) return;
            asm volatile("" ::: "memory");
            edge_body<NS, true>(of_half(a0), e);
            return;
        }
    edge_body<NS, false>(a, e);
}
template <int NS, int DM>
__global__ void KC_OCC(8) kc_gnum(ColArgs a0) {
    const ColArgs a = of_tracer(a0);
    int n;
    if (single_wave(a.m.N, a.remap, n)) gnum_body<NS, DM>(a, n);
}
template <int NS>
__global__ void KC_OCC(8) kc_tr(ColArgs a0) {
    const ColArgs a = of_tracer(a0);
    int w;
    if (single_wave((a.m.E + TR_EL - 1) / TR_EL, a.remap, w)) tr_body<NS>(a, w);
}
template <int NS, int DM, int NSL>
__global__ void KC_OCC(DM == 6 ? 6 : 5) kc_gather(ColArgs a0, int first, int count) {
    const ColArgs a = of_tracer(a0);
    int n;
    if (node_task(a, first, count, n)) gather_body<NS, DM, NSL>(a, n);
}
template <int NS>
__global__ void KC_OCC(8) kc_uv(ColArgs a, double2* g_uv) {
    int e;
    if (single_wave(a.m.E, a.remap, e)) uv_body<NS>(a, g_uv, e);
}

// the odd tracers' w cotangents onto the even ones'
__global__ void __launch_bounds__(256) kc_add(size_t n, double* x, const double* x1, double* y,
                                              const double* y1) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    if (x) x[i] = x[i] + x1[i];
    if (y) y[i] = y[i] + y1[i];
}

constexpr int WPB = 4;

// Meshes of at most this many nodes run two tracers per launch (workspace for both, if the
// plan has two tracer slots): one tracer's column kernels leave wavefront slots of a small
// mesh's chip idle or end in a mostly idle last round, and k_vimpl_reverse has one workgroup
// per CU or less (two steps of the pi mesh 542 -> 508 us, icosa-6 x 70 with the split 1621 ->
// 1530). Where one tracer's launches fill the chip the pair gains by short columns in halves
// (HALF_NODES): icosa-7 x 47 3519 -> 3411, x 70 4337 -> 4316. Above the line, which keeps
// the second set (15 node, 3 edge, 2 triangle arrays) below about 4 GB, every tracer is
// reversed alone and no column shares a wavefront.
constexpr int PAIR_NODES = 131072;
// From this many nodes on, the launches of two tracers put both tracers of a short node
// or edge column (31 levels and the bottom interface at most) into the halves of one
// wavefront in kc_limit, kc_vertex and kc_edge; the tables stay wave-uniform. icosa-7 x 47
// 3519 -> 3411 us (kc_limit 642 -> 602, kc_edge 601 -> 572, kc_vertex 514 -> 440), three
// tracers with 1 % of the nodes at eight neighbours 6061 -> 5753, x 70 4337 -> 4316; icosa-6
// x 47 922 -> 900. Smaller meshes need the wavefronts, and kernels without the halves, which
// take 16 registers less: icosa-5 x 60 324 us, 331 with them.
constexpr int HALF_NODES = 16384;

// the node kernels: shallow columns, then (nl > 64) deep ones
#define KC_NODES(KERN1, KERN2)                                                                \
    do {                                                                                      \
        const int ns = NS == 1 ? a.m.N : a.tab.nshallow, nd = a.m.N - ns;                     \
        if (ns) KERN1<<<dim3(blocks_for(ns, WPB), y), dim3(256), 0, s>>>(a, 0, ns);              \
        if (nd) KERN2<<<dim3(blocks_for(nd, WPB), y), dim3(256), 0, s>>>(a, ns, nd);             \
    } while (0)

template <int NS, int DM, bool HALVES>
int reverse_tracers(const ColArgs& a, const double* LOx, unsigned y, hipStream_t s) {
    kc_ghsc<<<dim3(blocks_for((a.m.N + GH_NODES - 1) / GH_NODES, WPB), y), dim3(256), 0, s>>>(a);
    KC_NODES((kc_limit<1, DM, HALVES>), (kc_limit<NS, DM, false>));
    if (a.w_i) {
        KC_NODES((kc_vertex<1, DM, true, HALVES>), (kc_vertex<NS, DM, true, false>));
        const int rc = launch_vimpl_reverse(a.m, a.w_i, a.hnn, a.dt, LOx, a.gLO, a.gwi,
                                            y == 2 ? a.gwi1 : nullptr, a.node_stride, s);
        if (rc) return rc;
        KC_NODES((kc_split<1>), (kc_split<NS>));
    } else {
        KC_NODES((kc_vertex<1, DM, false, HALVES>), (kc_vertex<NS, DM, false, false>));
    }
    kc_edge<NS, HALVES><<<dim3(blocks_for(a.m.D, WPB), y), dim3(256), 0, s>>>(a);
    kc_gnum<NS, DM><<<dim3(blocks_for(a.m.N, WPB), y), dim3(256), 0, s>>>(a);
    kc_tr<NS><<<dim3(blocks_for((a.m.E + TR_EL - 1) / TR_EL, WPB), y), dim3(256), 0, s>>>(a);
    KC_NODES((kc_gather<1, DM, NS>), (kc_gather<NS, DM, NS>));
    return check_launch("adjoint column kernels");
}

template <int NS>
int reverse_uv(const ColArgs& a, double* g_uv, hipStream_t s) {
    kc_uv<NS><<<dim3(blocks_for(a.m.E, WPB)), dim3(256), 0, s>>>(a, reinterpret_cast<double2*>(g_uv));
    return check_launch("kc_uv");
}

}  // namespace

// cotangent workspace of one tracer, in doubles (even: double2 arrays lie at its start)
static size_t even(size_t n) { return (n + 1) / 2 * 2; }
static size_t node_stride(const DevMesh& m) { return even((size_t)m.N * m.L * 15); }
static size_t edge_stride(const DevMesh& m) { return even((size_t)m.D * m.L * 3); }
static size_t elem_stride(const DevMesh& m) { return (size_t)m.E * m.L * 2; }

int adjoint_cols_tracers(const DevMesh& m) { return m.N <= PAIR_NODES ? 2 : 1; }
// (two tracers: and the second one's w cotangent; in one set, its w_i cotangent too)
size_t adjoint_cols_node(const DevMesh& m, int nt, int sets) {
    return sets * node_stride(m) + ((nt > 1) + (nt > sets)) * (size_t)m.N * m.L;
}
// (two tracers in one set: and the second one's vflux cotangent)
size_t adjoint_cols_edge(const DevMesh& m, int nt, int sets) {
    return sets * edge_stride(m) + (nt > sets) * (size_t)m.D * m.L;
}
size_t adjoint_cols_elem(const DevMesh& m, int sets) { return sets * elem_stride(m); }

int launch_backward_cols(const DevMesh& m, const NodeTab& tab, const int2* ekr, const FusedTape& tp,
                         const AdjointCols& w, const FusedTuning& tune, const fct_step_args* f,
                         const double* const* g_out, double* const* gT, double* const* gTold,
                         double* g_uv, double* g_w, double* g_wi, hipStream_t s) {
    const size_t NL = (size_t)m.N * m.L, DL = (size_t)m.D * m.L;
    ColArgs a{};
    a.m = m; a.tab = tab; a.ekr = ekr; a.remap = tune.remap(); a.dt = f->dt;
    a.helem = f->helem; a.w_e = f->w_e; a.w_i = f->w_i; a.Z3d = f->Z3d; a.zbar3 = f->zbar3;
    a.hnode = f->hnode; a.hnn = f->hnode_new;
    a.vflux = tp.vflux;
    double* p = w.node;
    auto take = [&](size_t n) { double* q = p; p += n * NL; return q; };
    // pairs first: 16-byte alignment whatever N * L
    for (double2** q : {&a.gpm, &a.tv, &a.sh, &a.gd, &a.gnum}) *q = reinterpret_cast<double2*>(take(2));
    for (double** q : {&a.ghsc, &a.gA, &a.gadfv, &a.gLO}) *q = take(1);
    double* own_wi = take(1);
    a.eg = reinterpret_cast<double2*>(w.edge);
    a.edge_up = w.edge_up;
    a.g_tr = reinterpret_cast<double2*>(w.elem);
    a.node_stride = node_stride(m); a.edge_stride = edge_stride(m); a.elem_stride = elem_stride(m);
    // Small meshes sum the even and the odd tracers' uv and w cotangents apart, whether a
    // launch takes two tracers or one (a plan with one slot): the bits do not depend on it.
    const bool pairs = w.tracers == 2 && f->ntracers >= 2;
    const bool own_set = w.sets == 2;      // the odd tracers' lie in the second set
    double* more = w.node + w.sets * a.node_stride;
    double* vf[2] = {w.edge + 2 * DL, w.edge + a.edge_stride + (own_set ? 2 * DL : 0)};
    double* gw[2] = {g_w, g_w ? more : nullptr};
    double* gwi[2] = {nullptr, nullptr};
    if (f->w_i) {
        gwi[0] = g_wi ? g_wi : own_wi;
        gwi[1] = own_set ? own_wi + a.node_stride : more + NL;
    }
    a.ud_off = w.ud_off; a.ud_ent = w.ud_ent; a.et_off = w.et_off; a.et_ent = w.et_ent;
    int rc;
    for (int j0 = 0; j0 < f->ntracers; j0 += tp.kw) {
        const int K = f->ntracers - j0 < tp.kw ? f->ntracers - j0 : tp.kw;
        if ((rc = launch_tape(m, tab, ekr, f, j0, K, tune, tp, s))) return rc;
        for (int j = 0, n = 1; j < K; j += n) {
            const int t = j0 + j, odd = pairs ? t & 1 : 0;
            n = pairs && !odd && K - j >= 2 ? 2 : 1;
            const int t1 = t + n - 1;
            a.first = pairs ? t < 2 : t == 0;
            const bool halves = n == 2 && m.N >= HALF_NODES;
            a.g_vf = vf[odd]; a.gw = gw[odd]; a.gwi = gwi[odd];
            a.gw1 = gw[1]; a.gwi1 = gwi[1];
            a.T = f->T[t]; a.Told = f->T_old[t]; a.g_out = g_out[t];
            a.gT = gT[t]; a.gTold = gTold[t];
            a.T1 = f->T[t1]; a.Told1 = f->T_old[t1]; a.g_out1 = g_out[t1];
            a.gT1 = gT[t1]; a.gTold1 = gTold[t1];
            a.LO = tp.LO + j * NL; a.adfh = tp.adfh + j * DL; a.adfv = tp.adfv + j * NL;
            a.pm = reinterpret_cast<const double2*>(tp.pf) + j * NL;
            a.gnode = reinterpret_cast<const double2*>(tp.gnode) + j * NL;
            const double* LOx = tp.LOx ? tp.LOx + j * NL : nullptr;
            const auto reverse = [&](auto ns) {
                constexpr int NS = decltype(ns)::value;
                if (tab.dm == 6)
                    return halves ? reverse_tracers<NS, 6, true>(a, LOx, n, s) : reverse_tracers<NS, 6, false>(a, LOx, n, s);
                return halves ? reverse_tracers<NS, 8, true>(a, LOx, n, s) : reverse_tracers<NS, 8, false>(a, LOx, n, s);
            };
            rc = m.L <= 64 ? reverse(std::integral_constant<int, 1>{}) : reverse(std::integral_constant<int, 2>{});
            if (rc) return rc;
        }
    }
    a.g_vf = vf[0];
    if (pairs) {
        a.g_vf1 = vf[1];
        double* wi = f->w_i ? g_wi : nullptr;
        if (g_w || wi) {
            kc_add<<<dim3((unsigned)((NL + 255) / 256)), dim3(256), 0, s>>>(NL, g_w, gw[1], wi, gwi[1]);
            if ((rc = check_launch("kc_add"))) return rc;
        }
    }
    if (!g_uv) return FCT_OK;
    return m.L <= 64 ? reverse_uv<1>(a, g_uv, s) : reverse_uv<2>(a, g_uv, s);
}

}  // namespace fct
