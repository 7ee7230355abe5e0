// Sea-ice FCT advection of the three ice tracers (fct_solve, fesom_jax/ice_adv.py:37-194):
// Taylor-Galerkin right-hand side, consistent-mass low- and high-order solves, element
// antidiffusive fluxes and the Zalesak limiter, on the surface nodes.
//
// Mapping: one thread per node and all three tracers per thread (the problem is 2-D;
// the tracers share every geometry load). Each node gathers over its elements in
// increasing element id, which is the order of the reference's scatter-add over (element,
// vertex); sums over an element's three vertices run ((x0 + x1) + x2). Six launches: the
// inputs packed per node, then five gather passes over the elements around every node:
// right-hand side + low-order solve, two high-order corrections (the second also stores
// each node's gamma * X + d, the vertex value of the antidiffusive fluxes), fluxes +
// bounds + ratios, limited fluxes + update.
//
// On meshes with the fused node tables (ki_*) a node's neighbours and elements come from
// tables with one row per slot ([slot][node], whole lines read), so that all its gathers
// leave together: the vertices of its elements are its neighbours (six gathers instead of
// eighteen), kept in the thread's own LDS column and picked by a 4-bit code per vertex. What
// bounded the walk over the element lists (k_ice_*, kept for other meshes) was the chain
// list entry -> element -> vertices, six times over: icosa-8 surface 371 us, 188 here
// (ki_hi 22, at the 19 us its 200 bytes per node take; ki_rhs 50, ki_ratio 42 and ki_apply
// 43 against 35, 22 and 21: they hold 200 registers of gathered values, so eight wavefronts
// per CU; capped to 168 registers they spill and take twice as long).
//
// Layout: the three tracers of a node sit together (dv4, the fourth slot carrying the
// node's inverse area where a pass needs it), (u, v) as a pair, and an element's gradient
// coefficients, volume and diffusion factor in four dv2.

#include <hip/hip_runtime.h>

#include "fct_common.h"

namespace fct {
namespace {

template <class T>
using gp = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gp<T> glb(T* p) { return (gp<T>)p; }

// packed per-node and per-element values as clang vectors (HIP's vector types are
// classes, which do not load through address-space pointers)
typedef double dv2 __attribute__((ext_vector_type(2)));
typedef double dv4 __attribute__((ext_vector_type(4)));
typedef int iv4 __attribute__((ext_vector_type(4)));

constexpr double ICE_FLUX_EPS = 1.0e-12;   // ice_adv.py:32
constexpr int ICE_K = 3;                   // a_ice, m_ice, m_snow

struct IceArgs {
    int N;
    double dt, diff, gamma;
    const int* ncsr_off;
    const int* ncsr;
    const iv4* el;          // [E] (v0, v1, v2, 1 if the element is open: ulevels <= 1)
    const dv2* eg;          // [E][4] (dx0, dx1), (dx2, dy0), (dy1, dy2), (vol, sqrt(vol/2e8))
    const int* nlev;        // [N*2] (ulevels_nod2D-1, nlevels_nod2D-1)
    const dv4* X;           // [N] (a_ice, m_ice, m_snow, 0), packed from the inputs
    const dv2* uv;          // [N] (u, v)
    double* out[ICE_K];     // tracers out
    dv4* rhs;               // [N] right-hand side
    dv4* xl;                // [N] low-order solution; .w = 1 / surface area
    dv4* d0;                // [N] high-order increment (ping)
    dv4* d1;                // [N] (pong)
    dv4* w;                 // [N] gamma * X + d with the final d; .w = 1 / surface area
    double* pp;             // [3][N] ratios
    double* pm;
};

__device__ __forceinline__ double comp(const dv4& v, int t) {
    return t == 0 ? v.x : (t == 1 ? v.y : v.z);
}
__device__ __forceinline__ bool node_open(const IceArgs& a, int n) {
    return glb(a.nlev)[2 * n] == 0;            // ulevels_nod2D <= 1
}
__device__ __forceinline__ int slot_of(int n, int v0, int v1) { return v0 == n ? 0 : (v1 == n ? 1 : 2); }
__device__ __forceinline__ double sum3(double x0, double x1, double x2) { return (x0 + x1) + x2; }
__device__ __forceinline__ double min1(double x) { return x > 1.0 ? 1.0 : x; }   // jnp.minimum(x, 1)

// The elements of node n in CSR order (increasing id). Each element's table entry is
// fetched one element ahead and its CSR entry two ahead, so that an element's vertex
// gathers need not wait behind the chain CSR entry -> element entry.
struct ElemWalk {
    int s, s1, e_next, e_after;
    iv4 ev_next;
    __device__ __forceinline__ ElemWalk(const IceArgs& a, int n) {
        s = glb(a.ncsr_off)[n];
        s1 = glb(a.ncsr_off)[n + 1];
        e_next = s < s1 ? glb(a.ncsr)[s] : 0;
        e_after = s + 1 < s1 ? glb(a.ncsr)[s + 1] : 0;
        ev_next = s < s1 ? glb(a.el)[e_next] : iv4{0, 0, 0, 0};
    }
    __device__ __forceinline__ bool next(const IceArgs& a, int& e, iv4& ev) {
        if (s >= s1) return false;
        e = e_next;
        ev = ev_next;
        e_next = e_after;
        if (s + 1 < s1) ev_next = glb(a.el)[e_next];
        if (s + 2 < s1) e_after = glb(a.ncsr)[s + 2];
        ++s;
        return true;
    }
};

// (mm X)[n]'s term of element e: vol/12 (X[n] + sum of the vertices)
__device__ __forceinline__ double mm_term(double vol, double xq, double x0, double x1, double x2) {
    return vol / 12.0 * (xq + sum3(x0, x1, x2));
}

// element tables, once per plan: vertices and open flag; gradient coefficients, volume
// and the diffusion factor sq (computed on the host)
__global__ void __launch_bounds__(256) k_ice_tables(int E, const int* __restrict__ en,
                                                    const int2* __restrict__ elev,
                                                    const double* __restrict__ gs,
                                                    const double* __restrict__ vol,
                                                    const double* __restrict__ sq,
                                                    iv4* __restrict__ el, dv2* __restrict__ eg) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    el[e] = iv4{en[3 * e], en[3 * e + 1], en[3 * e + 2], elev[e].x == 0 ? 1 : 0};
    eg[4 * e] = dv2{gs[6 * e], gs[6 * e + 1]};
    eg[4 * e + 1] = dv2{gs[6 * e + 2], gs[6 * e + 3]};
    eg[4 * e + 2] = dv2{gs[6 * e + 4], gs[6 * e + 5]};
    eg[4 * e + 3] = dv2{vol[e], sq[e]};
}

// the inputs packed per node
__global__ void __launch_bounds__(256) k_ice_pack(int N, const double* __restrict__ a0,
                                                  const double* __restrict__ a1,
                                                  const double* __restrict__ a2,
                                                  const double* __restrict__ u,
                                                  const double* __restrict__ v,
                                                  dv4* __restrict__ X, dv2* __restrict__ uv) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    X[n] = dv4{a0[n], a1[n], a2[n], 0.0};
    uv[n] = dv2{u[n], v[n]};
}

// pass 1: right-hand side (ice_adv.py:47-73), low-order solution (:76-87) and the first
// high-order approximation rhs / area (:101)
__global__ void __launch_bounds__(256) k_ice_rhs(IceArgs a, const double* __restrict__ area,
                                                 int L) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.N) return;
    const auto UV = glb(a.uv);
    const auto X = glb(a.X);
    double rhs[ICE_K] = {0.0, 0.0, 0.0}, mm[ICE_K] = {0.0, 0.0, 0.0};
    const dv4 xn = X[n];
    ElemWalk wk(a, n);
    int e;
    iv4 ev;
    while (wk.next(a, e, ev)) {
        const int vv[3] = {ev.x, ev.y, ev.z};
        const int q = slot_of(n, vv[0], vv[1]);
        const bool on = ev.w != 0;
        const dv2 g0 = glb(a.eg)[4 * e], g1 = glb(a.eg)[4 * e + 1];
        const dv2 g2 = glb(a.eg)[4 * e + 2], g3 = glb(a.eg)[4 * e + 3];
        const double dx[3] = {g0.x, g0.y, g1.x}, dy[3] = {g1.y, g2.x, g2.y};
        const double vol = g3.x;
        double Uv[3], Vv[3];
        dv4 xv[3];
        for (int i = 0; i < 3; ++i) {
            const dv2 w = UV[vv[i]];
            Uv[i] = w.x;
            Vv[i] = w.y;
            xv[i] = X[vv[i]];
        }
        const double um = sum3(Uv[0], Uv[1], Uv[2]), vm = sum3(Vv[0], Vv[1], Vv[2]);
        const double diff = a.diff * g3.y;
        const double udn_q = um * dx[q] + vm * dy[q];
        double ent[3];
        for (int j = 0; j < 3; ++j) {
            const double ta = (dx[q] * (um + Uv[j]) + dy[q] * (vm + Vv[j])) / 12.0;
            const double tb = diff * (dx[q] * dx[j] + dy[q] * dy[j]);
            const double udn_j = um * dx[j] + vm * dy[j];
            const double tc = 0.5 * a.dt * (udn_q * udn_j) / 9.0;
            ent[j] = vol * a.dt * (ta - tb - tc);
        }
        for (int t = 0; t < ICE_K; ++t) {
            const double x0 = comp(xv[0], t), x1 = comp(xv[1], t), x2 = comp(xv[2], t);
            const double c = (ent[0] * x0 + ent[1] * x1) + ent[2] * x2;
            const double xq = q == 0 ? x0 : (q == 1 ? x1 : x2);
            rhs[t] = rhs[t] + (on ? c : 0.0);
            mm[t] = mm[t] + (on ? mm_term(vol, xq, x0, x1, x2) : 0.0);
        }
    }
    const double ar = glb(area)[(size_t)n * L];
    const double inv = 1.0 / (ar > 0 ? ar : 1.0);
    const bool nc = node_open(a, n);
    double xl[ICE_K], d[ICE_K];
    for (int t = 0; t < ICE_K; ++t) {
        const double x = comp(xn, t);
        xl[t] = nc ? (rhs[t] + a.gamma * mm[t]) * inv + (1.0 - a.gamma) * x : x;
        d[t] = nc ? rhs[t] * inv : 0.0;
    }
    glb(a.rhs)[n] = dv4{rhs[0], rhs[1], rhs[2], 0.0};
    glb(a.xl)[n] = dv4{xl[0], xl[1], xl[2], inv};
    glb(a.d0)[n] = dv4{d[0], d[1], d[2], 0.0};
}

// pass 2 (twice): d <- d + (rhs - mm d) / area (ice_adv.py:102-104); the second pass also
// stores gamma * X + d (wout), the vertex value of the antidiffusive fluxes
__global__ void __launch_bounds__(256) k_ice_hi(IceArgs a, const dv4* din, dv4* dout,
                                                dv4* wout) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.N) return;
    const auto D = glb(din);
    double mm[ICE_K] = {0.0, 0.0, 0.0};
    // one element ahead: its area and vertex values load while this one is summed
    ElemWalk wk(a, n);
    int e;
    iv4 ev;
    bool more = wk.next(a, e, ev);
    double vol_n = 0.0;
    dv4 dn0 = {}, dn1 = {}, dn2 = {};
    if (more) {
        vol_n = glb(a.eg)[4 * e + 3].x;
        dn0 = D[ev.x]; dn1 = D[ev.y]; dn2 = D[ev.z];
    }
    while (more) {
        const int q = slot_of(n, ev.x, ev.y);
        const bool on = ev.w != 0;
        const double vol = vol_n;
        const dv4 d0 = dn0, d1 = dn1, d2 = dn2;
        more = wk.next(a, e, ev);
        if (more) {
            vol_n = glb(a.eg)[4 * e + 3].x;
            dn0 = D[ev.x]; dn1 = D[ev.y]; dn2 = D[ev.z];
        }
        for (int t = 0; t < ICE_K; ++t) {
            const double x0 = comp(d0, t), x1 = comp(d1, t), x2 = comp(d2, t);
            const double xq = q == 0 ? x0 : (q == 1 ? x1 : x2);
            mm[t] = mm[t] + (on ? mm_term(vol, xq, x0, x1, x2) : 0.0);
        }
    }
    const dv4 xl = glb(a.xl)[n];
    const double inv = xl.w;
    const bool nc = node_open(a, n);
    const dv4 dv = D[n], r = glb(a.rhs)[n];
    double dn[ICE_K];
    for (int t = 0; t < ICE_K; ++t) {
        const double d = comp(dv, t);
        dn[t] = nc ? d + (comp(r, t) - mm[t]) * inv : d;
    }
    glb(dout)[n] = dv4{dn[0], dn[1], dn[2], 0.0};
    if (wout) {
        const dv4 x = glb(a.X)[n];
        glb(wout)[n] = dv4{a.gamma * x.x + dn[0], a.gamma * x.y + dn[1],
                           a.gamma * x.z + dn[2], inv};
    }
}

// antidiffusive flux of element e at its vertex q for one tracer (ice_adv.py:125-130):
// ice_flux = ice_flux_num / 12
__device__ __forceinline__ double ice_flux_num(const double (&w)[3], int q, double vol,
                                               double inv_q) {
    const double s = sum3(w[0], w[1], w[2]) - 3.0 * w[q];
    return -s * (vol * inv_q);
}
__device__ __forceinline__ double ice_flux(double g, const double (&w)[3], int q, double vol,
                                           double inv_q) {
    return ice_flux_num(w, q, vol, inv_q) / 12.0;
}
// ice_flux(...) >= 0.0 from its numerator g, without the division: g / 12 rounds to a
// value >= 0 (or to -0) exactly when g >= -6 * 2^-1074 (|g / 12| <= 2^-1075 rounds to
// zero, ties to even); NaN compares false either way
__device__ __forceinline__ bool ice_flux_nonneg(double g) { return g >= -0x6p-1074; }

// pass 3: flux sums, cluster bounds and clipping ratios of every node (ice_adv.py:132-160)
__global__ void __launch_bounds__(256) k_ice_ratio(IceArgs a) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.N) return;
    const auto W = glb(a.w);
    const auto XL = glb(a.xl);
    const auto X = glb(a.X);
    const dv4 xln = XL[n];
    const double inv = xln.w;
    double fp[ICE_K] = {0.0, 0.0, 0.0}, fm[ICE_K] = {0.0, 0.0, 0.0};
    double hi[ICE_K], lo[ICE_K];
    for (int t = 0; t < ICE_K; ++t) { hi[t] = -INFINITY; lo[t] = INFINITY; }
    ElemWalk wk(a, n);
    int e;
    iv4 ev;
    while (wk.next(a, e, ev)) {
        const int vv[3] = {ev.x, ev.y, ev.z};
        const int q = slot_of(n, vv[0], vv[1]);
        const bool on = ev.w != 0;
        const double vol = glb(a.eg)[4 * e + 3].x;
        dv4 xv[3], lv[3], wv[3];
        for (int j = 0; j < 3; ++j) {
            xv[j] = X[vv[j]];
            lv[j] = XL[vv[j]];
            wv[j] = W[vv[j]];
        }
        for (int t = 0; t < ICE_K; ++t) {
            double w[3], eh = -INFINITY, el = INFINITY;
            for (int j = 0; j < 3; ++j) {
                const double x = comp(xv[j], t), l = comp(lv[j], t);
                w[j] = comp(wv[j], t);
                eh = fmax(eh, fmax(l, x));
                el = fmin(el, fmin(l, x));
            }
            const double f = on ? ice_flux(a.gamma, w, q, vol, inv) : 0.0;
            fp[t] = fp[t] + fmax(f, 0.0);
            fm[t] = fm[t] + fmin(f, 0.0);
            if (on) {
                hi[t] = fmax(hi[t], eh);
                lo[t] = fmin(lo[t], el);
            }
        }
    }
    const bool nc = node_open(a, n);
    for (int t = 0; t < ICE_K; ++t) {
        const size_t i = (size_t)t * a.N + n;
        const double h = isfinite(hi[t]) ? hi[t] : 0.0, l = isfinite(lo[t]) ? lo[t] : 0.0;
        const double xl = comp(xln, t);
        const double tmax = h - xl, tmin = l - xl;
        double p = fp[t] > 0.0 ? min1(tmax / (fp[t] > ICE_FLUX_EPS ? fp[t] : ICE_FLUX_EPS)) : 0.0;
        double m = fm[t] < 0.0 ? min1(tmin / (fm[t] < -ICE_FLUX_EPS ? fm[t] : -ICE_FLUX_EPS)) : 0.0;
        glb(a.pp)[i] = nc ? p : 0.0;
        glb(a.pm)[i] = nc ? m : 0.0;
    }
}

// pass 4: each element's fluxes limited by the smallest ratio of its vertices, summed
// into the node, added to the low-order solution (ice_adv.py:162-169)
__global__ void __launch_bounds__(256) k_ice_apply(IceArgs a) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.N) return;
    const auto W = glb(a.w);
    const auto PP = glb(a.pp), PM = glb(a.pm);
    double acc[ICE_K] = {0.0, 0.0, 0.0};
    // one element ahead: its area and vertex values load while this one is summed
    ElemWalk wk(a, n);
    int e;
    iv4 ev;
    bool more = wk.next(a, e, ev);
    double vol_n = 0.0;
    dv4 wn[3] = {};
    if (more) {
        vol_n = glb(a.eg)[4 * e + 3].x;
        wn[0] = W[ev.x]; wn[1] = W[ev.y]; wn[2] = W[ev.z];
    }
    while (more) {
        const int vv[3] = {ev.x, ev.y, ev.z};
        const int q = slot_of(n, vv[0], vv[1]);
        const bool on = ev.w != 0;
        const double vol = vol_n;
        // the vertices' gamma * X + d, with their inverse areas in the fourth slot
        const dv4 wv[3] = {wn[0], wn[1], wn[2]};
        more = wk.next(a, e, ev);
        if (more) {
            vol_n = glb(a.eg)[4 * e + 3].x;
            wn[0] = W[ev.x]; wn[1] = W[ev.y]; wn[2] = W[ev.z];
        }
        for (int t = 0; t < ICE_K; ++t) {
            const size_t o = (size_t)t * a.N;
            double w[3];
            for (int j = 0; j < 3; ++j) w[j] = comp(wv[j], t);
            // the element's factor takes each vertex's ratio by the sign of that vertex's
            // flux (0 when the element is closed); only the node's own flux is divided
            double ae = INFINITY, gq = 0.0;
            for (int j = 0; j < 3; ++j) {
                const double g = ice_flux_num(w, j, vol, wv[j].w);
                gq = j == q ? g : gq;
                ae = fmin(ae, !on || ice_flux_nonneg(g) ? PP[o + vv[j]] : PM[o + vv[j]]);
            }
            acc[t] = acc[t] + (on ? (gq / 12.0) * ae : 0.0);
        }
    }
    const dv4 xl = glb(a.xl)[n];
    for (int t = 0; t < ICE_K; ++t) glb(a.out[t])[n] = comp(xl, t) + acc[t];
}

// ---------------------------------------------------------------------------
// slot tables (meshes with node tables): neighbours, elements and vertex codes per slot
// ---------------------------------------------------------------------------
struct IceSlots {
    int N;
    const int* nbr;             // [DM][N] node of the slot
    const int* eid;             // [DM][N] element of the slot, increasing id
    const unsigned short* code; // [DM][N] 4 bits per vertex: the slot it is, or DM the node
                                // itself; bit 12: an open element (padding slots: not)
    const unsigned short* open; // [N] node open (ulevels_nod2D <= 1)
    const double* inv;          // [N] 1 / surface area
    const double* vol;          // [E]
};
constexpr int ICE_TB = 128;     // threads per workgroup of the slot passes

__global__ void __launch_bounds__(256) ki_slots(int N, int L, int dm, const int4* __restrict__ hdr,
                                                const int4* __restrict__ edge,
                                                const int4* __restrict__ elem,
                                                const int2* __restrict__ elev,
                                                const double* __restrict__ area, int* __restrict__ nbr,
                                                int* __restrict__ eid, unsigned short* __restrict__ code,
                                                unsigned short* __restrict__ open,
                                                double* __restrict__ inv) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    const int4 h = hdr[n];
    for (int q = 0; q < dm; ++q) {
        const int4 es = edge[(size_t)n * dm + q];
        const int e = elem[(size_t)n * dm + q].x;
        nbr[(size_t)q * N + n] = es.y;
        eid[(size_t)q * N + n] = e;
        const bool on = q < h.w && elev[e].x == 0;
        code[(size_t)q * N + n] = (unsigned short)((((unsigned)es.w >> 16) & 0xfffu) | (on ? 0x1000u : 0u));
    }
    open[n] = h.x == 0;
    const double ar = area[(size_t)n * L];
    inv[n] = 1.0 / (ar > 0 ? ar : 1.0);
}

// The thread's LDS column: row r of its DM neighbours' (and, last, its own) values.
template <int DM>
struct IceCol {
    double* p;
    __device__ __forceinline__ double& at(int row, int slot) const {
        return p[(size_t)(row * (DM + 1) + slot) * ICE_TB];
    }
};
__device__ __forceinline__ int vslot(unsigned c, int i) { return (int)(c >> (4 * i)) & 0xf; }
template <int DM>
__device__ __forceinline__ int own_vertex(unsigned c) {
    return vslot(c, 0) == DM ? 0 : (vslot(c, 1) == DM ? 1 : 2);
}
template <int DM>
__device__ __forceinline__ void slots_of(const IceSlots& t, int n, int (&nb)[DM], unsigned (&cd)[DM]) {
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        nb[q] = glb(t.nbr)[(size_t)q * t.N + n];
        cd[q] = glb(t.code)[(size_t)q * t.N + n];
    }
}

template <int DM>
__global__ void __launch_bounds__(ICE_TB) ki_rhs(IceArgs a, IceSlots t) {
    __shared__ double sh[5 * (DM + 1) * ICE_TB];
    const int n = blockIdx.x * ICE_TB + threadIdx.x;
    if (n >= a.N) return;
    const IceCol<DM> col{sh + threadIdx.x};
    int nb[DM], el[DM];
    unsigned cd[DM];
    slots_of<DM>(t, n, nb, cd);
#pragma unroll
    for (int q = 0; q < DM; ++q) el[q] = glb(t.eid)[(size_t)q * t.N + n];
    const dv4 xn = glb(a.X)[n];
    {
        dv4 x[DM + 1];
        dv2 w[DM + 1];
#pragma unroll
        for (int q = 0; q < DM; ++q) { x[q] = glb(a.X)[nb[q]]; w[q] = glb(a.uv)[nb[q]]; }
        x[DM] = xn;
        w[DM] = glb(a.uv)[n];
#pragma unroll
        for (int q = 0; q <= DM; ++q) {
            col.at(0, q) = x[q].x; col.at(1, q) = x[q].y; col.at(2, q) = x[q].z;
            col.at(3, q) = w[q].x; col.at(4, q) = w[q].y;
        }
    }
    double rhs[ICE_K] = {0.0, 0.0, 0.0}, mm[ICE_K] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < DM; ++s) {
        const size_t e = (size_t)el[s];
        const dv2 g0 = glb(a.eg)[4 * e], g1 = glb(a.eg)[4 * e + 1];
        const dv2 g2 = glb(a.eg)[4 * e + 2], g3 = glb(a.eg)[4 * e + 3];
        const int v[3] = {vslot(cd[s], 0), vslot(cd[s], 1), vslot(cd[s], 2)};
        const int q = own_vertex<DM>(cd[s]);
        const bool on = cd[s] & 0x1000u;
        const double dx[3] = {g0.x, g0.y, g1.x}, dy[3] = {g1.y, g2.x, g2.y};
        const double dxq = q == 0 ? dx[0] : (q == 1 ? dx[1] : dx[2]);
        const double dyq = q == 0 ? dy[0] : (q == 1 ? dy[1] : dy[2]);
        const double vol = g3.x;
        double U[3], V[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) { U[i] = col.at(3, v[i]); V[i] = col.at(4, v[i]); }
        const double um = sum3(U[0], U[1], U[2]), vm = sum3(V[0], V[1], V[2]);
        const double diff = a.diff * g3.y;
        const double udn_q = um * dxq + vm * dyq;
        double ent[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double ta = (dxq * (um + U[j]) + dyq * (vm + V[j])) / 12.0;
            const double tb = diff * (dxq * dx[j] + dyq * dy[j]);
            const double udn_j = um * dx[j] + vm * dy[j];
            const double tc = 0.5 * a.dt * (udn_q * udn_j) / 9.0;
            ent[j] = vol * a.dt * (ta - tb - tc);
        }
#pragma unroll
        for (int k = 0; k < ICE_K; ++k) {
            const double x0 = col.at(k, v[0]), x1 = col.at(k, v[1]), x2 = col.at(k, v[2]);
            const double c = (ent[0] * x0 + ent[1] * x1) + ent[2] * x2;
            rhs[k] = rhs[k] + (on ? c : 0.0);
            mm[k] = mm[k] + (on ? mm_term(vol, comp(xn, k), x0, x1, x2) : 0.0);
        }
    }
    const double inv = glb(t.inv)[n];
    const bool nc = glb(t.open)[n];
    double xl[ICE_K], d[ICE_K];
#pragma unroll
    for (int k = 0; k < ICE_K; ++k) {
        const double x = comp(xn, k);
        xl[k] = nc ? (rhs[k] + a.gamma * mm[k]) * inv + (1.0 - a.gamma) * x : x;
        d[k] = nc ? rhs[k] * inv : 0.0;
    }
    glb(a.rhs)[n] = dv4{rhs[0], rhs[1], rhs[2], 0.0};
    glb(a.xl)[n] = dv4{xl[0], xl[1], xl[2], inv};
    glb(a.d0)[n] = dv4{d[0], d[1], d[2], 0.0};
}

template <int DM>
__global__ void __launch_bounds__(ICE_TB) ki_hi(IceArgs a, IceSlots t, const dv4* din, dv4* dout,
                                                dv4* wout) {
    __shared__ double sh[3 * (DM + 1) * ICE_TB];
    const int n = blockIdx.x * ICE_TB + threadIdx.x;
    if (n >= a.N) return;
    const IceCol<DM> col{sh + threadIdx.x};
    int nb[DM];
    unsigned cd[DM];
    double vol[DM];
    slots_of<DM>(t, n, nb, cd);
#pragma unroll
    for (int q = 0; q < DM; ++q) vol[q] = glb(t.vol)[glb(t.eid)[(size_t)q * t.N + n]];
    const dv4 dv = glb(din)[n], r = glb(a.rhs)[n];
    {
        dv4 x[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) x[q] = glb(din)[nb[q]];
#pragma unroll
        for (int q = 0; q < DM; ++q) { col.at(0, q) = x[q].x; col.at(1, q) = x[q].y; col.at(2, q) = x[q].z; }
        col.at(0, DM) = dv.x; col.at(1, DM) = dv.y; col.at(2, DM) = dv.z;
    }
    double mm[ICE_K] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < DM; ++s) {
        const bool on = cd[s] & 0x1000u;
        const int v0 = vslot(cd[s], 0), v1 = vslot(cd[s], 1), v2 = vslot(cd[s], 2);
#pragma unroll
        for (int k = 0; k < ICE_K; ++k)
            mm[k] = mm[k] + (on ? mm_term(vol[s], comp(dv, k), col.at(k, v0), col.at(k, v1), col.at(k, v2))
                                : 0.0);
    }
    const double inv = glb(t.inv)[n];
    const bool nc = glb(t.open)[n];
    double dn[ICE_K];
#pragma unroll
    for (int k = 0; k < ICE_K; ++k) {
        const double d = comp(dv, k);
        dn[k] = nc ? d + (comp(r, k) - mm[k]) * inv : d;
    }
    if (dout) glb(dout)[n] = dv4{dn[0], dn[1], dn[2], 0.0};
    if (wout) {
        const dv4 x = glb(a.X)[n];
        glb(wout)[n] = dv4{a.gamma * x.x + dn[0], a.gamma * x.y + dn[1], a.gamma * x.z + dn[2], inv};
    }
}

// pp4, pm4: the ratios of the three tracers per node
template <int DM>
__global__ void __launch_bounds__(ICE_TB) ki_ratio(IceArgs a, IceSlots t, dv4* pp4, dv4* pm4) {
    __shared__ double sh[3 * (DM + 1) * ICE_TB];
    const int n = blockIdx.x * ICE_TB + threadIdx.x;
    if (n >= a.N) return;
    const IceCol<DM> col{sh + threadIdx.x};
    int nb[DM];
    unsigned cd[DM];
    double vol[DM];
    slots_of<DM>(t, n, nb, cd);
#pragma unroll
    for (int q = 0; q < DM; ++q) vol[q] = glb(t.vol)[glb(t.eid)[(size_t)q * t.N + n]];
    const dv4 xn = glb(a.X)[n], xln = glb(a.xl)[n], wn = glb(a.w)[n];
    dv4 xv[DM], lv[DM], wv[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) { xv[q] = glb(a.X)[nb[q]]; lv[q] = glb(a.xl)[nb[q]]; wv[q] = glb(a.w)[nb[q]]; }
    const double inv = xln.w;
    const bool nc = glb(t.open)[n];
    double p[ICE_K], m[ICE_K];
#pragma unroll
    for (int k = 0; k < ICE_K; ++k) {
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const double x = comp(xv[q], k), l = comp(lv[q], k);
            col.at(0, q) = comp(wv[q], k);
            col.at(1, q) = fmax(l, x);
            col.at(2, q) = fmin(l, x);
        }
        const double xl = comp(xln, k);
        col.at(0, DM) = comp(wn, k);
        col.at(1, DM) = fmax(xl, comp(xn, k));
        col.at(2, DM) = fmin(xl, comp(xn, k));
        double fp = 0.0, fm = 0.0, hi = -INFINITY, lo = INFINITY;
#pragma unroll
        for (int s = 0; s < DM; ++s) {
            const int v0 = vslot(cd[s], 0), v1 = vslot(cd[s], 1), v2 = vslot(cd[s], 2);
            const bool on = cd[s] & 0x1000u;
            // ice_flux with the node's own value as w[q]
            const double su = sum3(col.at(0, v0), col.at(0, v1), col.at(0, v2)) - 3.0 * comp(wn, k);
            const double f = on ? -su * (vol[s] * inv) / 12.0 : 0.0;
            fp = fp + fmax(f, 0.0);
            fm = fm + fmin(f, 0.0);
            const double eh = fmax(fmax(col.at(1, v0), col.at(1, v1)), col.at(1, v2));
            const double el = fmin(fmin(col.at(2, v0), col.at(2, v1)), col.at(2, v2));
            hi = on ? fmax(hi, eh) : hi;
            lo = on ? fmin(lo, el) : lo;
        }
        const double h = isfinite(hi) ? hi : 0.0, l = isfinite(lo) ? lo : 0.0;
        const double tmax = h - xl, tmin = l - xl;
        p[k] = fp > 0.0 ? min1(tmax / (fp > ICE_FLUX_EPS ? fp : ICE_FLUX_EPS)) : 0.0;
        m[k] = fm < 0.0 ? min1(tmin / (fm < -ICE_FLUX_EPS ? fm : -ICE_FLUX_EPS)) : 0.0;
        p[k] = nc ? p[k] : 0.0;
        m[k] = nc ? m[k] : 0.0;
    }
    glb(pp4)[n] = dv4{p[0], p[1], p[2], 0.0};
    glb(pm4)[n] = dv4{m[0], m[1], m[2], 0.0};
}

template <int DM>
__global__ void __launch_bounds__(ICE_TB) ki_apply(IceArgs a, IceSlots t, const dv4* pp4,
                                                   const dv4* pm4) {
    __shared__ double sh[4 * (DM + 1) * ICE_TB];
    const int n = blockIdx.x * ICE_TB + threadIdx.x;
    if (n >= a.N) return;
    const IceCol<DM> col{sh + threadIdx.x};
    int nb[DM];
    unsigned cd[DM];
    double vol[DM];
    slots_of<DM>(t, n, nb, cd);
#pragma unroll
    for (int q = 0; q < DM; ++q) vol[q] = glb(t.vol)[glb(t.eid)[(size_t)q * t.N + n]];
    const dv4 wn = glb(a.w)[n], ppn = glb(pp4)[n], pmn = glb(pm4)[n], xl = glb(a.xl)[n];
    dv4 wv[DM], pv[DM], mv[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) { wv[q] = glb(a.w)[nb[q]]; pv[q] = glb(pp4)[nb[q]]; mv[q] = glb(pm4)[nb[q]]; }
#pragma unroll
    for (int q = 0; q < DM; ++q) col.at(3, q) = wv[q].w;
    col.at(3, DM) = wn.w;
#pragma unroll
    for (int k = 0; k < ICE_K; ++k) {
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            col.at(0, q) = comp(wv[q], k);
            col.at(1, q) = comp(pv[q], k);
            col.at(2, q) = comp(mv[q], k);
        }
        col.at(0, DM) = comp(wn, k);
        col.at(1, DM) = comp(ppn, k);
        col.at(2, DM) = comp(pmn, k);
        double acc = 0.0;
#pragma unroll
        for (int s = 0; s < DM; ++s) {
            const int v[3] = {vslot(cd[s], 0), vslot(cd[s], 1), vslot(cd[s], 2)};
            const bool on = cd[s] & 0x1000u;
            double w[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) w[j] = col.at(0, v[j]);
            const double su = sum3(w[0], w[1], w[2]);
            // the element's factor takes each vertex's ratio by the sign of that vertex's
            // flux (0 when the element is closed); only the node's own flux is divided
            double ae = INFINITY, gq = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double g = -(su - 3.0 * w[j]) * (vol[s] * col.at(3, v[j]));
                gq = v[j] == DM ? g : gq;
                ae = fmin(ae, col.at(!on || ice_flux_nonneg(g) ? 1 : 2, v[j]));
            }
            acc = acc + (on ? (gq / 12.0) * ae : 0.0);
        }
        glb(a.out[k])[n] = comp(xl, k) + acc;
    }
}

template <int DM>
void ice_slot_passes(const IceArgs& a, const IceSlots& t, hipStream_t s) {
    const dim3 grid((a.N + ICE_TB - 1) / ICE_TB), block(ICE_TB);
    ki_rhs<DM><<<grid, block, 0, s>>>(a, t);
    ki_hi<DM><<<grid, block, 0, s>>>(a, t, a.d0, a.d1, nullptr);
    ki_hi<DM><<<grid, block, 0, s>>>(a, t, a.d1, nullptr, a.w);
    // the ratios take the place of the right-hand side and of the first correction
    ki_ratio<DM><<<grid, block, 0, s>>>(a, t, a.rhs, a.d1);
    ki_apply<DM><<<grid, block, 0, s>>>(a, t, a.rhs, a.d1);
}

}  // namespace

// rhs, xl, d0, d1, w, X as dv4, (u, v) as dv2, pp and pm: 32 doubles per node
size_t ice_workspace_doubles(int N) { return (size_t)32 * N; }
// el (iv4) and eg (four dv2): 10 doubles per element
size_t ice_table_doubles(int E) { return (size_t)10 * E; }
// inverse areas, then neighbours and elements (int), codes and open flags (16 bits)
size_t ice_slot_bytes(int N, int dm) { return (size_t)N * (8 + 8 * dm + 2 * (dm + 1)); }

namespace {
IceSlots slots_at(const DevMesh& m, int dm, void* mem) {
    IceSlots t{};
    const size_t N = (size_t)m.N;
    char* p = static_cast<char*>(mem);
    t.N = m.N;
    t.vol = m.earea;
    t.inv = reinterpret_cast<double*>(p);
    t.nbr = reinterpret_cast<int*>(p + 8 * N);
    t.eid = t.nbr + N * dm;
    t.code = reinterpret_cast<unsigned short*>(p + 8 * N + 8 * N * dm);
    t.open = t.code + N * dm;
    return t;
}
}  // namespace

int launch_ice_slots(const DevMesh& m, const NodeTab& tab, void* mem, hipStream_t s) {
    if (m.N == 0) return FCT_OK;
    const IceSlots t = slots_at(m, tab.dm, mem);
    ki_slots<<<(m.N + 255) / 256, 256, 0, s>>>(m.N, m.L, tab.dm, tab.hdr, tab.edge, tab.elem, m.elev,
                                              m.area, const_cast<int*>(t.nbr), const_cast<int*>(t.eid),
                                              const_cast<unsigned short*>(t.code),
                                              const_cast<unsigned short*>(t.open),
                                              const_cast<double*>(t.inv));
    return check_launch("ki_slots");
}

int launch_ice_tables(const DevMesh& m, const double* sq, double* tab, hipStream_t s) {
    if (m.E == 0) return FCT_OK;
    iv4* el = reinterpret_cast<iv4*>(tab);
    dv2* eg = reinterpret_cast<dv2*>(tab + 2 * (size_t)m.E);
    k_ice_tables<<<(m.E + 255) / 256, 256, 0, s>>>(m.E, m.en, m.elev, m.gs, m.earea, sq, el, eg);
    return check_launch("k_ice_tables");
}

int launch_ice_fct(const DevMesh& m, const IceCall& c, double* work, const double* tab, int dm,
                   void* slots, hipStream_t s) {
    if (m.N == 0) return FCT_OK;
    IceArgs a{};
    a.N = m.N;
    a.dt = c.dt;
    a.diff = c.diff;
    a.gamma = c.gamma;
    a.ncsr_off = m.ncsr_off;
    a.ncsr = m.ncsr;
    a.el = reinterpret_cast<const iv4*>(tab);
    a.eg = reinterpret_cast<const dv2*>(tab + 2 * (size_t)m.E);
    a.nlev = reinterpret_cast<const int*>(m.nlev);
    for (int t = 0; t < ICE_K; ++t) a.out[t] = c.out[t];
    const size_t N = (size_t)m.N;
    dv4* w4 = reinterpret_cast<dv4*>(work);
    a.rhs = w4;
    a.xl = w4 + N;
    a.d0 = w4 + 2 * N;
    a.d1 = w4 + 3 * N;
    a.w = w4 + 4 * N;
    dv4* X = w4 + 5 * N;
    dv2* uv = reinterpret_cast<dv2*>(work + 24 * N);
    a.X = X;
    a.uv = uv;
    a.pp = work + 26 * N;
    a.pm = work + 29 * N;
    const dim3 grid((m.N + 255) / 256), block(256);
    k_ice_pack<<<grid, block, 0, s>>>(m.N, c.X[0], c.X[1], c.X[2], c.u, c.v, X, uv);
    if (dm) {
        const IceSlots t = slots_at(m, dm, slots);
        if (dm == 6) ice_slot_passes<6>(a, t, s);
        else ice_slot_passes<8>(a, t, s);
        return check_launch("ki");
    }
    k_ice_rhs<<<grid, block, 0, s>>>(a, m.area, m.L);
    k_ice_hi<<<grid, block, 0, s>>>(a, a.d0, a.d1, nullptr);
    k_ice_hi<<<grid, block, 0, s>>>(a, a.d1, a.d0, a.w);
    k_ice_ratio<<<grid, block, 0, s>>>(a);
    k_ice_apply<<<grid, block, 0, s>>>(a);
    return check_launch("k_ice");
}

}  // namespace fct
