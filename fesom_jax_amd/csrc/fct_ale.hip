// Vertical velocity from continuity, compute_w (fesom_jax/ale.py:309-365): the
// per-level antisymmetric edge divergence summed into each node, the bottom-to-top
// cumulative sum over the column, and the division by the interface area.
//
// Mapping: one 64-lane wavefront per node, lane = level (two slots for nl <= 128). The
// divergence sums the node's (edge, side) list in increasing 2e+side order from +0.0,
// the order of the reference's flattened segment sum (ops.py:56-81). The cumulative
// sum is sequential from the bottom, w[k] = w[k+1] + div[k], the order of the original
// C loop (for nz = nzmax-1 .. nzmin: w[nz] += w[nz+1]), run by one lane per column on
// the columns staged in LDS.
//
// Three forms of the divergence, term by term the same arithmetic in the same order.
// k_compute_w_tab (meshes whose nodes have rings) loads each of a node's triangles once:
// icosa-8 x 70 478 us, 278 for the compulsory bytes at the rate of a copy; with (u, v,
// helem) taken from LDS rows by slot and four columns summed per workgroup 890.
// k_compute_w_vf (other meshes with node tables) takes the terms from the FCT's edge volume
// flux, computed once per edge by kf_vflux: 869 us on that mesh (436 and 471), 1253 by
// k_compute_w.
//   term(e, k) = (v1 dx1 - u1 dy1) h1 - (v2 dx2 - u2 dy2) h2 = -vflux(e, k)
// exactly: x - y = -(y - x) and (-x) h = -(x h) in IEEE arithmetic, and a masked triangle
// gives +0 in both; a sum that starts at +0.0 absorbs the sign of a zero.
// k_compute_w evaluates each (edge, side) from the edge's two triangles, so that a node
// loads every triangle around it twice.

#include <hip/hip_runtime.h>

#include "fct_wave.h"

namespace fct {
namespace {

template <class T>
using gp = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gp<T> glb(T* p) { return (gp<T>)p; }

// stage 2 and 3 of k_compute_w and k_compute_w_vf for node n (valid: n < nod2D), whose divergence is div.
// Blocks are FCT_W_WPB wavefronts, one node each; every thread reaches the barriers.
constexpr int FCT_W_WPB = 4;
template <int NS>
__device__ __forceinline__ void finish_w(const DevMesh& m, int n, bool valid, int lane,
                                         const double (&div)[NS], double* w_) {
    __shared__ double s_col[FCT_W_WPB][128];
    const int L = m.L, wv = (int)(threadIdx.x >> 6);
    const auto nlev = glb(reinterpret_cast<const int*>(m.nlev));
    // stage 2: w[k] = w[k+1] + div[k], from the last level up to the surface interface
    // (the divergence is zero at and below nzmax on a consistent mesh, so the sum
    // starts at the bottom interface in practice; starting at the last level keeps
    // the oracle's reversed cumulative sum exactly, signed zeros included). The columns
    // go through LDS so that one lane per column runs the serial sum.
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = lane + 64 * s;
        if (k < L) s_col[wv][k] = div[s];
    }
    __syncthreads();
    if (threadIdx.x < FCT_W_WPB) {
        const int c = (int)threadIdx.x;
        const int nn = (int)blockIdx.x * FCT_W_WPB + c;
        if (nn < m.N) {
            const int zmin = nlev[2 * nn];
            double acc = 0.0;
#pragma unroll 8
            for (int k = L - 1; k >= zmin; --k) {
                const double d = s_col[c][k];
                acc = k == L - 1 ? d : acc + d;
                s_col[c][k] = acc;
            }
        }
    }
    __syncthreads();
    if (!valid) return;
    const auto w = glb(w_);
    const auto area = glb(m.area);
    const int nzmin = nlev[2 * n];
    const int nzmax = nlev[2 * n + 1];   // iface range end
    // stage 3: / area (safe), zero outside the interface range [nzmin, nzmax]
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = lane + 64 * s;
        if (k >= L) continue;
        const double wk = k >= nzmin ? s_col[wv][k] : 0.0;
        const size_t i = (size_t)n * L + k;
        const double a = area[i];
        const double v = wk / (a > 0.0 ? a : 1.0);
        w[i] = (k >= nzmin && k <= nzmax) ? v : 0.0;
    }
}

// divergence of node n from its own triangles (see the top of the file) into its LDS column:
// the ring gives each edge's two triangles at fixed slots; the terms go through the lane's
// LDS column into the node table's 2e+side order, which is that of the CSR list. On 8-slot
// tables a node with up to six neighbours takes the 6-slot loops.
template <int NS, int DM, int ST>
__device__ __forceinline__ void ring_divergence(const DevMesh& m, const NodeTab& tab, int n, int4 hd,
                                                const double* uv_, const double* helem_,
                                                double* term, double* col) {
    const int lane = threadIdx.x & 63, L = m.L;
    int4 r[DM];
    double4 cr[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) r[q] = ldc(tab.ring, (size_t)n * ST + q);
#pragma unroll
    for (int q = 0; q < DM; ++q) cr[q] = ldc(m.cross, r[q].z < 0 ? 0 : r[q].z >> 1);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = lane + 64 * s;
        double d = 0.0;
        if (k < hd.y) {      // no triangle reaches below the node's wet layers
            double2 w[DM];
            double h[DM];
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                const size_t i = (size_t)r[q].y * L + k;
                w[q] = ldv(reinterpret_cast<const double2*>(uv_), i);
                h[q] = G(helem_)[i];
            }
            bool in[DM];
#pragma unroll
            for (int q = 0; q < DM; ++q)
                in[q] = q > 0 && (r[q].w & FCT_RING_DUP) ? in[q > 0 ? q - 1 : 0] : in_bytes(r[q].w, 0, k);
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                if (r[q].z < 0) continue;
                const int b = (q + DM - 1) % DM;
                const bool prev = r[q].w & FCT_RING_PREV;    // the edge's triangles: (b, q) or (q, b)
                const double xb = prev ? cr[q].x : cr[q].z, yb = prev ? cr[q].y : cr[q].w;
                const double xq = prev ? cr[q].z : cr[q].x, yq = prev ? cr[q].w : cr[q].y;
                const double tb = in[b] ? (w[b].y * xb - w[b].x * yb) * h[b] : 0.0;
                const double tq = in[q] ? (w[q].y * xq - w[q].x * yq) * h[q] : 0.0;
                const double t = prev ? tb + -tq : tq + -tb;   // sign * where(mask, term, 0)
                term[((r[q].w >> 16) & 0xf) * 64] = (r[q].z & 1) ? -t : t;
            }
#pragma unroll
            for (int q = 0; q < DM; ++q)
                if (q < (hd.z & 0xff)) d = d + term[q * 64];
        }
        if (k < L) col[k] = d;
    }
}

// A workgroup's C columns are summed up together, one per lane of its first wavefront.
template <int NS, int DM>
__global__ void __launch_bounds__(256) k_compute_w_tab(DevMesh m, NodeTab tab, int C, int remap,
                                                       const double* uv, const double* helem,
                                                       double* w_) {
    extern __shared__ double s_w[];       // C columns of nl | 1, then the waves' terms
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int L = m.L, P = L | 1;
    const int n0 = (int)block_tile(remap) * C;
    const int nc = min(C, m.N - n0);
    double* term = s_w + C * P + wv * DM * 64 + lane;
#pragma unroll 1
    for (int c = wv; c < nc; c += 4) {
        const int4 hd = ldc(tab.hdr, n0 + c);
        if (DM > 6 && (hd.z & 0xff) <= 6)
            ring_divergence<NS, 6, DM>(m, tab, n0 + c, hd, uv, helem, term, s_w + c * P);
        else
            ring_divergence<NS, DM, DM>(m, tab, n0 + c, hd, uv, helem, term, s_w + c * P);
    }
    __syncthreads();
    if ((int)threadIdx.x < nc) {
        const int zmin = m.nlev[n0 + threadIdx.x].x;
        double* col = s_w + threadIdx.x * P;
        double acc = col[L - 1];
#pragma unroll 8
        for (int k = L - 2; k >= zmin; --k) {
            acc = acc + col[k];
            col[k] = acc;
        }
    }
    __syncthreads();
#pragma unroll 4
    for (int c = wv; c < nc; c += 4) {
        const int2 nr = m.nlev[n0 + c];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = lane + 64 * s;
            if (k >= L) continue;
            const size_t i = (size_t)(n0 + c) * L + k;
            double v = 0.0;
            if (k >= nr.x && k <= nr.y) {
                const double a = G(m.area)[i];
                v = s_w[c * P + k] / (a > 0.0 ? a : 1.0);
            }
            G(w_)[i] = v;
        }
    }
}

// divergence from the edge volume flux (see the top of the file); the node's edge slots
// come from the fused node table, in the same 2e+side order as the CSR list
template <int NS, int DM>
__global__ void __launch_bounds__(256) k_compute_w_vf(DevMesh m, NodeTab tab,
                                                      const int2* ekr, const double* vflux,
                                                      double* w_) {
    const int lane = threadIdx.x & 63;
    // the node index is wave-uniform: scalar registers, so the table loads are scalar
    const int n0 = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const bool valid = n0 < m.N;
    const int n = valid ? n0 : m.N - 1;
    const int L = m.L;
    const int cnt = ldc(tab.hdr, n).z & 0xff;
    int code[DM];
    int2 kr[DM];
#pragma unroll
    for (int q = 0; q < DM; ++q) {
        code[q] = ldc(tab.edge, (size_t)n * DM + q).x;
        kr[q] = ldc(ekr, code[q] >> 1);
    }
    double div[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int k = lane + 64 * s;
        const int kc = k < L ? k : L - 1;
        double vf[DM];
#pragma unroll
        for (int q = 0; q < DM; ++q) vf[q] = G(vflux)[(size_t)(code[q] >> 1) * L + kc];
        double d = 0.0;
#pragma unroll
        for (int q = 0; q < DM; ++q) {
            const bool use = q < cnt && k >= kr[q].x && k < kr[q].y;
            d = d + (use ? ((code[q] & 1) ? vf[q] : -vf[q]) : 0.0);
        }
        div[s] = d;
    }
    finish_w<NS>(m, n, valid, lane, div, w_);
}

template <int NS>
__global__ void __launch_bounds__(256) k_compute_w(DevMesh m, const double* uv_,
                                                   const double* helem_, double* w_) {
    const int lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const bool valid = n0 < m.N;
    const int n = valid ? n0 : m.N - 1;
    const int L = m.L;
    const auto uv = glb(uv_);
    const auto helem = glb(helem_);
    const auto off = glb(m.ecsr_off), lst = glb(m.ecsr);
    const auto etri = glb(reinterpret_cast<const int*>(m.edge_tri));
    const auto elev = glb(reinterpret_cast<const int*>(m.elev));
    const auto cross = glb(reinterpret_cast<const double*>(m.cross));
    const int s0 = off[n], s1 = off[n + 1];

    // stage 1: div[k] = sum over the node's (edge, side) of +-c[e][k]
    double div[NS];
    for (int s = 0; s < NS; ++s) div[s] = 0.0;
    for (int i = s0; i < s1; ++i) {
        const int code = lst[i];
        const int e = code >> 1;
        const int el1 = etri[2 * e], el2 = etri[2 * e + 1];
        const double dx1 = cross[4 * (size_t)e], dy1 = cross[4 * (size_t)e + 1];
        const double dx2 = cross[4 * (size_t)e + 2], dy2 = cross[4 * (size_t)e + 3];
        const int a1 = el1 >= 0 ? el1 : 0, a2 = el2 >= 0 ? el2 : 0;
        const int lo1 = elev[2 * a1], hi1 = elev[2 * a1 + 1];
        const int lo2 = elev[2 * a2], hi2 = elev[2 * a2 + 1];
        for (int s = 0; s < NS; ++s) {
            const int k = lane + 64 * s;
            if (k >= L) continue;
            const size_t i1 = (size_t)a1 * L + k, i2 = (size_t)a2 * L + k;
            const bool m1 = el1 >= 0 && k >= lo1 && k < hi1;
            const bool m2 = el2 >= 0 && k >= lo2 && k < hi2;
            // loads are unconditional (the indices are in bounds) and masked afterwards,
            // so all of them are in flight at once
            const double u1 = uv[2 * i1], v1 = uv[2 * i1 + 1], h1 = helem[i1];
            const double u2 = uv[2 * i2], v2 = uv[2 * i2 + 1], h2 = helem[i2];
            const double t1 = m1 ? (v1 * dx1 - u1 * dy1) * h1 : 0.0;
            const double t2 = m2 ? (v2 * dx2 - u2 * dy2) * h2 : 0.0;
            const double c = t1 + -t2;              // sign * where(mask, term, 0), summed
            div[s] = div[s] + ((code & 1) ? -c : c);
        }
    }

    finish_w<NS>(m, n, valid, lane, div, w_);
}

}  // namespace

int launch_compute_w(const DevMesh& m, const double* uv, const double* helem, double* w,
                     hipStream_t s) {
    if (m.N == 0) return FCT_OK;
    const int wpb = FCT_W_WPB;
    const dim3 grid((m.N + wpb - 1) / wpb), block(64 * wpb);
    if (m.L <= 64)
        k_compute_w<1><<<grid, block, 0, s>>>(m, uv, helem, w);
    else if (m.L <= 128)
        k_compute_w<2><<<grid, block, 0, s>>>(m, uv, helem, w);
    else
        return set_error(FCT_E_UNSUPPORTED, "compute_w supports nl <= 128 (got %d)", m.L);
    return check_launch("k_compute_w");
}

int launch_compute_w_vf(const DevMesh& m, const NodeTab& tab, const int2* ekr,
                        const double* vflux, double* w, hipStream_t s) {
    if (m.N == 0) return FCT_OK;
    const int wpb = FCT_W_WPB;
    const dim3 grid((m.N + wpb - 1) / wpb), block(64 * wpb);
    if (tab.dm == 6 && m.L <= 64) k_compute_w_vf<1, 6><<<grid, block, 0, s>>>(m, tab, ekr, vflux, w);
    else if (tab.dm == 6) k_compute_w_vf<2, 6><<<grid, block, 0, s>>>(m, tab, ekr, vflux, w);
    else if (m.L <= 64) k_compute_w_vf<1, 8><<<grid, block, 0, s>>>(m, tab, ekr, vflux, w);
    else k_compute_w_vf<2, 8><<<grid, block, 0, s>>>(m, tab, ekr, vflux, w);
    return check_launch("k_compute_w_vf");
}

int launch_compute_w_tab(const DevMesh& m, const NodeTab& tab, int remap, const double* uv,
                         const double* helem, double* w, hipStream_t s) {
    if (m.N == 0) return FCT_OK;
    if (m.L > 128) return set_error(FCT_E_UNSUPPORTED, "compute_w supports nl <= 128 (got %d)", m.L);
    // Columns per workgroup. Fewer leave the column sums exposed, more leave fewer workgroups:
    // icosa-8 x 70 took 590, 504, 478, 526 and 698 us with 4, 8, 16, 32 and 64; icosa-6 x 70
    // (29 thousand nodes) 40, 37 and 42 with 4, 8 and 16; icosa-7 x 70 on an 8-slot table,
    // whose term rows take more of the LDS, 154, 148 and 171.
    const int C = tab.dm == 6 && m.N >= 65536 ? 16 : 8;
    const dim3 grid((m.N + C - 1) / C), block(256);
    const size_t lds = ((size_t)C * (m.L | 1) + 4 * 64 * tab.dm) * sizeof(double);
    if (tab.dm == 6 && m.L <= 64) k_compute_w_tab<1, 6><<<grid, block, lds, s>>>(m, tab, C, remap, uv, helem, w);
    else if (tab.dm == 6) k_compute_w_tab<2, 6><<<grid, block, lds, s>>>(m, tab, C, remap, uv, helem, w);
    else if (m.L <= 64) k_compute_w_tab<1, 8><<<grid, block, lds, s>>>(m, tab, C, remap, uv, helem, w);
    else k_compute_w_tab<2, 8><<<grid, block, lds, s>>>(m, tab, C, remap, uv, helem, w);
    return check_launch("k_compute_w_tab");
}

}  // namespace fct
