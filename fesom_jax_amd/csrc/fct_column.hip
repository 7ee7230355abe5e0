// Column solves of the implicit vertical advection (adv_tra_vert_impl,
// fesom_jax/tracer_adv.py:487-529, with ops.tdma, ops.py:121-168) and their reverse mode.
//
// Mapping: a workgroup of four wavefronts takes C consecutive node columns, which are one
// contiguous run of values in every field: the rows of the tridiagonal systems are formed
// with one thread per value (whole lines read, the loads of two values per thread in
// flight) and left in LDS. The Thomas recurrence, serial in the level, then runs one
// column (and tracer) per lane out of LDS, and the results go back one thread per value.
// C keeps four workgroups on a CU, so that some load or store while another is in its
// recurrence: of icosa-7 x 70 with two tracers (195 us) the recurrence is 60 us beyond the
// loads and stores. One thread per column straight from memory, the form this replaces,
// fetched a line for every value: 1331 us per tracer.
//
// LDS rows are P = odd >= nl + 1 doubles, so that lanes of one instruction on different
// columns at one level fall into different banks.

#include <algorithm>

#include "fct_common.h"

namespace fct {

namespace {

constexpr int VI_MAXC = 16;                   // columns per workgroup at most
constexpr size_t VI_LDS = 40 * 1024 - 512;    // four workgroups in a CU's 160 KB

inline int vi_pitch(int L) { return (L + 1) | 1; }
inline int vi_columns(int L, int arrays) {
    const size_t col = (size_t)arrays * vi_pitch(L) * sizeof(double);
    return (int)std::min<size_t>(VI_MAXC, VI_LDS / col);
}

template <int K>
struct VimplIO {
    const double* X[K];
    double* out[K];        // may be X itself: a workgroup reads and writes its own columns
};

// The Thomas recurrence on rows [lo, hi) of one column: sub-, main and superdiagonal A, B,
// Q and right-hand side D; Q becomes cp and D the solution. Rows are read four (back
// substitution: eight) at a time, ahead of the recurrence, past the column's end too: those
// values go nowhere, and the LDS array has VI_SLACK doubles behind its last column.
constexpr int VI_SLACK = 16;
__device__ __forceinline__ void thomas_column(const double* A, const double* B, double* Q,
                                              double* D, int lo, int hi) {
    double cp = 0.0, dp = 0.0, a[4], b[4], q[4], d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { a[i] = A[lo + i]; b[i] = B[lo + i]; q[i] = Q[lo + i]; d[i] = D[lo + i]; }
    for (int k = lo; k < hi; k += 4) {
        double na[4], nb[4], nq[4], nd[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            na[i] = A[k + 4 + i]; nb[i] = B[k + 4 + i]; nq[i] = Q[k + 4 + i]; nd[i] = D[k + 4 + i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double mm = b[i] - a[i] * cp;
            cp = q[i] / mm;
            dp = (d[i] - a[i] * dp) / mm;
            if (k + i < hi) { Q[k + i] = cp; D[k + i] = dp; }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) { a[i] = na[i]; b[i] = nb[i]; q[i] = nq[i]; d[i] = nd[i]; }
    }
    if (lo >= hi) return;
    int g = lo + (hi - lo - 1) / 8 * 8;
    double x = 0.0, c8[8], d8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) { c8[i] = Q[g + i]; d8[i] = D[g + i]; }
    for (; g >= lo; g -= 8) {
        double nc[8], nd[8];
        const int p = g > lo ? g - 8 : g;
#pragma unroll
        for (int i = 0; i < 8; ++i) { nc[i] = Q[p + i]; nd[i] = D[p + i]; }
#pragma unroll
        for (int i = 7; i >= 0; --i) {
            if (g + i < hi) {
                x = d8[i] - c8[i] * x;
                D[g + i] = x;
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) { c8[i] = nc[i]; d8[i] = nd[i]; }
    }
}

// A workgroup's C columns are one contiguous run of C * nl values; element i of it is level
// i % nl of column i / nl (the float quotient is exact for i < 2^16: the nearest multiple
// of 1 / nl is at least 0.5 / nl away).
struct ColLevel {
    int c, k;
    int2 nr;
    bool in;       // one of the workgroup's elements, on a wet layer
};
__device__ __forceinline__ ColLevel col_level(const DevMesh& m, int n0, int count, float inv, int i) {
    ColLevel e;
    e.in = i < count;
    const int j = e.in ? i : 0;
    e.c = (int)(((float)j + 0.5f) * inv);
    e.k = j - e.c * m.L;
    e.nr = m.nlev[n0 + e.c];
    e.in = e.in && in_layer(e.nr, e.k);
    return e;
}

// MASK: X holds values on wet layers only (the fused path's LO); dry neighbours count as
// the 0 that a dense LO has there, and only wet layers are written.
template <int K, bool MASK>
__global__ void __launch_bounds__(256)
k_vimpl(DevMesh m, int C, const double* __restrict__ w_i, const double* __restrict__ hnn, double dt,
        VimplIO<K> io) {
    extern __shared__ double sh[];
    constexpr int U = 2;      // elements per thread whose loads are in flight together
    const int L = m.L, P = (L + 1) | 1, S = C * P;
    const int n0 = blockIdx.x * C;
    const int nc = min(C, m.N - n0), count = nc * L;
    const float inv = 1.0f / (float)L;
    const size_t g0 = (size_t)n0 * L;
    for (int i0 = threadIdx.x; i0 < count; i0 += 256 * U) {
        ColLevel e[U];
        VimplRow r[U];
        double Tc[U][K], Td[U][K], Tu[U][K];
#pragma unroll
        for (int u = 0; u < U; ++u) e[u] = col_level(m, n0, count, inv, i0 + 256 * u);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!e[u].in) continue;
            const size_t i = g0 + i0 + 256 * u;
            const int k = e[u].k;
            r[u] = vimpl_row(m, w_i, hnn, dt, i - k, k, e[u].nr);
#pragma unroll
            for (int j = 0; j < K; ++j) {
                Tc[u][j] = io.X[j][i];
                Td[u][j] = k > 0 ? io.X[j][i - 1] : Tc[u][j];
                Tu[u][j] = k + 1 < L ? io.X[j][i + 1] : 0.0;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!e[u].in) continue;
            const int k = e[u].k;
            double* s = sh + e[u].c * P + k;
            s[0] = r[u].a;
            s[S] = r[u].b;
            s[2 * S] = r[u].c;
#pragma unroll
            for (int j = 0; j < K; ++j) {
                double td = Td[u][j], tu = Tu[u][j];
                if (MASK) {
                    td = (k == 0 || k > e[u].nr.x) ? td : 0.0;
                    tu = k + 1 < e[u].nr.y ? tu : 0.0;
                }
                s[(3 + j) * S] = -(r[u].a * td + r[u].b_adv * Tc[u][j] + r[u].c * tu);
            }
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < nc * K) {
        const int c = (int)threadIdx.x / K, j = (int)threadIdx.x - c * K;
        const int2 nr = m.nlev[n0 + c];
        double* A = sh + c * P;
        // the K lanes of a column write the same cp
        thomas_column(A, A + S, A + 2 * S, A + (3 + j) * S, nr.x, nr.y);
    }
    __syncthreads();
    for (int i0 = threadIdx.x; i0 < count; i0 += 256 * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + 256 * u >= count) break;
            const ColLevel e = col_level(m, n0, count, inv, i0 + 256 * u);
            if (MASK && !e.in) continue;
            const size_t i = g0 + i0 + 256 * u;
#pragma unroll
            for (int j = 0; j < K; ++j)
                io.out[j][i] = io.X[j][i] + (e.in ? sh[(3 + j) * S + e.c * P + e.k] : 0.0);
        }
    }
}

template <int K, bool MASK>
int vimpl_call(const DevMesh& m, const double* w_i, const double* hnn, double dt,
               const VimplIO<K>& io, hipStream_t s) {
    const int C = vi_columns(m.L, 3 + K);
    const size_t lds = ((size_t)(3 + K) * C * vi_pitch(m.L) + VI_SLACK) * sizeof(double);
    k_vimpl<K, MASK><<<dim3((m.N + C - 1) / C), dim3(256), lds, s>>>(m, C, w_i, hnn, dt, io);
    return check_launch("k_vimpl");
}

}  // namespace

bool vimpl_fits(int L) { return vi_columns(L, 5) >= 1; }

int launch_vimpl(const DevMesh& m, const double* w_i, const double* hnn, double dt,
                 const double* X, double* out, hipStream_t s) {
    VimplIO<1> io{{X}, {out}};
    return vimpl_call<1, false>(m, w_i, hnn, dt, io, s);
}

int launch_vimpl_wet(const DevMesh& m, const double* w_i, const double* hnn, double dt, double* X,
                     int K, hipStream_t s) {
    const size_t NL = (size_t)m.N * m.L;
    for (int j = 0; j < K; j += 2) {
        int rc;
        if (K - j >= 2) {
            VimplIO<2> io{{X + j * NL, X + (j + 1) * NL}, {X + j * NL, X + (j + 1) * NL}};
            rc = vimpl_call<2, true>(m, w_i, hnn, dt, io, s);
        } else {
            VimplIO<1> io{{X + j * NL}, {X + j * NL}};
            rc = vimpl_call<1, true>(m, w_i, hnn, dt, io, s);
        }
        if (rc) return rc;
    }
    return FCT_OK;
}

}  // namespace fct
