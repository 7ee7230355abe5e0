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

#include "fct_column.h"

namespace fct {

namespace {

// cotangents of max(x, y) / min(x, y) for x
__device__ __forceinline__ double vmax_x(double g, double x, double y) {
    return x > y ? g : (x == y ? 0.5 * g : 0.0);
}
__device__ __forceinline__ double vmin_x(double g, double x, double y) {
    return x < y ? g : (x == y ? 0.5 * g : 0.0);
}

template <int K>
struct VimplIO {
    const double* X[K];
    double* out[K];        // may be X itself: a workgroup reads and writes its own columns
};

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

// Reverse mode of the solve (as jax.grad reverses the two scans of ops.tdma): on entry gX
// holds the cotangent of the solved values, on exit that of X, and the cotangent of w_i is
// added to gwi; X and gX hold values on wet layers only. The recurrences of the forward
// solve and of its reverse run one column per lane out of LDS, eight arrays per column;
// everything else one thread per value (VR_U values per thread at most: a workgroup's LDS
// holds 2.4 per thread). With gwi1 the launch takes two tracers (grid.y): the second one's X
// at N * L, gX at gX_stride, its w_i cotangent added to gwi1. One thread per column from memory took 883 us per tracer at
// icosa-6 x 70.
constexpr int VR_U = 3, VR_ARRAYS = 8;
static_assert(VI_LDS <= (size_t)VR_U * 256 * VR_ARRAYS * sizeof(double), "values per thread");

__global__ void __launch_bounds__(256)
k_vimpl_reverse(DevMesh m, int C, const double* __restrict__ w_i, const double* __restrict__ hnn,
                double dt, const double* __restrict__ X, double* __restrict__ gX,
                double* __restrict__ gwi, double* __restrict__ gwi1, size_t gX_stride) {
    extern __shared__ double sh[];
    if (blockIdx.y) {      // the second tracer of the launch
        X += (size_t)m.N * m.L; gX += gX_stride; gwi = gwi1;
    }
    const int L = m.L, P = (L + 1) | 1, S = C * P;
    const int n0 = blockIdx.x * C;
    const int nc = min(C, m.N - n0), count = nc * L;
    const float inv = 1.0f / (float)L;
    const size_t g0 = (size_t)n0 * L;
    ColLevel e[VR_U];
    VimplRow r[VR_U];
    double Td[VR_U], Tc[VR_U], Tu[VR_U], gin[VR_U];
#pragma unroll
    for (int u = 0; u < VR_U; ++u) {
        const int idx = threadIdx.x + 256 * u;
        e[u] = col_level(m, n0, count, inv, idx);
        if (!e[u].in) continue;
        const size_t i = g0 + idx;
        const int k = e[u].k;
        r[u] = vimpl_row(m, w_i, hnn, dt, i - k, k, e[u].nr);
        Tc[u] = X[i];
        Td[u] = k == 0 ? Tc[u] : (k > e[u].nr.x ? X[i - 1] : 0.0);
        Tu[u] = k + 1 < e[u].nr.y ? X[i + 1] : 0.0;
        gin[u] = gX[i];
    }
#pragma unroll
    for (int u = 0; u < VR_U; ++u) {
        if (!e[u].in) continue;
        double* q = sh + e[u].c * P + e[u].k;
        q[0] = r[u].a;
        q[S] = r[u].b;
        q[2 * S] = r[u].c;
        q[3 * S] = -(r[u].a * Td[u] + r[u].b_adv * Tc[u] + r[u].c * Tu[u]);
        q[7 * S] = gin[u];
    }
    __syncthreads();
    if ((int)threadIdx.x < nc) {
        const int2 nr = m.nlev[n0 + threadIdx.x];
        double* A = sh + threadIdx.x * P;
        double *B = A + S, *Q = A + 2 * S, *D = A + 3 * S, *CP = A + 4 * S, *DP = A + 5 * S;
        double *Xs = A + 6 * S, *Gs = A + 7 * S;
        double cp = 0.0, dp = 0.0;
#pragma unroll 4
        for (int k = nr.x; k < nr.y; ++k) {
            const double a = A[k], mm = B[k] - a * cp;
            cp = Q[k] / mm;
            dp = (D[k] - a * dp) / mm;
            B[k] = mm; CP[k] = cp; DP[k] = dp;
        }
        double x = 0.0;
        Xs[nr.y] = 0.0;
#pragma unroll 4
        for (int k = nr.y - 1; k >= nr.x; --k) {
            x = DP[k] - CP[k] * x;
            Xs[k] = x;
        }
        double carry = 0.0;
#pragma unroll 4
        for (int k = nr.x; k < nr.y; ++k) {
            const double g = Gs[k] + carry;
            Gs[k] = g;
            carry = -g * CP[k];
        }
        // down the forward sweep's rows: cotangents of the numerator (Gs), of the
        // denominator (B) and of the superdiagonal (Xs, one slot up: x[k+1] is spent)
        double gcc = 0.0, gdc = 0.0;
#pragma unroll 2
        for (int k = nr.y - 1; k >= nr.x; --k) {
            const double a = A[k], mm = B[k];
            const double num = D[k] - a * (k > nr.x ? DP[k - 1] : 0.0);
            const double GC = -Gs[k] * Xs[k + 1] + gcc, GD = Gs[k] + gdc;
            const double i2 = 1.0 / (mm * mm);
            const double gn = GD / mm;
            const double gm = (-GD * num) * i2 + (-GC * Q[k]) * i2;
            gdc = -gn * a;
            gcc = -gm * a;
            Gs[k] = gn;
            B[k] = gm;
            Xs[k + 1] = GC / mm;
        }
    }
    __syncthreads();
    double gwu[VR_U];
#pragma unroll
    for (int u = 0; u < VR_U; ++u) {
        if (!e[u].in) continue;
        const VimplRow& R = r[u];
        double* q = sh + e[u].c * P + e[u].k;
        const bool below = e[u].k > e[u].nr.x;
        const double gn = q[7 * S], gm = q[S], gs = -gn;
        const double g_a = (-gn * (below ? q[5 * S - 1] : 0.0) + -gm * (below ? q[4 * S - 1] : 0.0)) +
                           gs * Td[u];
        const double g_c = q[6 * S + 1] + gs * Tu[u];
        const double g_badv = gs * Tc[u] + gm;
        const double gaa = g_a * R.v_top, gca = g_c * R.v_bot;
        const double gt = g_badv * R.v_top, gb = g_badv * R.v_bot;
        gwu[u] = R.surf ? gt : vmin_x(gaa, R.wu, 0.0) + vmax_x(gt, R.wu, 0.0);
        q[3 * S] = R.bot ? 0.0 : -vmin_x(gb, R.wd, 0.0) - vmax_x(gca, R.wd, 0.0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < VR_U; ++u) {
        if (!e[u].in) continue;
        const size_t i = g0 + threadIdx.x + 256 * u;
        const double* q = sh + e[u].c * P + e[u].k;
        const bool above = e[u].k + 1 < e[u].nr.y, below = e[u].k > e[u].nr.x;
        double g = gin[u] - q[7 * S] * r[u].b_adv;
        if (e[u].k == 0) g -= q[7 * S] * r[u].a;
        if (above) g -= q[7 * S + 1] * q[1];
        if (below) g -= q[7 * S - 1] * q[2 * S - 1];
        gX[i] = g;
        gwi[i] += gwu[u] + (below ? q[3 * S - 1] : 0.0);
    }
}

}  // namespace

bool vimpl_fits(int L) { return vi_columns(L, 5) >= 1; }

int launch_vimpl(const DevMesh& m, const double* w_i, const double* hnn, double dt,
                 const double* X, double* out, hipStream_t s) {
    VimplIO<1> io{{X}, {out}};
    return vimpl_call<1, false>(m, w_i, hnn, dt, io, s);
}

int launch_vimpl_wet(const DevMesh& m, const double* w_i, const double* hnn, double dt,
                     const double* X, double* out, int K, hipStream_t s) {
    const size_t NL = (size_t)m.N * m.L;
    for (int j = 0; j < K; j += 2) {
        int rc;
        if (K - j >= 2) {
            VimplIO<2> io{{X + j * NL, X + (j + 1) * NL}, {out + j * NL, out + (j + 1) * NL}};
            rc = vimpl_call<2, true>(m, w_i, hnn, dt, io, s);
        } else {
            VimplIO<1> io{{X + j * NL}, {out + j * NL}};
            rc = vimpl_call<1, true>(m, w_i, hnn, dt, io, s);
        }
        if (rc) return rc;
    }
    return FCT_OK;
}

int launch_vimpl_reverse(const DevMesh& m, const double* w_i, const double* hnn, double dt,
                         const double* X, double* gX, double* gwi, double* gwi1, size_t gX_stride,
                         hipStream_t s) {
    const int C = vi_columns(m.L, VR_ARRAYS);
    const size_t lds = ((size_t)VR_ARRAYS * C * vi_pitch(m.L) + VI_SLACK) * sizeof(double);
    k_vimpl_reverse<<<dim3((m.N + C - 1) / C, gwi1 ? 2 : 1), dim3(256), lds, s>>>(
        m, C, w_i, hnn, dt, X, gX, gwi, gwi1, gX_stride);
    return check_launch("k_vimpl_reverse");
}

}  // namespace fct
