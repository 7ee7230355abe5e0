// Tridiagonal systems of node columns in LDS: what the kernels of fct_column.hip and
// fct_vdiff.hip share (fct_column.hip describes the mapping). LDS rows are P = odd >= nl + 1
// doubles, so that lanes on different columns at one level fall into different banks.
#pragma once

#include <algorithm>

#include "fct_common.h"

namespace fct {

constexpr int VI_MAXC = 16;                   // columns per workgroup at most
constexpr size_t VI_LDS = 40 * 1024 - 512;    // four workgroups in a CU's 160 KB

inline int vi_pitch(int L) { return (L + 1) | 1; }
inline int vi_columns(int L, int arrays) {
    const size_t col = (size_t)arrays * vi_pitch(L) * sizeof(double);
    return (int)std::min<size_t>(VI_MAXC, VI_LDS / col);
}

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

}  // namespace fct
