// Device helpers of the wavefront-per-column kernels (lane l of slot s holds level
// k = 64*s + l): lane shifts, the block -> tile map, and typed loads.
#pragma once

#include "fct_common.h"

namespace fct {

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

// value of lane l-1 (wave_shr:1) of a 64-bit register, lane 0 keeping `first`, and of
// lane l+1 (wave_shl:1), lane 63 keeping `last` (the DPP move leaves a lane whose source
// is out of range at its old value). Called with all 64 lanes active: a lane whose
// source lane is switched off would keep the old value too. The edge value goes in as
// the old value rather than through a select on the lane index, so the compiler has no
// select to turn into a branch around the move (which would switch off the lanes it
// reads from); the empty asm keeps the move where it is written.
__device__ __forceinline__ double wave_prev(double v, double first) {
    int2 x = __builtin_bit_cast(int2, v);
    const int2 o = __builtin_bit_cast(int2, first);
    x.x = __builtin_amdgcn_update_dpp(o.x, x.x, 0x138, 0xf, 0xf, false);
    x.y = __builtin_amdgcn_update_dpp(o.y, x.y, 0x138, 0xf, 0xf, false);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return __builtin_bit_cast(double, x);
}
__device__ __forceinline__ double wave_next(double v, double last) {
    int2 x = __builtin_bit_cast(int2, v);
    const int2 o = __builtin_bit_cast(int2, last);
    x.x = __builtin_amdgcn_update_dpp(o.x, x.x, 0x130, 0xf, 0xf, false);
    x.y = __builtin_amdgcn_update_dpp(o.y, x.y, 0x130, 0xf, 0xf, false);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return __builtin_bit_cast(double, x);
}
__device__ __forceinline__ double lane_value(double v, int l) {
    int2 x = __builtin_bit_cast(int2, v);
    x.x = __builtin_amdgcn_readlane(x.x, l);
    x.y = __builtin_amdgcn_readlane(x.y, l);
    return __builtin_bit_cast(double, x);
}

// Two columns of up to 32 levels share a wavefront (HALF): lane = 32 * column + level.
template <bool HALF>
__device__ __forceinline__ int col_lane() { return HALF ? lane_id() & 31 : lane_id(); }

// wave_prev of the two half-wavefront columns, `first` at each one's level 0: row_bcast:15
// puts lanes 15 and 47 into rows 1 and 3, row_shr:1 then moves within the rows and leaves
// lanes 16 and 48 at that, lanes 0 and 32 at `first`. (wave_next serves both halves: it
// hands lane 31 the other column's level 0, and no caller uses that lane's.)
__device__ __forceinline__ double half_prev(double v, double first) {
    int2 x = __builtin_bit_cast(int2, v), o = __builtin_bit_cast(int2, first);
    o.x = __builtin_amdgcn_update_dpp(o.x, x.x, 0x142, 0xa, 0xf, false);
    o.y = __builtin_amdgcn_update_dpp(o.y, x.y, 0x142, 0xa, 0xf, false);
    x.x = __builtin_amdgcn_update_dpp(o.x, x.x, 0x111, 0xf, 0xf, false);
    x.y = __builtin_amdgcn_update_dpp(o.y, x.y, 0x111, 0xf, 0xf, false);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return __builtin_bit_cast(double, x);
}

// value at level k-1 of a column held as NS slots; `at0` is used at k = 0
template <int NS, bool HALF = false>
__device__ __forceinline__ void col_prev(const double (&v)[NS], double (&o)[NS], double at0) {
    if constexpr (HALF) {
        static_assert(NS == 1);
        o[0] = half_prev(v[0], at0);
        return;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
        o[s] = wave_prev(v[s], (s > 0) ? lane_value(v[s > 0 ? s - 1 : 0], 63) : at0);
}
// ... the column's own level 0 at k = 0
template <int NS, bool HALF = false>
__device__ __forceinline__ void col_prev_own(const double (&v)[NS], double (&o)[NS]) {
    col_prev<NS, HALF>(v, o, HALF ? v[0] : lane_value(v[0], 0));
}

// value at level k+1; `atend` is used past the last slot lane
template <int NS>
__device__ __forceinline__ void col_next(const double (&v)[NS], double (&o)[NS], double atend) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
        o[s] = wave_next(v[s], (s + 1 < NS) ? lane_value(v[s + 1 < NS ? s + 1 : s], 0) : atend);
}

template <int NS>
__device__ __forceinline__ double col_bcast0(const double (&v)[NS]) { return lane_value(v[0], 0); }

__device__ __forceinline__ double ab2(double told, double t) { return AB_OLD * told + AB_NEW * t; }

__device__ __forceinline__ bool in_bytes(int packed, int shift, int k) {
    const int lo = (packed >> shift) & 0xff, hi = (packed >> (shift + 8)) & 0xff;
    return k >= lo && k < hi;
}

// Block -> tile remap. Workgroups are dealt to the X XCDs round-robin (block b to XCD
// b % X), and node and edge order is spatially local, so giving each XCD runs of C
// consecutive tiles keeps most neighbours of a tile in the same L2. remap = X | C << 8;
// C = 0 gives each XCD one contiguous range of the whole grid. With C > 0 the grid's
// tail beyond the last whole round of X * C blocks keeps hardware order, so the map
// is a bijection on [0, gridDim.x) for any grid size.
__device__ __forceinline__ unsigned block_tile(int remap) {
    const unsigned b = blockIdx.x, G = gridDim.x;
    const unsigned X = (unsigned)remap & 0xffu, C = (unsigned)remap >> 8;
    if (X <= 1) return b;
    const unsigned x = b % X, i = b / X;
    if (C == 0) {
        const unsigned q = G / X, r = G % X;
        return x * q + (x < r ? x : r) + i;
    }
    const unsigned span = X * C;
    if (b >= G - G % span) return b;
    return ((i / C) * X + x) * C + i % C;
}

// Wavefront -> task index: the wavefronts of the (remapped) grid, numbered.
__device__ __forceinline__ bool single_wave(int64_t total, int remap, int& w) {
    const int64_t ww = ((int64_t)block_tile(remap) * blockDim.x + threadIdx.x) >> 6;
    if (ww >= total) return false;
    w = __builtin_amdgcn_readfirstlane((int)ww);
    return true;
}

// Memory is accessed through global-address-space pointers (G). Pointers that a
// batched kernel reads from its descriptor array are generic to the compiler, which
// would otherwise emit flat loads for them.
template <class T>
using gptr = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gptr<T> G(T* p) { return (gptr<T>)p; }

// HIP's vector types are classes; load and store them as clang vectors of the same size.
typedef int fct_iv2 __attribute__((ext_vector_type(2)));
typedef int fct_iv4 __attribute__((ext_vector_type(4)));
typedef double fct_dv2 __attribute__((ext_vector_type(2)));
typedef double fct_dv4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int2 ldv(const int2* p, size_t i) {
    return __builtin_bit_cast(int2, ((gptr<const fct_iv2>)p)[i]);
}
__device__ __forceinline__ int4 ldv(const int4* p, size_t i) {
    return __builtin_bit_cast(int4, ((gptr<const fct_iv4>)p)[i]);
}
__device__ __forceinline__ double2 ldv(const double2* p, size_t i) {
    return __builtin_bit_cast(double2, ((gptr<const fct_dv2>)p)[i]);
}
__device__ __forceinline__ double4 ldv(const double4* p, size_t i) {
    return __builtin_bit_cast(double4, ((gptr<const fct_dv4>)p)[i]);
}
// Loads at wave-uniform addresses of data that the same launch does not write (mesh tables;
// the adjoint's edge signs, from an earlier launch on the stream: the scalar cache is
// invalidated where a kernel starts), through the constant address space so that the compiler
// issues scalar loads: they go through the scalar cache and leave the vector memory pipeline
// to the column gathers.
template <class T>
using cptr = __attribute__((address_space(4))) const T*;
__device__ __forceinline__ int ldc(const int* p, size_t i) { return ((cptr<int>)p)[i]; }
__device__ __forceinline__ double ldc(const double* p, size_t i) { return ((cptr<double>)p)[i]; }
__device__ __forceinline__ int2 ldc(const int2* p, size_t i) {
    return __builtin_bit_cast(int2, ((cptr<fct_iv2>)p)[i]);
}
__device__ __forceinline__ int4 ldc(const int4* p, size_t i) {
    return __builtin_bit_cast(int4, ((cptr<fct_iv4>)p)[i]);
}
__device__ __forceinline__ double2 ldc(const double2* p, size_t i) {
    return __builtin_bit_cast(double2, ((cptr<fct_dv2>)p)[i]);
}
__device__ __forceinline__ double4 ldc(const double4* p, size_t i) {
    return __builtin_bit_cast(double4, ((cptr<fct_dv4>)p)[i]);
}
__device__ __forceinline__ void stv(double2* p, size_t i, double2 v) {
    ((gptr<fct_dv2>)p)[i] = __builtin_bit_cast(fct_dv2, v);
}

// workgroups of `wpb` wavefronts for `waves` tasks
inline unsigned blocks_for(int64_t waves, int wpb) { return (unsigned)((waves + wpb - 1) / wpb); }

}  // namespace fct
