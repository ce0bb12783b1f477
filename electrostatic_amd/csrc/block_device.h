// block_device.h -- device pieces shared by the dense-block kernels: FP64
// MFMA, lane moves, and the pivoted inverse of one 32 x 32 complex matrix by
// one wavefront.
#pragma once

#include <hip/hip_runtime.h>

#include "negf_internal.h"

namespace negf {

typedef __attribute__((ext_vector_type(4))) double d4;

constexpr int BM = 32;               // orbitals per block
constexpr int BLD = 33;              // LDS row stride (doubles)
constexpr int BPL = BM * BLD;        // doubles per LDS plane
constexpr int BGL = BM * BM;         // doubles per plane in global memory (row-major, unpadded)

__device__ __forceinline__ d4 mfma64(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ double mag2(double re, double im) { return re * re + im * im; }

// max that keeps a NaN (so that a NaN never reads as converged)
__device__ __forceinline__ double nan_max(double a, double b) { return (a > b || a != a) ? a : b; }

// 64-bit value of another lane by a DPP move (CTRL: a compile-time DPP
// control word; all lanes active).
template <int CTRL>
__device__ __forceinline__ unsigned long long dpp64(unsigned long long v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v & 0xffffffffull), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, 0xF, 0xF, false);
    return ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
}

// LDS written by lanes of this wavefront is visible to its later reads.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 32-bit pivot key: |a|^2 rounded to float (non-negative, so its bits order
// as an unsigned integer) with the low 5 mantissa bits replaced by 31 - row:
// the largest key is a largest magnitude (to float precision, enough for a
// pivot choice) and, among equal ones, the smallest row.  0: no candidate.
__device__ __forceinline__ unsigned pivot_key32(double m, int i)
{
    return (__float_as_uint((float)m) & ~31u) | (unsigned)(31 - i);
}

template <int CTRL>
__device__ __forceinline__ unsigned max_dpp(unsigned v)
{
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
    return o > v ? o : v;
}

// max over the 64 lanes, read from lane 63: quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror and row_mirror give every lane its row's
// maximum; row_bcast:15 and row_bcast:31 carry the rows into lane 63.
__device__ __forceinline__ unsigned wave_max32(unsigned v)
{
    v = max_dpp<0xB1>(v);
    v = max_dpp<0x4E>(v);
    v = max_dpp<0x141>(v);
    v = max_dpp<0x140>(v);
    v = max_dpp<0x142>(v);
    v = max_dpp<0x143>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ double dpp_swap1(double x)
{
    return __longlong_as_double((long long)dpp64<0xB1>((unsigned long long)__double_as_longlong(x)));
}

__device__ __forceinline__ double readlane_f64(double x, int src)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)(b & 0xffffffffll), src);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)((unsigned long long)b >> 32), src);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// 1 / d for d > 0: hardware reciprocal estimate refined by two Newton-Raphson
// steps y <- y + y (1 - d y), each of which squares the relative error.
__device__ __forceinline__ double recip_nr(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = fma(y, fma(-d, y, 1.0), y);
    return fma(y, fma(-d, y, 1.0), y);
}

// Inverse of the complex matrix (Mre, Mim) (LDS planes, row stride BLD) by
// one wavefront, in place: Gauss-Jordan with partial pivoting.  Lane l holds
// row i = l / 2, columns h * 16 .. h * 16 + 15 (h = l % 2) in registers.
// Rows are never swapped: step k takes as pivot the largest |a_ik| among the
// rows not yet used (|a_ik|^2 compared in float precision, ties to the
// smallest row), found by a 64-lane maximum.
// A pivot row is not divided by its pivot: each row keeps a scale s_i (1 until
// it is the pivot, then 1 / pivot) and holds M / s_i, which leaves every
// update in the form a_ij -= (a_ik / pivot) a_pj with the stored values; the
// scales are applied once at the end.  The pivot element and the pivot row's
// entries in column k + 1 are read from their lanes (v_readlane), so the next
// pivot search waits on no memory; every lane fetches the pivot row's other
// entries of its columns from the pivot row's lane of the same half by lane
// shuffles (ds_bpermute), so no LDS store, wait and reload sits in a step.
// perm (32 ints of LDS) records the pivot order.  The result is written back
// through the pivot order: A^-1[q(i)][perm[j]] = s_i M[i][j], with q(i) the
// step whose pivot was row i.
__device__ __forceinline__ void gj_inverse_wave(double* Mre, double* Mim, int* perm, int lane)
{
    const int i = lane >> 1, h = lane & 1;
    double ar[16], ai[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        ar[r] = Mre[i * BLD + h * 16 + r];
        ai[r] = Mim[i * BLD + h * 16 + r];
    }
    unsigned used = 0u;  // bit x: row x has been a pivot (wave-uniform)
    int qrow = 0;
    double sr = 1.0, si = 0.0;
    for (int kh = 0; kh < 2; ++kh) {
#pragma unroll
        for (int kr = 0; kr < 16; ++kr) {
            const int k = kh * 16 + kr;
            // pivot: column k is register kr of the lanes with h == kh
            unsigned key = 0u;
            if (h == kh && !((used >> i) & 1u)) key = pivot_key32(mag2(ar[kr], ai[kr]), i);
            key = wave_max32(key);
            const int p = key == 0u ? __builtin_ctz(~used) : 31 - (int)(key & 31u);
            used |= 1u << p;
            if (i == p) {
                if (h == 0) perm[k] = p;
                qrow = k;
            }
            // 1 / pivot from the lane holding (p, k)
            const double pr = readlane_f64(ar[kr], 2 * p + kh), pim = readlane_f64(ai[kr], 2 * p + kh);
            const double iv = recip_nr(pr * pr + pim * pim);
            const double ir = pr * iv, ii = -pim * iv;
            // multiplier of this row: a_ik / pivot (a_ik from the lane of this row holding column k)
            const double orr = dpp_swap1(ar[kr]), oi = dpp_swap1(ai[kr]);
            const double fr = (h == kh) ? ar[kr] : orr, fi = (h == kh) ? ai[kr] : oi;
            double mr = fr * ir - fi * ii, mi = fr * ii + fi * ir;
            if (i == p) {
                mr = 0.0;
                mi = 0.0;
                sr = ir;
                si = ii;
            }
            // register c (column k + 1 in the lanes of its half) first, with the
            // pivot row's entries read from its two lanes: the next pivot search
            // then waits on no shuffle
            const int c = (kr + 1) & 15;
            {
                const double x0r = readlane_f64(ar[c], 2 * p), x0i = readlane_f64(ai[c], 2 * p);
                const double x1r = readlane_f64(ar[c], 2 * p + 1), x1i = readlane_f64(ai[c], 2 * p + 1);
                const double xr = h ? x1r : x0r, xi = h ? x1i : x0i;
                ar[c] = fma(-mr, xr, fma(mi, xi, ar[c]));
                ai[c] = fma(-mr, xi, fma(-mi, xr, ai[c]));
            }
            // the other entries of the pivot row, from the lane of its same half
            // (the pivot row itself is not updated: m = 0)
            const int src = 2 * p + h;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (r == c) continue;
                const double2 x = make_double2(__shfl(ar[r], src, 64), __shfl(ai[r], src, 64));
                ar[r] = fma(-mr, x.x, fma(mi, x.y, ar[r]));
                ai[r] = fma(-mr, x.y, fma(-mi, x.x, ai[r]));
            }
            if (h == kh) {
                ar[kr] = (i == p) ? 1.0 : -mr;
                ai[kr] = (i == p) ? 0.0 : -mi;
            }
        }
    }
    wave_sync();
    int pj[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) pj[r] = perm[h * 16 + r];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int o = qrow * BLD + pj[r];
        Mre[o] = sr * ar[r] - si * ai[r];
        Mim[o] = sr * ai[r] + si * ar[r];
    }
    wave_sync();
}

}  // namespace negf
