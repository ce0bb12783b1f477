// block_split.hip -- dense-block chain whose coupling joins only part of each
// block: Sancho-Rubio leads and the block recursive Green's function sweep on
// parts of at most 16 orbitals, FP64 MFMA for gfx950.
//
// A tube cut into blocks of two rings (and any chain whose T connects only
// the second part of a block with the first part of the next) is also a chain
// of twice as many blocks of half the size, with the couplings H_01 (inside a
// block) and T_10 (to the next) in turn.  An inverse and the products of a
// 16-orbital block cost an eighth of a 32-orbital block's, so the same diag
// G^R takes a quarter of the operations.  The mathematics per block is that of
// block_rgf.hip (Compute_RhoEq NEGF_Common.cpp:3667-3754 with blocks in place
// of scalars).
//
// Registers.  Lane l = 16 q + i of a wavefront holds the elements (i, q + 4 v),
// v = 0..3, of a 16 x 16 matrix: 16 registers for a complex one.  That is the
// A operand of v_mfma_f64_16x16x4f64 (A[l % 16][l / 16 + 4 v]) and, for the
// transposed matrix, its B operand; the result comes back with rows and
// columns exchanged, so
//   prod(A, B) = B A^T
// maps this layout to itself, and no operand of a product passes through LDS:
// with g symmetric and C the real coupling to the next part,
//   Q = prod(g, C^T) = C^T g,   S = prod(Q, C^T) = C^T g C.
//
// Inverse.  The matrices are complex symmetric, so they are inverted by the
// symmetric sweep on blocks of four rows and columns J: with P = A_JJ,
//   A_JJ <- -P^-1,  A_iJ <- A_iJ P^-1,  A_ij <- A_ij - A_iJ P^-1 A_jJ^T,
// which keeps A symmetric and ends at -A^-1.  The columns J are one register
// (lane (i, q) holds A[i][4 t + q]), four elimination steps on it give P^-1 and
// A_iJ P^-1, and the rank-4 update of everything else is one MFMA per real
// product whose operands are that register before and after: no row is
// gathered, and only the pivot column crosses the rows of 16 lanes
// (ds_bpermute; the pivot row goes along a DPP row by row_newbcast).
//
// Direct assembly.  G_b = (E - H_b - v_b - S_left - S_right)^-1 from the left and
// the right self-energy of each part, as the scalar sweep forms 1 / (alpha - X -
// Y); not G_b = g_b + X G_{b+1} X^T, whose two terms cancel where the unfinished
// chain has an edge state near E.  Against a dense inverse the diagonal is
// then off by 1e-14 .. 3e-11 where that backward recursion is off by
// 1e-14 .. 3e-8 ((7..16,0) tubes, E within 0.15 eV of the disordered edge
// states, Im E = 1e-5 eV).
//
// Parallelism.  Each energy has two wavefronts, one per lead.  Both sweep to the
// middle storing the self-energy on each of their parts (4 KiB), meet once, and
// go on into the other half, where each inverts two matrices per part at once
// (its own g and, with the other's stored self-energy, G).
//
// Bound by the FP64 VALU issue of the elimination steps (about 55 instructions
// per pivot; row broadcasts as 64-bit DPP moves and a third-order reciprocal step).
// One copy of the code serves blocks of both parities, 31 against 72 KB when it is
// written out twice, at the same time.  Measured, 500 blocks of 32 orbitals, 1024
// energies: sweep 8.6 ms against 20.5 ms for the 32-orbital sweep (one wavefront
// per energy, pivoted inverse of 1600 cycles per step) and 9.0 ms with 32-bit DPP
// moves and two Newton steps; leads 1.08 ms against 4.5 ms (four wavefronts and a
// barrier per pivot step); 40 blocks of 20 orbitals, 143 energies: 0.31 against
// 1.6 ms and 0.27 against 0.53 ms.
#include "block_split.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "block_device.h"

namespace negf {

// element (i, q + 4 v) in re[v], im[v] of lane 16 q + i
struct M16 {
    d4 re, im;
};

__device__ __forceinline__ M16 zero16() { return M16{d4{0, 0, 0, 0}, d4{0, 0, 0, 0}}; }

// c + B A^T over the first NS columns of both (columns beyond are zero);
// real operands have one plane
template <int NS>
__device__ __forceinline__ M16 prod_cr(const M16& a, const d4& b, M16 c)
{
#pragma unroll
    for (int v = 0; v < NS / 4; ++v) {
        c.re = mfma64(a.re[v], b[v], c.re);
        c.im = mfma64(a.im[v], b[v], c.im);
    }
    return c;
}
template <int NS>
__device__ __forceinline__ M16 prod_rc(const d4& a, const M16& b, M16 c)
{
#pragma unroll
    for (int v = 0; v < NS / 4; ++v) {
        c.re = mfma64(a[v], b.re[v], c.re);
        c.im = mfma64(a[v], b.im[v], c.im);
    }
    return c;
}
template <int NS>
__device__ __forceinline__ M16 prod_cc(const M16& a, const M16& b, M16 c)
{
#pragma unroll
    for (int v = 0; v < NS / 4; ++v) {
        c.re = mfma64(a.re[v], b.re[v], c.re);
        c.im = mfma64(a.re[v], b.im[v], c.im);
        c.re = mfma64(-a.im[v], b.im[v], c.re);
        c.im = mfma64(a.im[v], b.re[v], c.im);
    }
    return c;
}

__device__ __forceinline__ double bperm64(int addr, double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)b);
    const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// max over the 16 lanes of a DPP row
__device__ __forceinline__ unsigned row_max32(unsigned v)
{
    v = max_dpp<0xB1>(v);
    v = max_dpp<0x4E>(v);
    v = max_dpp<0x141>(v);
    return max_dpp<0x140>(v);
}

// One elimination step of inverse16s on column k = 16 RP + 4 KV + kq with the
// pivot in a row of part PP.
template <int NR, int RP, int KV, int PP>
__device__ __forceinline__ void gj_update(M16 (&a)[NR][NR], const double (&cr)[NR], const double (&ci)[NR], double ir,
                                          double ii, int pl, bool mine, double (&sr)[NR], double (&si)[NR], int lane)
{
    const bool prow = (lane & 15) == pl;
    const int src = ((lane & 48) + pl) * 4;
    double mr[NR], mi[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        mr[r] = fma(cr[r], ir, -ci[r] * ii);
        mi[r] = fma(cr[r], ii, ci[r] * ir);
        if (r == PP) {
            mr[r] = prow ? 0.0 : mr[r];
            mi[r] = prow ? 0.0 : mi[r];
            sr[r] = prow ? ir : sr[r];
            si[r] = prow ? ii : si[r];
        }
    }
#pragma unroll
    for (int c = 0; c < NR; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double xr = bperm64(src, a[PP][c].re[v]), xi = bperm64(src, a[PP][c].im[v]);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                a[r][c].re[v] -= fma(mr[r], xr, -mi[r] * xi);
                a[r][c].im[v] -= fma(mr[r], xi, mi[r] * xr);
            }
        }
    // the column itself
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const double vr = r == PP && prow ? 1.0 : -mr[r], vi = r == PP && prow ? 0.0 : -mi[r];
        a[r][RP].re[KV] = mine ? vr : a[r][RP].re[KV];
        a[r][RP].im[KV] = mine ? vi : a[r][RP].im[KV];
    }
}

// Inverse, in place, of a matrix of NR x NR parts of 16 x 16 by one wavefront,
// rows and columns from NS on in each part those of the identity: Gauss-Jordan
// with partial pivoting (the rule of gj_inverse_wave: rows are not exchanged,
// a pivot row is not divided by its pivot but keeps the scale s).  The pivot
// column crosses the rows of 16 lanes by ds_bpermute, the pivot row goes to
// the other rows the same way, and the pivot by v_readlane.  The product of an
// update is formed before it is subtracted (one rounding at the size of the
// element, not two).  lds: two planes
// of 16 NR x (16 NR + 1) of this wavefront, through which the result returns to
// the natural order.
template <int NR, int NS>
__device__ __forceinline__ void inverse16s(M16 (&a)[NR][NR], double* lds, int lane)
{
    constexpr int ld = 16 * NR + 1, plane = 16 * NR * ld;
    const int i = lane & 15, q = lane >> 4;
    unsigned used = 0u;  // rows that have been a pivot (wave-uniform)
    int perm = lane;     // lane k: the pivot row of column k
    int qrow[NR];        // column whose pivot this lane's row was
    double sr[NR], si[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        qrow[r] = 16 * r + i;
        sr[r] = 1.0;
        si[r] = 0.0;
    }
    auto column = [&](auto rp_c, auto kv_c) {
        constexpr int RP = decltype(rp_c)::value, KV = decltype(kv_c)::value;
#pragma unroll 1
        for (int kq = 0; kq < 4; ++kq) {
            const int k = 16 * RP + 4 * KV + kq;
            const int addr = (kq * 16 + i) * 4;
            double cr[NR], ci[NR];
            unsigned key = 0u;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                cr[r] = bperm64(addr, a[r][RP].re[KV]);
                ci[r] = bperm64(addr, a[r][RP].im[KV]);
                const bool free = (NS == 16 || i < NS) && !((used >> (16 * r + i)) & 1u);
                const unsigned kk = free ? pivot_key32(mag2(cr[r], ci[r]), 16 * r + i) : 0u;
                key = kk > key ? kk : key;
            }
            key = (unsigned)__builtin_amdgcn_readfirstlane((int)row_max32(key));
            constexpr unsigned live = NS == 16 ? 0xffffu : (1u << NS) - 1u;
            const unsigned left = ~used & (NR == 2 ? live | live << 16 : live);
            const int p = key == 0u ? __builtin_ctz(left) : 31 - (int)(key & 31u);
            used |= 1u << p;
            perm = lane == k ? p : perm;
            const int pl = p & 15;
            const bool hi = NR == 2 && p >= 16;  // wave-uniform
            const double pr = readlane_f64(hi ? cr[NR - 1] : cr[0], pl), pi = readlane_f64(hi ? ci[NR - 1] : ci[0], pl);
            const double iv = recip_nr(fma(pr, pr, pi * pi));
            const double ir = pr * iv, ii = -pi * iv;
            const bool mine = q == kq;
#pragma unroll
            for (int r = 0; r < NR; ++r) qrow[r] = 16 * r + i == p ? k : qrow[r];
            if (hi)
                gj_update<NR, RP, KV, NR - 1>(a, cr, ci, ir, ii, pl, mine, sr, si, lane);
            else
                gj_update<NR, RP, KV, 0>(a, cr, ci, ir, ii, pl, mine, sr, si, lane);
        }
    };
    auto part = [&](auto rp_c) {
        column(rp_c, std::integral_constant<int, 0>());
        if constexpr (NS > 4) column(rp_c, std::integral_constant<int, 1>());
        if constexpr (NS > 8) column(rp_c, std::integral_constant<int, 2>());
        if constexpr (NS > 12) column(rp_c, std::integral_constant<int, 3>());
    };
    part(std::integral_constant<int, 0>());
    if constexpr (NR == 2) part(std::integral_constant<int, 1>());
    // A^-1[qrow][perm_j] = s_i M[i][j]
#pragma unroll
    for (int c = 0; c < NR; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = __builtin_amdgcn_ds_bpermute((16 * c + q + 4 * v) * 4, perm);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const double x = a[r][c].re[v], y = a[r][c].im[v];
                lds[qrow[r] * ld + j] = fma(sr[r], x, -si[r] * y);
                lds[plane + qrow[r] * ld + j] = fma(sr[r], y, si[r] * x);
            }
        }
    wave_sync();
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int c = 0; c < NR; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int x = 16 * r + i, y = 16 * c + q + 4 * v;
                a[r][c].re[v] = lds[x * ld + y];
                a[r][c].im[v] = lds[plane + x * ld + y];
            }
    wave_sync();
}

// value of lane K of this lane's row of 16 (DPP row_newbcast)
template <int K>
__device__ __forceinline__ double row_lane(double x)
{
    return __builtin_amdgcn_mov_dpp(x, 0x150 + K, 0xF, 0xF, true);
}

// A multiplier of a later row above the limit (squared here) sends the matrix to
// the pivoted inverse16s.  The sweep of the chain (256): up to 6% of the blocks at
// energies within the edge states of a disordered (16,0) tube, under 1%
// elsewhere; the bits lost there are fewer than the condition of those blocks
// costs (diag G within 1e-10 of the dense inverse given Sigma, as with a limit
// of 8, which took 16 instead of 9 ms for 500 x 1024 as half of those blocks
// are inverted twice).
// The leads (4): the doublings amplify every error.  Mean of log10(error of Sigma,
// 80-bit references) less that of the 32-orbital kernel, ring tubes and random chains of 8 to 32
// orbitals, Im E 1e-5 .. 0.1 / on the contour (largest of a chain and Im E), and the time
// of a solve of 40 blocks of 20 orbitals: limit 8 0.16 / -0.08 (0.58), 652 us; 5 0.08 /
// -0.08 (0.28), 688; 4 0.05 / -0.08 (0.14), 730; 3 0.02 / -0.08 (0.12), 883; pivoted always
// 0.01 / 0.01 (0.12), 857.  256 costs up to four digits.
constexpr double CHAIN_GROW2 = 256.0 * 256.0, LEAD_GROW2 = 4.0 * 4.0;

// Elimination step on column 4 T + K of a panel x (columns 4 T .. 4 T + 3; lane
// (i, q): row i, column 4 T + q), pivot in row 4 T + K of the panel's own part.
// x[1] (if NR = 2): the panel's rows in the other part, check: not yet pivots.
// Ends with -A_iJ P^-1 in the other rows and P^-1 in rows J.  In the leads (NR = 2) the
// products are formed before they are added, as in inverse16s.
template <int T, int K, int NR>
__device__ __forceinline__ void panel_step(double2 (&x)[NR], int lane, bool& grow, bool check = false)
{
    constexpr int row = 4 * T + K;
    asm volatile("" : "+v"(lane));  // the lane masks are made here: kept over all steps they spill
    const int i = lane & 15;
    const int addr = (K * 16 + i) * 4;
    const bool col = (lane >> 4) == K, prow = i == row;
    double2 c[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) c[r] = make_double2(bperm64(addr, x[r].x), bperm64(addr, x[r].y));
    const double pr = row_lane<row>(c[0].x), pi = row_lane<row>(c[0].y);
    // 1 / |pivot|^2: estimate and one third-order step y (1 + e + e^2), e = 1 - d y
    const double d = fma(pr, pr, pi * pi), y = __builtin_amdgcn_rcp(d), ee = fma(-d, y, 1.0);
    const double iv = fma(y, fma(ee, ee, ee), y);
    const double ir = pr * iv, ni = pi * iv;  // 1 / pivot = ir - i ni
    double rr = row_lane<row>(x[0].x), ri = row_lane<row>(x[0].y);
    rr = col ? 1.0 : rr;
    ri = col ? 0.0 : ri;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        // -c / pivot
        double fr = -fma(c[r].x, ir, c[r].y * ni), fi = fma(c[r].x, ni, -c[r].y * ir);
        const bool big = !(fma(fr, fr, fi * fi) <= (NR == 1 ? CHAIN_GROW2 : LEAD_GROW2));
        grow |= r == 0 ? big && i > row : check && big;
        const bool p = r == 0 && prow;
        fr = p ? ir : fr;
        fi = p ? -ni : fi;
        const bool z = p || col;
        const double br = z ? 0.0 : x[r].x, bi = z ? 0.0 : x[r].y;
        if (NR == 1) {
            x[r].x = fma(fr, rr, fma(-fi, ri, br));
            x[r].y = fma(fr, ri, fma(fi, rr, bi));
        } else {
            x[r].x = br + fma(fr, rr, -fi * ri);
            x[r].y = bi + fma(fr, ri, fi * rr);
        }
    }
}

template <int T>
__device__ __forceinline__ void panel_steps(double2 (&x)[2], int lane, bool& grow, bool check)
{
    panel_step<T, 0, 2>(x, lane, grow, check);
    panel_step<T, 1, 2>(x, lane, grow, check);
    panel_step<T, 2, 2>(x, lane, grow, check);
    panel_step<T, 3, 2>(x, lane, grow, check);
}

// a(i, j) += sum_k o[j][k] b[i][k] for panels o and b (SUM: the sum formed first)
template <bool SUM = false>
__device__ __forceinline__ void rank4(M16& a, const double2& o, const double2& b)
{
    if constexpr (SUM) {
        M16 c = zero16();
        rank4(c, o, b);
        a.re += c.re;
        a.im += c.im;
        return;
    }
    a.re = mfma64(o.x, b.x, a.re);
    a.im = mfma64(o.x, b.y, a.im);
    a.re = mfma64(-o.y, b.y, a.re);
    a.im = mfma64(o.y, b.x, a.im);
}

// rows 4 T .. 4 T + 3 set to zero
template <int T>
__device__ __forceinline__ void clear_rows(M16& a, int lane)
{
    const bool z = ((lane & 15) >> 2) == T;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        a.re[v] = z ? 0.0 : a.re[v];
        a.im[v] = z ? 0.0 : a.im[v];
    }
}

// a <- -a^-1 for NB complex symmetric matrices at once (independent chains of
// instructions), NS rows and columns not those of the identity (the others end
// at 1 instead of -1 and meet only zeros).
template <int NS, int NB, int T = 0>
__device__ __forceinline__ void sweep16(M16 (&a)[NB], int lane, bool (&grow)[NB])
{
    double2 x[NB][1], o[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) x[n][0] = o[n] = make_double2(a[n].re[T], a[n].im[T]);
#pragma unroll
    for (int n = 0; n < NB; ++n) panel_step<T, 0, 1>(x[n], lane, grow[n]);
#pragma unroll
    for (int n = 0; n < NB; ++n) panel_step<T, 1, 1>(x[n], lane, grow[n]);
#pragma unroll
    for (int n = 0; n < NB; ++n) panel_step<T, 2, 1>(x[n], lane, grow[n]);
#pragma unroll
    for (int n = 0; n < NB; ++n) panel_step<T, 3, 1>(x[n], lane, grow[n]);
#pragma unroll
    for (int n = 0; n < NB; ++n) {
        clear_rows<T>(a[n], lane);
        rank4(a[n], o[n], x[n][0]);
        a[n].re[T] = -x[n][0].x;
        a[n].im[T] = -x[n][0].y;
    }
    if constexpr (4 * T + 4 < NS) sweep16<NS, NB, T + 1>(a, lane, grow);
}

// -a^-1 of NB matrices, by sweep16 or, where that grows, with pivoting
template <int NS, int NB>
__device__ __forceinline__ void neg_inverse16(M16 (&a)[NB], double* lds, int lane)
{
    M16 keep[NB];
    bool grow[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
        keep[n] = a[n];
        grow[n] = false;
    }
    sweep16<NS, NB>(a, lane, grow);
    // (one copy of the elimination for all matrices)
    bool any[NB];
    bool some = false;
#pragma unroll
    for (int n = 0; n < NB; ++n) some |= any[n] = __any(grow[n]);
    if (!some) return;
#pragma unroll 1
    for (int k = 0; k < NB; ++k) {
        if (!any[NB == 1 ? 0 : k]) continue;
        M16 b[1][1] = {{NB == 2 && k ? keep[NB - 1] : keep[0]}};
        inverse16s<1, NS>(b, lds, lane);
        b[0][0].re = -b[0][0].re;
        b[0][0].im = -b[0][0].im;
        if (NB == 2 && k)
            a[NB - 1] = b[0][0];
        else
            a[0] = b[0][0];
    }
}

constexpr int SLD = 17;            // row stride of a 16 x 16 LDS plane
constexpr int SPL = 16 * SLD;

// transposed through LDS (two planes of SPL)
__device__ __forceinline__ M16 transpose16(const M16& m, double* lds, int lane)
{
    const int i = lane & 15, q = lane >> 4;
    M16 t;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        lds[i * SLD + q + 4 * v] = m.re[v];
        lds[SPL + i * SLD + q + 4 * v] = m.im[v];
    }
    wave_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        t.re[v] = lds[(q + 4 * v) * SLD + i];
        t.im[v] = lds[SPL + (q + 4 * v) * SLD + i];
    }
    wave_sync();
    return t;
}

// (m + m^T) / 2.  The sweep reads columns where rows are meant, which is only
// right (and only stable over a chain of inverses or doublings: an antisymmetric
// rounding error grows from one to the next) for an exactly symmetric matrix.
__device__ __forceinline__ M16 symmetric16(const M16& m, double* lds, int lane)
{
    const M16 t = transpose16(m, lds, lane);
    return M16{0.5 * (m.re + t.re), 0.5 * (m.im + t.im)};
}

// -A^-1 of the 32 x 32 complex symmetric matrix of the parts pp, rp (rows R,
// columns P) and rr, by the sweep over the columns of P, then of R.  On return
// rp holds the rows P, columns R.
template <int NS, int T = 0>
__device__ __forceinline__ void sweep32_part(M16& own, M16& cross, M16& other, int lane, bool& grow, bool check)
{
    double2 x[2] = {make_double2(own.re[T], own.im[T]), make_double2(cross.re[T], cross.im[T])};
    const double2 o0 = x[0], o1 = x[1];
    panel_steps<T>(x, lane, grow, check);
    clear_rows<T>(own, lane);
    rank4<true>(own, o0, x[0]);
    rank4<true>(cross, o0, x[1]);
    rank4<true>(other, o1, x[1]);
    own.re[T] = -x[0].x;
    own.im[T] = -x[0].y;
    cross.re[T] = -x[1].x;
    cross.im[T] = -x[1].y;
    if constexpr (4 * T + 4 < NS) {
        if (__any(grow)) return;  // the caller discards the matrix
        sweep32_part<NS, T + 1>(own, cross, other, lane, grow, check);
    }
}

template <int NS>
__device__ __forceinline__ bool sweep32(M16& pp, M16& rp, M16& rr, double* lds, int lane)
{
    // the columns of P, then (parts exchanged, one copy of the code) those of R
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        bool grow = false;
        sweep32_part<NS>(pp, rp, rr, lane, grow, half == 0);
        if (__any(grow)) return false;
        if (half == 0) rp = transpose16(rp, lds, lane);
        const M16 t = pp;
        pp = rr;
        rr = t;
    }
    return true;
}

// E - H - diag(v) - ... of one part: the diagonal of rows i < np gets (er, ei)
// less the potential; padding rows get 1.
__device__ __forceinline__ void add_diag(M16& a, double er, double ei, int np, int lane)
{
    const int i = lane & 15, q = lane >> 4;
    const double dr = i < np ? er : 1.0, di = i < np ? ei : 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (q + 4 * v == i) {
            a.re[v] += dr;
            a.im[v] += di;
        }
}

__device__ __forceinline__ d4 load_real16(const double* __restrict__ m, bool transpose, int lane)
{
    const int i = lane & 15, q = lane >> 4;
    d4 r;
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = transpose ? m[(q + 4 * v) * 16 + i] : m[i * 16 + q + 4 * v];
    return r;
}

__device__ __forceinline__ void store16(double2* __restrict__ dst, const M16& m, int lane)
{
#pragma unroll
    for (int v = 0; v < 4; ++v) dst[v * 64 + lane] = make_double2(m.re[v], m.im[v]);
}
__device__ __forceinline__ M16 load16(const double2* __restrict__ src, int lane)
{
    M16 m;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const double2 x = src[v * 64 + lane];
        m.re[v] = x.x;
        m.im[v] = x.y;
    }
    return m;
}

// Block RGF of one energy (blockIdx.x) by two wavefronts, one from each lead.
// Part beta = 0 .. 2 nb - 1 has the orbitals of part beta % 2 of block beta / 2;
// wavefront side = 0 takes beta = j and side = 1 beta = 2 nb - 1 - j at step j,
// j = 0 .. 2 nb - 1.  The coupling from step j to step j + 1 joins the same pair
// of parts on both sides (H_01 for even j, T_10 for odd), read from its other
// end on the right.  Sn is the negated self-energy of the parts already passed.
template <int NS>
__global__ __launch_bounds__(128, 2) void split_rgf_kernel(SplitChain c, int e0, const double2* __restrict__ E,
                                                           const double2* __restrict__ coef,
                                                           const double* __restrict__ sigma, double2* scratch,
                                                           double* __restrict__ part, double2* __restrict__ diag)
{
    __shared__ double lds_all[2][2 * SPL];
    const int lane = threadIdx.x & 63, side = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double* lds = lds_all[side];
    const int el = blockIdx.x, e = e0 + el;
    const int nb = c.nb, m = c.m, h = c.h;
    const int i = lane & 15, q = lane >> 4;
    const double2 z = E[e], cf = coef[e];
    double2* own = scratch + ((size_t)el * 2 + side) * nb * 256;            // Sn of this side's first nb parts
    const double2* other = scratch + ((size_t)el * 2 + 1 - side) * nb * 256;
    d4 H[2], Ct[2];  // of even and odd steps: on-site, and the coupling's transpose
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        H[p] = load_real16(c.mats + (side ? 1 - p : p) * 256, false, lane);
        Ct[p] = load_real16(c.mats + (2 + p) * 256, side == 0, lane);
    }
    auto pot = [&](int j) {  // potential of this lane's orbital at step j
        const int beta = side ? 2 * nb - 1 - j : j, p = beta & 1;
        const int np = p ? m - h : h;
        return c.v[(size_t)(beta >> 1) * BM + p * h + min(i, np - 1)];
    };
    M16 Sn = load16(reinterpret_cast<const double2*>(sigma) + ((size_t)e * 2 + side) * 256, lane);
    Sn.re = -Sn.re;
    Sn.im = -Sn.im;
    double vj = pot(0);
    // E - H - v + Sn of step j, and the potential of the next step.  H[0], Ct[0] are
    // those of the present step: exchanged after each step, one copy of the code
    // serves both parities (the inverses unrolled for each filled the
    // instruction cache)
    auto matrix = [&](int j) {
        M16 A;
        A.re = Sn.re - H[0];
        A.im = Sn.im;
        add_diag(A, z.x - vj, z.y, (side ^ (j & 1)) ? m - h : h, lane);
        vj = pot(min(j + 1, 2 * nb - 1));
        return A;
    };
    auto advance = [&](const M16& gn) {  // gn = -g
        const M16 Q = prod_cr<NS>(gn, Ct[0], zero16());
        Sn = symmetric16(prod_cr<NS>(Q, Ct[0], zero16()), lds, lane);
        const d4 th = H[0], tc = Ct[0];
        H[0] = H[1];
        Ct[0] = Ct[1];
        H[1] = th;
        Ct[1] = tc;
    };
    // ---- to the middle
#pragma unroll 1
    for (int j = 0; j < nb; ++j) {
        store16(own + (size_t)j * 256, Sn, lane);
        M16 a[1] = {matrix(j)};
        neg_inverse16<NS, 1>(a, lds, lane);
        advance(a[0]);
    }
    __syncthreads();  // the other side's self-energies are stored
    // ---- through the other half
    M16 So = load16(other + (size_t)(nb - 1) * 256, lane);
#pragma unroll 1
    for (int j = nb; j < 2 * nb; ++j) {
        M16 a[2];
        a[0] = matrix(j);
        a[1] = M16{a[0].re + So.re, a[0].im + So.im};
        So = load16(other + (size_t)max(2 * nb - 2 - j, 0) * 256, lane);
        neg_inverse16<NS, 2>(a, lds, lane);
        const int beta = side ? 2 * nb - 1 - j : j, bp = beta & 1;
        if (i < (bp ? m - h : h) && (i & 3) == q) {
            const int v = i >> 2;
            const d4 re = a[1].re, im = a[1].im;
            const double gr = -(v == 0 ? re[0] : v == 1 ? re[1] : v == 2 ? re[2] : re[3]);
            const double gi = -(v == 0 ? im[0] : v == 1 ? im[1] : v == 2 ? im[2] : im[3]);
            const size_t o = (size_t)e * nb * m + (size_t)(beta >> 1) * m + bp * h + i;
            part[o] = fma(cf.x, gi, cf.y * gr);
            if (diag) diag[o] = make_double2(gr, gi);
        }
        advance(a[0]);
    }
}

// Sancho-Rubio decimation of one energy (blockIdx.x) by one wavefront per lead
// (side 0 left, 1 right).  Part P = side is the lead's surface part that
// couples to the device, part R the other; the inter-block coupling has the one
// nonzero part a (rows P, columns R), which stays so under alpha <- alpha G
// alpha, and beta = alpha^T.  With G = (E - eps)^-1 (32 x 32, parts PP .. RR):
//   eps_PP += a G_RR a^T (and the surface's),  eps_RR += a^T G_PP a,
//   a <- a G_RP a,   Sigma = a0 g_RR a0^T on part P,  g = (E - eps_s)^-1.
// The bare parts (E - H_PP) can be singular on the real axis, where the sweep
// over P grows and the pivoted 32-column elimination takes over; G_PR is then the mean of
// it and the transpose of G_RP (the sweep's are one matrix).  The updates
// of eps are made exactly symmetric: without that an antisymmetric rounding
// error doubles with every iteration (1e-8 of Sigma after 22 at E = -0.9 + 1e-5i
// on the (16,0) tube; 7e-13 with it).
template <int NS>
__global__ __launch_bounds__(128, 1) void split_sr_kernel(SplitChain c, const double2* __restrict__ E, double Uc0,
                                                          double Uc1, double tol, int max_iter,
                                                          double* __restrict__ sigma, int* __restrict__ iters)
{
    __shared__ double lds_all[2][2 * BPL];
    const int lane = threadIdx.x & 63, side = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e = blockIdx.x;
    double* lds = lds_all[side];
    const double2 z = E[e];
    const double er = z.x - (side ? Uc1 : Uc0), ei = z.y;
    const int nP = side ? c.m - c.h : c.h, nR = c.m - nP;
    const d4 HP = load_real16(c.mats + side * 256, false, lane), HR = load_real16(c.mats + (1 - side) * 256, false, lane);
    const d4 HPR = load_real16(c.mats + 2 * 256, side == 1, lane);  // H_01, or its transpose
    const d4 HRP = load_real16(c.mats + 2 * 256, side == 0, lane);
    const d4 zr = d4{0, 0, 0, 0};
    const d4 a0 = load_real16(c.mats + 3 * 256, side == 0, lane);   // T_10^T (left), T_10 (right)
    M16 a = M16{a0, zr}, at = M16{load_real16(c.mats + 3 * 256, side == 1, lane), zr};
    M16 es = M16{HP, zr}, eP = es, eR = M16{HR, zr};
    // -G of the on-site matrices p, r: parts PP, PR, RR
    auto green = [&](const M16& p, const M16& r, M16& gpp, M16& gpr, M16& grr) {
        gpp = M16{-p.re, -p.im};
        gpr = M16{-HRP, zr};  // rows R, columns P until the sweep exchanges them
        grr = M16{-r.re, -r.im};
        add_diag(gpp, er, ei, nP, lane);
        add_diag(grr, er, ei, nR, lane);
        if (sweep32<NS>(gpp, gpr, grr, lds, lane)) return;
        M16 G[2][2] = {{M16{-p.re, -p.im}, M16{-HPR, zr}}, {M16{-HRP, zr}, M16{-r.re, -r.im}}};
        add_diag(G[0][0], er, ei, nP, lane);
        add_diag(G[1][1], er, ei, nR, lane);
        inverse16s<2, NS>(G, lds, lane);
        gpp = M16{-G[0][0].re, -G[0][0].im};
        const M16 t = transpose16(G[1][0], lds, lane);
        gpr = M16{-0.5 * (G[0][1].re + t.re), -0.5 * (G[0][1].im + t.im)};
        grr = M16{-G[1][1].re, -G[1][1].im};
    };
    // the last pass (conv or it == max_iter) is the surface's own G, of es; one
    // copy of the elimination serves both
    int it = 0;
    bool conv = false;
    M16 sg;
    for (;;) {
        const bool last = conv || it >= max_iter;
        M16 gpp, gpr, grr;
        green(last ? es : eP, last ? M16{HR, zr} : eR, gpp, gpr, grr);
        if (last) {
            const M16 Y = prod_cr<NS>(grr, a0, zero16());                   // -a0 g_RR
            sg = symmetric16(prod_rc<NS>(a0, Y, zero16()), lds, lane);      // -a0 g_RR a0^T
            break;
        }
        ++it;
        const M16 Y = prod_cc<NS>(grr, a, zero16());    // -a G_RR
        const M16 d = symmetric16(prod_cc<NS>(a, Y, zero16()), lds, lane);  // -a G_RR a^T
        es.re -= d.re;
        es.im -= d.im;
        eP.re -= d.re;
        eP.im -= d.im;
        const M16 Y2 = prod_cc<NS>(gpp, at, zero16());  // -a^T G_PP
        const M16 d2 = symmetric16(prod_cc<NS>(at, Y2, zero16()), lds, lane);  // -a^T G_PP a
        eR.re -= d2.re;
        eR.im -= d2.im;
        const M16 Y3 = prod_cc<NS>(gpr, a, zero16());   // -a G_RP
        a = prod_cc<NS>(at, Y3, zero16());              // -a G_RP a
        a.re = -a.re;
        a.im = -a.im;
        at = transpose16(a, lds, lane);
        double mx = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) mx = nan_max(mx, mag2(a.re[v], a.im[v]));
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) mx = nan_max(mx, __shfl_xor(mx, off));
        conv = mx < tol * tol;
    }
    sg.re = -sg.re;
    sg.im = -sg.im;
    store16(reinterpret_cast<double2*>(sigma) + ((size_t)e * 2 + side) * 256, sg, lane);
    if (lane == 0) iters[e * 2 + side] = conv ? it : -it;
}

int split_part_size(int m, const double* T, int ld)
{
    int rmin = m, cmax = -1;
    for (int i = 0; i < m; ++i)
        for (int j = 0; j < m; ++j)
            if (T[i * ld + j] != 0.0) {
                rmin = std::min(rmin, i);
                cmax = std::max(cmax, j);
            }
    int best = 0;
    for (int h = std::max({1, cmax + 1, m - 16}); h <= std::min({m - 1, rmin, 16}); ++h)
        if (!best || std::max(h, m - h) < std::max(best, m - best)) best = h;
    return best;
}

void split_matrices(int m, int h, const double* H0, const double* T, int ld, double* mats)
{
    std::fill(mats, mats + 4 * 256, 0.0);
    for (int i = 0; i < h; ++i) {
        for (int j = 0; j < h; ++j) mats[i * 16 + j] = H0[i * ld + j];
        for (int j = h; j < m; ++j) mats[2 * 256 + i * 16 + j - h] = H0[i * ld + j];
    }
    for (int i = h; i < m; ++i) {
        for (int j = h; j < m; ++j) mats[256 + (i - h) * 16 + j - h] = H0[i * ld + j];
        for (int j = 0; j < h; ++j) mats[3 * 256 + (i - h) * 16 + j] = T[i * ld + j];
    }
}

// columns in use, rounded up to the MFMA's four
static int split_ns(const SplitChain& c) { return (std::max(c.h, c.m - c.h) + 3) / 4 * 4; }

hipError_t split_sancho_rubio(const SplitChain& c, int nE, const double2* E, double Uc0, double Uc1, double tol,
                              int max_iter, double* sigma, int* iters, hipStream_t st)
{
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nE), dim3(128), 0, st, c, E, Uc0, Uc1, tol, max_iter, sigma, iters);
    };
    switch (split_ns(c)) {
        case 4: launch(split_sr_kernel<4>); break;
        case 8: launch(split_sr_kernel<8>); break;
        case 12: launch(split_sr_kernel<12>); break;
        default: launch(split_sr_kernel<16>); break;
    }
    return hipGetLastError();
}

hipError_t split_rgf(const SplitChain& c, int e0, int n, const double2* E, const double2* coef, const double* sigma,
                     double2* scratch, double* part, double2* diag, hipStream_t st)
{
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(n), dim3(128), 0, st, c, e0, E, coef, sigma, scratch, part, diag);
    };
    switch (split_ns(c)) {
        case 4: launch(split_rgf_kernel<4>); break;
        case 8: launch(split_rgf_kernel<8>); break;
        case 12: launch(split_rgf_kernel<12>); break;
        default: launch(split_rgf_kernel<16>); break;
    }
    return hipGetLastError();
}

}  // namespace negf
