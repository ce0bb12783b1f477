// surrogate.hip -- 1D-convolutional surrogate U -> Q of a tube's NEGF
// charge, with hand-written BF16 MFMA (FP32 accumulate) inference, tangent
// and training kernels for gfx950.  It has no counterpart in the reference:
// it seeds and preconditions the batched Broyden SCF, while the exact NEGF
// computes every residual that decides convergence.
//
// Network (sites n = 0..N-1, zero padding at the chain ends):
//   x0[n] = (U_n / 0.5 eV, exp(-min(n, N-1-n) / 16), f)   3 channels, padded to 32
//   5 x   x = tanh(conv9(x) + b)                          64 channels
//   q[n]  = conv9(x) + b                                  1 channel, padded to 32
//   Q_n   = mean_Q + scale_Q q_n
// f is a per-sample scalar feature (e.g. the drain bias), 0 when unused.
//
// Layouts: activations bf16 [b][n][c] (channels fastest); weights bf16
// [co][tap][ci] with FP32 master copies for Adam; the transposed, flipped
// copy Wt[ci][tap][co] = W[co][8 - tap][ci] turns the data gradient into a
// forward convolution.
//
// The five convolutions into 64 channels (forward, tangent, or the data
// gradient of layers 5..1) and the last layer run as one launch over tiles of
// sites, the activations in LDS (sg_chain_kernel).  Every convolution is an
// implicit GEMM on v_mfma_f32_16x16x32_bf16: M = 16 output channels, N = 16
// sites, K = 9 taps x input channels.  Operand layout: lane l
// holds A[i][k] with i = l % 16 and B[k][j] with j = l % 16 for the same
// eight k of its 16-lane group, and receives D[i][j] for i = 4 (l / 16) + v,
// v = 0..3, j = l % 16.  (Which eight k a lane group holds does not matter:
// A and B use the same assignment, so the sum over k is unchanged.)
#include "surrogate.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>

#include "negf_material.h"

namespace negf {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f4;

__device__ __forceinline__ f4 mfma_bf16(const bf16x8& a, const bf16x8& b, const f4& c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// tanh for a result rounded to BF16: x P(x^2) / Q(x^2) with the coefficients of
// a weighted least-squares fit to tanh(x) / x on [0, 4] (relative error below
// 4e-7), beyond 4 the value at 4 (0.99933, which rounds to 1).  Nine
// instructions and one v_rcp_f32; the epilogues of a layer take as long as its
// MFMAs, so this is the other half of the kernel's time.
__device__ __forceinline__ float sg_tanh(float x)
{
    x = __builtin_amdgcn_fmed3f(x, -4.0f, 4.0f);
    const float s = x * x;
    const float p = fmaf(s, fmaf(s, 1.75496324e-3f, 1.18174323e-1f), 9.99999645e-1f);
    const float q = fmaf(s, fmaf(s, fmaf(s, 7.30915899e-5f, 1.89287477e-2f), 4.51504160e-1f), 1.0f);
    return x * p * __builtin_amdgcn_rcpf(q);
}

// ---- the whole network on a tile of sites
//   SG_FWD   x_1 = tanh(conv(x_0) + b_0), ..., x_5; q = conv(x_5) + b_5
//   SG_TAN   the tangent of the same: t_{l+1} = conv(t_l) (1 - x_{l+1}^2)
//   SG_BWD   data gradients: dz_4 = conv(dq; Wt_5) (1 - x_5^2), ..., dz_0
// One workgroup of 8 wavefronts per (tile of T sites, sample).  All layers are
// computed on the window of T + 40 sites (the last one needs four more sites on
// each side per layer before it; what lies further out is not used), from one
// LDS buffer into the other, so no activation makes a round trip through
// memory; with STORE the tile's part of every layer is also written out.
//
// The window has 16 R sites and lane i of an operand holds site r + R i of row r:
// the tap shift is then another row, not another lane, and the fragments of
// rows r - 4 .. r + U + 3 serve U output rows: 2 (U + 8) LDS reads for 18 U
// MFMAs (a layout with lane = neighbouring site needs 18 U).  Wavefront w makes
// output channels 16 (w % 4) .. + 15 of half of the rows, its 18 weight
// fragments in registers and those of the next layer on their way.
// The first layer has one or three real channels: their nine taps fill one K
// block (im2col in LDS).  The last layer has one output channel: its nine taps
// are the M rows, z[tap][s] = sum_ci W[tap][ci] x[s][ci], summed as
// q[n] = sum_tap z[tap][n + tap - 4].
// Bound by MFMA and the epilogues' VALU (tanh): a row of a layer takes 500 cycles
// of a CU, its MFMAs 290 and its epilogues about 350 (two wavefronts per SIMD,
// partly overlapped; epilogues placed between the next rows' MFMAs by hand
// and raised priorities for half of the wavefronts gained nothing), and about 15 us
// per workgroup are latencies of the layers' first loads and barriers.
// Measured, 128 x 2048 sites: 105 us for the forward pass against 185 us for one
// launch per layer (each LDS fragment read for two MFMAs, activations through
// memory); 32 x 2048 with the activations written: 50 against 107 us, the data
// gradients of layers 5..1: 46 against 87 us.
enum SgMode { SG_FWD = 0, SG_TAN = 1, SG_BWD = 2 };
constexpr int CH_HALO = SG_HALO * (SG_LAYERS - 1);  // window sites beyond the tile, per side
constexpr int CH_RMAX = 36;                         // rows of a window: 153 KiB of LDS
constexpr int CH_WMAX = 16 * CH_RMAX;

struct SgChainArgs {
    int N, T, R;                        // sites per sample and tile, rows of a window (16 R >= T + 2 CH_HALO)
    const double* in;                   // U or V [B][N]
    const double* feat;                 // [B] or null
    const __bf16* dq;                   // SG_BWD: gradient at the output [B][N]
    const __bf16* w[SG_LAYERS];         // weights of step s: layer s, or layer 5 - s transposed
    const float* bias[SG_LAYERS];
    __bf16* x[SG_LAYERS];               // x_1 .. x_5 (index 1 ..): written (SG_FWD, STORE) or read
    __bf16* dz[SG_LAYERS];              // SG_BWD: dz_0 .. dz_4, written
    float* q;                           // output [B][N] (may be null)
    double* Q;                          // mean + scale q (may be null)
    double mean, scale;
};

template <int U>
struct ChOut {
    f4 acc[U];
};

// U output rows from r0 on: acc[u] += sum over taps and channels.  Row r = -4 ..
// R + 3 of a lane (i, g) is the site s = r + R i; 16-byte chunk c of a site lies
// at c ^ (s / R mod 8), and s / R is i - 1 (below row 0), i or i + 1 (from row R
// on): olo, omid, ohi are the byte offsets of chunk g of site R i in those cases.
template <int U>
__device__ __forceinline__ void ch_rows(const char* buf, int olo, int omid, int ohi, int r0, int R,
                                        const bf16x8 (&a)[SG_KW][2], ChOut<U>& o)
{
#pragma unroll
    for (int t = 0; t < U + 2 * SG_HALO; ++t) {
        const int row = r0 - SG_HALO + t;  // wave-uniform
        const int off = row < 0 ? olo : row >= R ? ohi : omid;
        const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(buf + row * 128 + off);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(buf + row * 128 + (off ^ 64));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int tap = t - u;
            if (tap < 0 || tap >= SG_KW) continue;
            o.acc[u] = mfma_bf16(a[tap][0], b0, o.acc[u]);
            o.acc[u] = mfma_bf16(a[tap][1], b1, o.acc[u]);
        }
    }
}

// tanh (SG_FWD) or (1 - y^2) (y: this lane's four channels of xp) of one row,
// rounded to BF16, zero outside the sample, into the other buffer
template <int MODE>
__device__ __forceinline__ void ch_store(const f4& acc, uint2 xp, bool inside, char* dst)
{
    const __bf16* y = reinterpret_cast<const __bf16*>(&xp);
    f4 z;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (MODE == SG_FWD) {
            z[v] = sg_tanh(acc[v]);
        } else {
            const float yv = (float)y[v];
            z[v] = acc[v] * fmaf(-yv, yv, 1.0f);
        }
    }
    uint2 r = __builtin_bit_cast(uint2, __builtin_convertvector(z, bf16x4));
    if (!inside) r = make_uint2(0u, 0u);
    *reinterpret_cast<uint2*>(dst) = r;
}

template <int MODE, bool STORE>
__global__ __launch_bounds__(512) void sg_chain_kernel(SgChainArgs p)
{
    __shared__ __attribute__((aligned(16))) char buf[2][(CH_WMAX + 2 * SG_HALO) * 128];
    __shared__ __bf16 plane[SG_IN][CH_WMAX + 4 * SG_HALO];  // inputs of sites -8 .. W + 7
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int cw = w & 3, rg = w >> 2;  // this wavefront's channels and rows
    const int N = p.N, T = p.T, R = p.R, W = 16 * R;
    const int b = blockIdx.y;
    const int n0 = blockIdx.x * T, nw = n0 - CH_HALO;  // first site of the tile and of the window
    const size_t base = (size_t)b * N;
    // ---- inputs
    for (int k = tid; k < W + 4 * SG_HALO; k += 512) {
        const int n = nw - 2 * SG_HALO + k;
        const bool in = n >= 0 && n < N;
        const int nc = min(max(n, 0), N - 1);
        __bf16 v0 = (__bf16)0.0f, v1 = v0, v2 = v0;
        if (MODE == SG_BWD) {
            v0 = p.dq[base + nc];
        } else {
            v0 = (__bf16)(float)(p.in[base + nc] * 2.0);
            if (MODE == SG_FWD) {
                v1 = (__bf16)expf(-(float)min(nc, N - 1 - nc) * 0.0625f);
                v2 = (__bf16)(float)(p.feat ? p.feat[b] : 0.0);
            }
        }
        plane[0][k] = in ? v0 : (__bf16)0.0f;
        plane[1][k] = in ? v1 : (__bf16)0.0f;
        plane[2][k] = in ? v2 : (__bf16)0.0f;
    }
    // first layer's weights: k = 8 g + e is tap e of input g (g < 3), and tap 8 of input e (g = 3)
    bf16x8 a0;
    {
        const __bf16* w0 = p.w[0] + (size_t)(16 * cw + i) * SG_KW * SG_CP;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            a0[e] = g < 3 ? w0[e * SG_CP + g] : e < 3 ? w0[8 * SG_CP + e] : (__bf16)0.0f;
    }
    bf16x8 a[SG_KW][2], an[SG_KW][2];
    auto load_w = [&](const __bf16* wl, bf16x8 (&d)[SG_KW][2]) {
        const __bf16* wr = wl + (size_t)(16 * cw + i) * SG_KW * SG_C + 8 * g;
#pragma unroll
        for (int t = 0; t < SG_KW; ++t)
#pragma unroll
            for (int k = 0; k < 2; ++k) d[t][k] = *reinterpret_cast<const bf16x8*>(wr + t * SG_C + 32 * k);
    };
    load_w(p.w[1], a);
    // the four sites beyond each end of buffer 0 stay zero (buffer 1: below)
    auto zero_ends = [&](char* bf) {
        if (tid < 64) {
            const int s = tid >> 3, c = tid & 7;  // sites -4 .. -1, W .. W + 3
            *reinterpret_cast<uint4*>(bf + (s < 4 ? s : W + s) * 128 + c * 16) = make_uint4(0u, 0u, 0u, 0u);
        }
    };
    zero_ends(buf[0]);
    __syncthreads();
    // im2col of the first layer in buffer 1: site s at 64 s bytes, chunk g at g ^ (s / R mod 4)
    for (int s = tid; s < W; s += 512) {
        __attribute__((aligned(16))) __bf16 col[32];
#pragma unroll
        for (int gg = 0; gg < 3; ++gg)
#pragma unroll
            for (int e = 0; e < 8; ++e) col[8 * gg + e] = plane[gg][s + SG_HALO + e];
#pragma unroll
        for (int e = 0; e < 8; ++e) col[24 + e] = e < 3 ? plane[e][s + SG_HALO + 8] : (__bf16)0.0f;
        const int f = (s / R) & 3;
#pragma unroll
        for (int gg = 0; gg < 4; ++gg)
            *reinterpret_cast<uint4*>(buf[1] + s * 64 + ((gg ^ f) << 4)) = reinterpret_cast<const uint4*>(col)[gg];
    }
    __syncthreads();
    const int olo = (4 + R * i) * 128 + ((g ^ ((i - 1) & 7)) << 4);
    const int omid = (4 + R * i) * 128 + ((g ^ (i & 7)) << 4);
    const int ohi = (4 + R * i) * 128 + ((g ^ ((i + 1) & 7)) << 4);
    const int half = (R + 1) >> 1;
    const int rb = rg ? half : 0, re = rg ? R : half;  // this wavefront's rows
    const int ch = 16 * cw + 4 * g;                    // this lane's first output channel
    const int dst0 = (4 + R * i) * 128 + (((2 * cw + (g >> 1)) ^ (i & 7)) << 4) + (g & 1) * 8;
    // step st makes layer output x_{st+1} (forward, tangent) or dz_{4-st}; the x it is scaled with:
    auto scale_src = [&](int st) { return p.x[MODE == SG_BWD ? SG_LAYERS - 1 - st : st + 1]; };
    auto load_xp = [&](const __bf16* xs, int r) {
        if (MODE == SG_FWD) return make_uint2(0u, 0u);
        const int n = min(max(nw + r + R * i, 0), N - 1);
        return *reinterpret_cast<const uint2*>(xs + (base + n) * SG_C + ch);
    };
    f4 bias0 = f4{0.f, 0.f, 0.f, 0.f};
    auto load_bias = [&](int st) {
        if (MODE == SG_FWD) {
#pragma unroll
            for (int v = 0; v < 4; ++v) bias0[v] = p.bias[st][ch + v];
        }
    };
    auto inside = [&](int r) { return (unsigned)(nw + r + R * i) < (unsigned)N; };
    // ---- first layer
    load_bias(0);
    {
        const __bf16* xs = MODE == SG_FWD ? nullptr : scale_src(0);
        for (int r = rb; r < re; ++r) {
            const uint2 xp = load_xp(xs, r);
            const int s = r + R * i;
            const bf16x8 bb = *reinterpret_cast<const bf16x8*>(buf[1] + s * 64 + ((g ^ (i & 3)) << 4));
            const f4 acc = mfma_bf16(a0, bb, bias0);
            ch_store<MODE>(acc, xp, inside(r), buf[0] + r * 128 + dst0);
        }
    }
    __syncthreads();
    zero_ends(buf[1]);
    __syncthreads();
    // the tile's sites of a buffer to memory, whole lines
    auto write_out = [&](const char* src, __bf16* dst) {
        const int nt = min(T, N - n0);
        for (int k = tid; k < nt * 8; k += 512) {
            const int t = k >> 3, c = k & 7, s = CH_HALO + t;
            const uint4 v = *reinterpret_cast<const uint4*>(src + (s + 4) * 128 + ((c ^ ((s / R) & 7)) << 4));
            *reinterpret_cast<uint4*>(dst + (base + n0 + t) * SG_C + c * 8) = v;
        }
    };
    // ---- hidden layers
#pragma unroll 1
    for (int st = 1; st < SG_LAYERS - 1; ++st) {
        const char* src = buf[(st + 1) & 1];
        char* dst = buf[st & 1];
        if (st + 1 < SG_LAYERS - 1) load_w(p.w[st + 1], an);
        if (STORE) write_out(src, MODE == SG_BWD ? p.dz[SG_LAYERS - 1 - st] : p.x[st]);
        load_bias(st);
        const __bf16* xs = MODE == SG_FWD ? nullptr : scale_src(st);
        auto pass = [&](auto u_c, int r0) {
            constexpr int U = decltype(u_c)::value;
            ChOut<U> o;
            uint2 xp[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                o.acc[u] = bias0;
                xp[u] = load_xp(xs, r0 + u);
            }
            ch_rows<U>(src, olo, omid, ohi, r0, R, a, o);
#pragma unroll
            for (int u = 0; u < U; ++u)
                ch_store<MODE>(o.acc[u], xp[u], inside(r0 + u), dst + (r0 + u) * 128 + dst0);
        };
        int r = rb;
#pragma unroll 1
        for (; r + 8 <= re; r += 8) pass(std::integral_constant<int, 8>(), r);
        if (r + 4 <= re) {
            pass(std::integral_constant<int, 4>(), r);
            r += 4;
        }
        if (r + 2 <= re) {
            pass(std::integral_constant<int, 2>(), r);
            r += 2;
        }
        if (r < re) pass(std::integral_constant<int, 1>(), r);
#pragma unroll
        for (int t = 0; t < SG_KW; ++t)
#pragma unroll
            for (int k = 0; k < 2; ++k) a[t][k] = an[t][k];
        __syncthreads();
    }
    const char* last = buf[0];
    if (STORE) write_out(last, MODE == SG_BWD ? p.dz[0] : p.x[SG_LAYERS - 1]);
    if (MODE == SG_BWD) return;
    // ---- last layer: z[tap][s] into buffer 1, then the nine shifted sums
    float* z = reinterpret_cast<float*>(buf[1]);
    bf16x8 a5[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(p.w[SG_LAYERS - 1] + (size_t)min(i, SG_KW - 1) * SG_C + 32 * k + 8 * g);
        bf16x8 zero;
#pragma unroll
        for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;
        a5[k] = i < SG_KW ? v : zero;
    }
    for (int r = w; r < R; r += 8) {
        const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(last + r * 128 + omid);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(last + r * 128 + (omid ^ 64));
        f4 acc = f4{0.f, 0.f, 0.f, 0.f};
        acc = mfma_bf16(a5[0], b0, acc);
        acc = mfma_bf16(a5[1], b1, acc);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (4 * g + v < SG_KW) z[(4 * g + v) * CH_WMAX + r + R * i] = acc[v];
    }
    __syncthreads();
    const float b5 = MODE == SG_FWD ? p.bias[SG_LAYERS - 1][0] : 0.0f;
    for (int t = tid; t < min(T, N - n0); t += 512) {
        float qv = b5;
#pragma unroll
        for (int tap = 0; tap < SG_KW; ++tap) qv += z[tap * CH_WMAX + CH_HALO + t + tap - SG_HALO];
        const size_t o = base + n0 + t;
        if (p.q) p.q[o] = qv;
        if (p.Q) p.Q[o] = p.mean + p.scale * (double)qv;
    }
}

// Tile length: the one that keeps the CUs (one workgroup each) busy with the
// fewest rows in all, rounds of workgroups x rows per wavefront.
static void chain_tile(int N, int B, int* T, int* R)
{
    const int cus = 256;
    long long best = -1;
    for (int tiles = 1; tiles <= (N + 15) / 16; ++tiles) {
        // (a shift of four sites must stay within one row of the next lane: r >= 4)
        const int t = (N + tiles - 1) / tiles, r = std::max(4, (t + 2 * CH_HALO + 15) / 16);
        if (r > CH_RMAX) continue;
        const long long rounds = ((long long)tiles * B + cus - 1) / cus;
        const long long cost = rounds * ((r + 1) / 2 + 3);  // 3: the fixed part of a workgroup, in rows
        if (best < 0 || cost < best) {
            best = cost;
            *T = t;
            *R = r;
        }
    }
}

// ---- parameter gradients of all layers in one launch
//   dW_l[co][tap][ci] = sum_s dZ_l[s][co] X_l[s + tap - 4][ci],  db_l[co] = sum_s dZ_l[s][co]
// (s over the sites of all samples, X = 0 outside a sample) as MFMA GEMMs with
// M = co, N = ci, K = sites.  K runs over channels-fastest arrays, so an
// operand fragment needs eight sites of one channel: a thread loads 8 sites x
// 8 channels (eight 16-byte loads) and transposes them with v_perm_b32, half
// an instruction per value.  A chunk of 256 sites is kept in LDS as 32 rows
// with element e of row r the site r + 32 e: the tap shift s + tap - 4 is then
// another row, never another element, so every fragment is one aligned
// 16-byte read and the rows of tap 4..8 are those of tap 0..4 four rows on
// (one K step of 32 sites), held in registers: 45 reads feed 72 MFMAs.
// Jobs (blockIdx.y): 4 hidden layers x 4 tiles of 16 input channels (wavefront
// w: output channels 16 w..16 w + 15, nine taps), then the first layer (3 real
// inputs x 9 taps as the 27 columns of two tiles) and the last (9 taps as the
// rows, one output channel).  Each workgroup walks a run of chunks and writes
// one partial copy; sg_wreduce_kernel sums the copies in order.
// At 32 x 2048 sites all six layers take 37 us (MFMA time 9 us; the rest is
// the global loads and transposes of each chunk, three workgroups per CU
// covering for each other) and the sum of the copies 7 us.  One launch per
// layer with 2-byte transposing loads and a serial bias sum took 4.7 ms.
constexpr int WG_R = 32;                 // rows of a chunk
constexpr int WG_SITES = 8 * WG_R;       // sites of a chunk
constexpr int WG_XR = WG_R + 2 * SG_HALO;
constexpr int WG_JOBS = 4 * (SG_LAYERS - 2) + 2;
constexpr int WG_GROUPS = 42;            // partial copies at most: 18 jobs x 42 workgroups fill 256 CUs three deep

typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

struct SgWgradArgs {
    const __bf16* dz[SG_LAYERS];  // gradient at layer l's output [site][64], l < 5
    const __bf16* x[SG_LAYERS];   // hidden layer l's input [site][64]
    const __bf16* dq;             // gradient at the output [site]
    const double* U;              // the potentials and features of the first layer's inputs
    const double* feat;
    int woff[SG_LAYERS], boff[SG_LAYERS];
    int N, cps, nchunks, per;     // sites and chunks per sample, chunks, chunks per workgroup
    int nparam;
    float* P;                     // [copy][nparam]
};

// eight channels of the eight sites n + 32 e of one sample (zero outside it)
__device__ __forceinline__ void wg_load(const __bf16* __restrict__ src, int C, int n, int N, u32x4 (&v)[8])
{
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int m = n + WG_R * e;
        v[e] = *reinterpret_cast<const u32x4*>(src + (size_t)min(max(m, 0), N - 1) * C);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int m = n + WG_R * e;
        if (m < 0 || m >= N) v[e] = u32x4{0u, 0u, 0u, 0u};
    }
}

// transposed: channel c of the eight at row[(c ^ swz) * 8], its eight sites together
__device__ __forceinline__ void wg_store(const u32x4 (&v)[8], __bf16* row, int swz)
{
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        u32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            o[q] = __builtin_amdgcn_perm(v[2 * q + 1][c >> 1], v[2 * q][c >> 1], c & 1 ? 0x07060302u : 0x05040100u);
        *reinterpret_cast<u32x4*>(row + (c ^ swz) * 8) = o;
    }
}

__global__ __launch_bounds__(256, 3) void sg_wgrad_kernel(SgWgradArgs a)
{
    __shared__ __attribute__((aligned(16))) __bf16 wide[WG_R * SG_C * 8];      // 64 channels, no halo
    __shared__ __attribute__((aligned(16))) __bf16 halo[WG_XR * 16 * 8];       // 16 channels or 3 planes, with halo
    const int job = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int c0 = blockIdx.x * a.per, c1 = min(a.nchunks, c0 + a.per);
    if (c0 >= c1) return;  // (the grid is rounded up: see the launch)
    const int N = a.N;
    float* P = a.P + (size_t)blockIdx.x * a.nparam;
    // wide tile: thread = (row tid / 8, channel octet tid % 8); the octet's number
    // is mixed into the position inside it, so that 8 threads write 8 bank groups
    const int wr = tid >> 3, wo = tid & 7;
    __bf16* wdst = wide + (wr * SG_C + wo * 8) * 8;
    const int wcol = 16 * w + i;                              // this lane's channel of the wide tile
    const __bf16* wsrc = wide + (g * SG_C + (wcol & ~7) + ((wcol & 7) ^ (wcol >> 3))) * 8;
    __attribute__((aligned(16))) __bf16 one8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) one8[e] = (__bf16)1.0f;
    const bf16x8 ones = *reinterpret_cast<const bf16x8*>(one8);

    if (job < WG_JOBS - 2) {
        const int l = 1 + (job >> 2), tile = job & 3;
        const __bf16* dz = a.dz[l];
        const __bf16* x = a.x[l] + tile * 16;
        // halo tile: thread < 80 = (row tid / 2, octet tid % 2)
        const int hr = tid >> 1, ho = tid & 1;
        const bool hx = tid < 2 * WG_XR;
        u32x4 vw[8];
        auto load = [&](int c) {
            const int b = c / a.cps, n0 = (c - b * a.cps) * WG_SITES;
            wg_load(dz + (size_t)b * N * SG_C + wo * 8, SG_C, n0 + wr, N, vw);
        };
        f4 acc[SG_KW], accb = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < SG_KW; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
        if (c0 < c1) load(c0);
        for (int c = c0; c < c1; ++c) {
            wg_store(vw, wdst, wo);
            if (hx) {
                const int b = c / a.cps, n0 = (c - b * a.cps) * WG_SITES;
                u32x4 vh[8];
                wg_load(x + (size_t)b * N * SG_C + ho * 8, SG_C, n0 + hr - SG_HALO, N, vh);
                wg_store(vh, halo + (hr * 16 + ho * 8) * 8, hr & 7);
            }
            __syncthreads();
            if (c + 1 < c1) load(c + 1);
            // fragment rho: row rho + g of the halo tile (tap t of step st: rho = 4 st + t)
            auto frag = [&](int rho) {
                const int row = rho + g;
                return *reinterpret_cast<const bf16x8*>(halo + (row * 16 + (i ^ (row & 7))) * 8);
            };
            bf16x8 win[SG_KW];
#pragma unroll
            for (int t = 0; t < 5; ++t) win[t] = frag(t);
#pragma unroll
            for (int st = 0; st < WG_R / 4; ++st) {
#pragma unroll
                for (int t = 5; t < SG_KW; ++t) win[t] = frag(4 * st + t);
                const bf16x8 av = *reinterpret_cast<const bf16x8*>(wsrc + 4 * st * SG_C * 8);
#pragma unroll
                for (int t = 0; t < SG_KW; ++t) acc[t] = mfma_bf16(av, win[t], acc[t]);
                if (tile == 0) accb = mfma_bf16(av, ones, accb);
#pragma unroll
                for (int t = 0; t < 5; ++t) win[t] = win[t + 4];
            }
            __syncthreads();
        }
        float* Pw = P + a.woff[l];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int co = 16 * w + 4 * g + v;
#pragma unroll
            for (int t = 0; t < SG_KW; ++t) Pw[(co * SG_KW + t) * SG_C + tile * 16 + i] = acc[t][v];
            if (tile == 0 && i == 0) P[a.boff[l] + co] = accb[v];
        }
        return;
    }
    // first and last layer: one tile of 64 channels without halo, and planes of
    // single channels with halo (3 inputs, or the one output gradient)
    const bool first = job == WG_JOBS - 2;
    const int l = first ? 0 : SG_LAYERS - 1;
    const __bf16* wsr = first ? a.dz[0] : a.x[SG_LAYERS - 1];
    const int np = first ? SG_IN : 1;
    u32x4 vw[8];
    f4 acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}}, accb = acc[0];
    // first layer: this lane's columns (input, tap) of the two tiles; last: its row (tap)
    int prow[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int col = min(16 * t + i, SG_IN * SG_KW - 1);
        prow[t] = first ? col / SG_KW * WG_XR + col % SG_KW : 2 * SG_HALO - min(i, SG_KW - 1);
    }
    for (int c = c0; c < c1; ++c) {
        const int b = c / a.cps, n0 = (c - b * a.cps) * WG_SITES;
        wg_load(wsr + (size_t)b * N * SG_C + wo * 8, SG_C, n0 + wr, N, vw);
        wg_store(vw, wdst, wo);
        for (int q = tid; q < np * WG_XR * 8; q += 256) {
            const int p = q / (WG_XR * 8), r = q - p * WG_XR * 8, row = r >> 3, e = r & 7;
            const int n = n0 + row - SG_HALO + WG_R * e;
            const int nc = min(max(n, 0), N - 1);
            __bf16 v;
            if (!first)
                v = a.dq[(size_t)b * N + nc];
            else if (p == 0)
                v = (__bf16)(float)(a.U[(size_t)b * N + nc] * 2.0);
            else if (p == 1)
                v = (__bf16)expf(-(float)min(nc, N - 1 - nc) * 0.0625f);
            else
                v = (__bf16)(float)(a.feat ? a.feat[b] : 0.0);
            halo[q] = n >= 0 && n < N ? v : (__bf16)0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int st = 0; st < WG_R / 4; ++st) {
            const bf16x8 wv = *reinterpret_cast<const bf16x8*>(wsrc + 4 * st * SG_C * 8);
            const bf16x8 p0 = *reinterpret_cast<const bf16x8*>(halo + (prow[0] + 4 * st + g) * 8);
            if (first) {
                const bf16x8 p1 = *reinterpret_cast<const bf16x8*>(halo + (prow[1] + 4 * st + g) * 8);
                acc[0] = mfma_bf16(wv, p0, acc[0]);
                acc[1] = mfma_bf16(wv, p1, acc[1]);
                accb = mfma_bf16(wv, ones, accb);
            } else {
                acc[0] = mfma_bf16(p0, wv, acc[0]);
                accb = mfma_bf16(p0, ones, accb);
            }
        }
        __syncthreads();
    }
    float* Pw = P + a.woff[l];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int m = 4 * g + v;
        if (first) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int col = 16 * t + i;
                if (col < SG_IN * SG_KW) Pw[((16 * w + m) * SG_KW + col % SG_KW) * SG_CP + col / SG_KW] = acc[t][v];
            }
            if (i == 0) P[a.boff[0] + 16 * w + m] = accb[v];
        } else {
            if (m < SG_KW) Pw[m * SG_C + 16 * w + i] = acc[0][v];
            if (w == 0 && i == 0 && m == SG_HALO) P[a.boff[l]] = accb[v];  // tap 4: the sum of dq itself
        }
    }
}

// out[j] = sum_k P[k][j] in copy order; entries of padding channels are 0.
__global__ __launch_bounds__(256) void sg_wreduce_kernel(int ncopies, SgWgradArgs a, float* __restrict__ out)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= a.nparam) return;
    const int r5 = j - a.woff[SG_LAYERS - 1], b5 = j - a.boff[SG_LAYERS - 1];
    const bool pad = (j < a.boff[0] && j % SG_CP >= SG_IN) || (r5 >= SG_KW * SG_C && b5 < 0) || b5 > 0;
    float s = 0.f;
    if (!pad) {
#pragma unroll 8
        for (int k = 0; k < ncopies; ++k) s += a.P[(size_t)k * a.nparam + j];
    }
    out[j] = s;
}

__global__ void sg_output_kernel(long long n, const float* __restrict__ q, double mean, double scale,
                                 double* __restrict__ Q)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) Q[i] = mean + scale * (double)q[i];
}

// Mean squared error of the normalised output; dq = 2 (q - t) / n; one partial
// sum per block.
__global__ __launch_bounds__(256) void sg_loss_kernel(long long n, const float* __restrict__ q,
                                                      const double* __restrict__ Qt, double mean, double inv_scale,
                                                      __bf16* __restrict__ dq, float* __restrict__ part)
{
    __shared__ float red[256];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (i < n) {
        const float t = (float)((Qt[i] - mean) * inv_scale);
        const float d = q[i] - t;
        l = d * d;
        dq[i] = (__bf16)(2.0f * d / (float)n);
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void sg_adam_kernel(int n, float* __restrict__ w, const float* __restrict__ gr, float* __restrict__ m,
                               float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const float gj = gr[j];
    const float mj = b1 * m[j] + (1.f - b1) * gj;
    const float vj = b2 * v[j] + (1.f - b2) * gj * gj;
    m[j] = mj;
    v[j] = vj;
    w[j] -= lr * (mj / c1) / (sqrtf(vj / c2) + eps);
}

// FP32 masters W [COUT][9][CIN] -> bf16 Wb (same layout, padding rows and
// columns forced to zero) and Wt [CIN][9][COUT] = W[co][8 - tap][ci].
__global__ void sg_pack_kernel(int cin, int cout, int cin_real, int cout_real, const float* __restrict__ W,
                               __bf16* __restrict__ Wb, __bf16* __restrict__ Wt)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= cin * cout * SG_KW) return;
    const int co = j / (SG_KW * cin);
    const int r = j - co * SG_KW * cin;
    const int tap = r / cin, ci = r - tap * cin;
    const float x = (co < cout_real && ci < cin_real) ? W[j] : 0.f;
    Wb[j] = (__bf16)x;
    Wt[((size_t)ci * SG_KW + (SG_KW - 1 - tap)) * cout + co] = (__bf16)x;
}

__global__ void sg_gather_kernel(int N, int B, const int* __restrict__ idx, const double* __restrict__ U,
                                 const double* __restrict__ Q, const double* __restrict__ F, double* __restrict__ bU,
                                 double* __restrict__ bQ, double* __restrict__ bF)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)N * B) return;
    const int b = (int)(q / N), n = (int)(q - (long long)b * N);
    const size_t src = (size_t)idx[b] * N + n;
    bU[q] = U[src];
    bQ[q] = Q[src];
    if (n == 0) bF[b] = F ? F[idx[b]] : 0.0;
}

static int real_cin(int l) { return l == 0 ? SG_IN : SG_C; }
static int real_cout(int l) { return l == SG_LAYERS - 1 ? 1 : SG_C; }

Surrogate::~Surrogate()
{
    if (st) {
        (void)hipStreamSynchronize(st);
        (void)hipStreamDestroy(st);
    }
}

int Surrogate::init(int N_, unsigned long long seed)
{
    N = N_;
    int off = 0;
    for (int l = 0; l < SG_LAYERS; ++l) {
        woff.push_back(off);
        off += sg_cout(l) * SG_KW * sg_cin(l);
        boff.push_back(off);
        off += sg_cout(l);
    }
    nparam = off;
    // uniform initialisation with variance 1 / fan-in (real channels only)
    std::vector<float> w(nparam, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < SG_LAYERS; ++l) {
        const float lim = std::sqrt(3.0f / (float)(real_cin(l) * SG_KW));
        std::uniform_real_distribution<float> dist(-lim, lim);
        for (int co = 0; co < real_cout(l); ++co)
            for (int tap = 0; tap < SG_KW; ++tap)
                for (int ci = 0; ci < real_cin(l); ++ci)
                    w[woff[l] + ((size_t)co * SG_KW + tap) * sg_cin(l) + ci] = dist(rng);
    }
    int rc;
    NEGF_HIP_TRY(hipStreamCreate(&st));
    for (DevBuf* b : {&d_w, &d_m, &d_v, &d_g})
        if ((rc = b->ensure(sizeof(float) * nparam))) return rc;
    if ((rc = d_wb.ensure(2 * (size_t)nparam))) return rc;
    if ((rc = d_wt.ensure(2 * (size_t)nparam))) return rc;
    std::vector<float> z(nparam, 0.f);
    NEGF_HIP_TRY(hipMemcpy(d_w.p, w.data(), sizeof(float) * nparam, hipMemcpyHostToDevice));
    NEGF_HIP_TRY(hipMemcpy(d_m.p, z.data(), sizeof(float) * nparam, hipMemcpyHostToDevice));
    NEGF_HIP_TRY(hipMemcpy(d_v.p, z.data(), sizeof(float) * nparam, hipMemcpyHostToDevice));
    NEGF_HIP_TRY(hipMemcpy(d_g.p, z.data(), sizeof(float) * nparam, hipMemcpyHostToDevice));
    if ((rc = pack(st))) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(st));
    return NEGF_OK;
}

int Surrogate::pack(hipStream_t s)
{
    for (int l = 0; l < SG_LAYERS; ++l) {
        const int cin = sg_cin(l), cout = sg_cout(l);
        const int n = cin * cout * SG_KW;
        hipLaunchKernelGGL(sg_pack_kernel, dim3((n + 255) / 256), dim3(256), 0, s, cin, cout, real_cin(l),
                           real_cout(l), d_w.as<float>() + woff[l], d_wb.as<__bf16>() + woff[l],
                           d_wt.as<__bf16>() + woff[l]);
    }
    NEGF_HIP_TRY(hipGetLastError());
    return NEGF_OK;
}

int Surrogate::ensure_batch(int B)
{
    if (B <= capB) return NEGF_OK;
    int rc;
    const size_t sites = (size_t)B * N;
    for (int l = 1; l < SG_LAYERS; ++l)
        if ((rc = d_act[l].ensure(2 * sites * SG_C))) return rc;
    if ((rc = d_act[SG_LAYERS].ensure(sizeof(float) * sites))) return rc;
    capB = B;
    return NEGF_OK;
}

template <int MODE, bool STORE>
static int chain(SgChainArgs& p, int N, int B, hipStream_t s)
{
    p.N = N;
    chain_tile(N, B, &p.T, &p.R);
    // samples along y, at most 65535 at a time
    for (int b0 = 0; b0 < B; b0 += 65535) {
        SgChainArgs q = p;
        const size_t o = (size_t)b0 * N;
        if (q.in) q.in += o;
        if (q.feat) q.feat += b0;
        if (q.dq) q.dq += o;
        if (q.q) q.q += o;
        if (q.Q) q.Q += o;
        for (int l = 0; l < SG_LAYERS; ++l) {
            if (q.x[l]) q.x[l] += o * SG_C;
            if (q.dz[l]) q.dz[l] += o * SG_C;
        }
        hipLaunchKernelGGL((sg_chain_kernel<MODE, STORE>), dim3((N + p.T - 1) / p.T, std::min(B - b0, 65535)), dim3(512),
                           0, s, q);
    }
    NEGF_HIP_TRY(hipGetLastError());
    return NEGF_OK;
}

// arguments common to the passes: weights of the layers in the order of the steps
static SgChainArgs chain_args(Surrogate& g, bool backward)
{
    SgChainArgs p;
    std::memset(&p, 0, sizeof(p));
    for (int st = 0; st < SG_LAYERS; ++st) {
        const int l = backward ? SG_LAYERS - 1 - st : st;
        p.w[st] = (backward ? g.d_wt : g.d_wb).as<__bf16>() + g.woff[l];
        p.bias[st] = g.d_w.as<float>() + g.boff[l];
    }
    return p;
}

int Surrogate::forward(int B, const double* dU, const double* dfeat, hipStream_t s)
{
    int rc;
    if ((rc = ensure_batch(B))) return rc;
    SgChainArgs p = chain_args(*this, false);
    p.in = dU;
    p.feat = dfeat;
    for (int l = 1; l < SG_LAYERS; ++l) p.x[l] = d_act[l].as<__bf16>();
    p.q = d_act[SG_LAYERS].as<float>();
    return chain<SG_FWD, true>(p, N, B, s);
}

// The pass's output as doubles.  A tile reads its neighbours' inputs, so an
// output that overlaps the inputs goes through the float buffer.
template <int MODE>
int Surrogate::chain_to(SgChainArgs& p, int B, double mean, double* dQ, hipStream_t s)
{
    const long long n = (long long)B * N;
    const double* lo = dQ;
    const double* hi = dQ + n;
    const bool overlap = (p.in < hi && lo < p.in + n) || (p.feat && p.feat < hi && lo < p.feat + B);
    p.mean = mean;
    p.scale = scale_Q;
    if (!overlap) {
        p.Q = dQ;
        return chain<MODE, false>(p, N, B, s);
    }
    int rc;
    if ((rc = d_act[SG_LAYERS].ensure(sizeof(float) * (size_t)n))) return rc;
    p.q = d_act[SG_LAYERS].as<float>();
    if ((rc = chain<MODE, false>(p, N, B, s))) return rc;
    hipLaunchKernelGGL(sg_output_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, p.q, mean, scale_Q, dQ);
    NEGF_HIP_TRY(hipGetLastError());
    return NEGF_OK;
}

int Surrogate::evaluate(int B, const double* dU, const double* dfeat, double* dQ, hipStream_t s)
{
    SgChainArgs p = chain_args(*this, false);
    p.in = dU;
    p.feat = dfeat;
    return chain_to<SG_FWD>(p, B, mean_Q, dQ, s);
}

// forward-mode tangent: t_{l+1} = conv(W_l, t_l) (1 - x_{l+1}^2), dq = conv(W_5, t_5)
int Surrogate::jvp(int B, const double* dV, double* dout, hipStream_t s)
{
    if (B > capB) {
        set_error("surrogate tangent needs a forward of at least %d samples first", B);
        return NEGF_EARG;
    }
    SgChainArgs p = chain_args(*this, false);
    p.in = dV;
    for (int l = 1; l < SG_LAYERS; ++l) p.x[l] = d_act[l].as<__bf16>();
    return chain_to<SG_TAN>(p, B, 0.0, dout, s);
}

int Surrogate::backward(int B, const double* dU, const double* dfeat, const double* dQt, double* loss, hipStream_t s)
{
    int rc;
    const long long sites = (long long)B * N;
    const int lblocks = (int)((sites + 255) / 256);
    if ((rc = d_loss.ensure(sizeof(float) * lblocks))) return rc;
    for (int l = 0; l < SG_LAYERS; ++l)
        if ((rc = d_dz[l].ensure(2 * (size_t)sites * (l == SG_LAYERS - 1 ? 1 : SG_C)))) return rc;
    __bf16* dq = d_dz[SG_LAYERS - 1].as<__bf16>();
    hipLaunchKernelGGL(sg_loss_kernel, dim3(lblocks), dim3(256), 0, s, sites, d_act[SG_LAYERS].as<float>(), dQt,
                       mean_Q, 1.0 / scale_Q, dq, d_loss.as<float>());
    // data gradients of layers 5..1, kept for the one launch that forms all weight gradients
    SgChainArgs p = chain_args(*this, true);
    p.dq = dq;
    for (int l = 1; l < SG_LAYERS; ++l) p.x[l] = d_act[l].as<__bf16>();
    for (int l = 0; l < SG_LAYERS - 1; ++l) p.dz[l] = d_dz[l].as<__bf16>();
    if ((rc = chain<SG_BWD, true>(p, N, B, s))) return rc;
    SgWgradArgs a;
    for (int l = 0; l < SG_LAYERS; ++l) {
        a.dz[l] = l < SG_LAYERS - 1 ? d_dz[l].as<__bf16>() : nullptr;
        a.x[l] = l > 0 ? d_act[l].as<__bf16>() : nullptr;
        a.woff[l] = woff[l];
        a.boff[l] = boff[l];
    }
    a.dq = dq;
    a.U = dU;
    a.feat = dfeat;
    a.N = N;
    a.cps = (N + WG_SITES - 1) / WG_SITES;
    a.nchunks = B * a.cps;
    a.per = (a.nchunks + WG_GROUPS - 1) / WG_GROUPS;
    a.nparam = nparam;
    const int copies = (a.nchunks + a.per - 1) / a.per;
    if ((rc = d_part.ensure(sizeof(float) * (size_t)copies * nparam))) return rc;
    a.P = d_part.as<float>();
    // Workgroups go to the eight XCDs in turn: with a multiple of eight runs, the
    // jobs of one run share an XCD and find each other's chunks in its L2
    // (37 against 48 us at 32 x 2048 sites).
    hipLaunchKernelGGL(sg_wgrad_kernel, dim3((copies + 7) / 8 * 8, WG_JOBS), dim3(256), 0, s, a);
    hipLaunchKernelGGL(sg_wreduce_kernel, dim3((nparam + 255) / 256), dim3(256), 0, s, copies, a, d_g.as<float>());
    NEGF_HIP_TRY(hipGetLastError());
    if (loss) {
        std::vector<float> h(lblocks);
        NEGF_HIP_TRY(hipMemcpyAsync(h.data(), d_loss.p, sizeof(float) * lblocks, hipMemcpyDeviceToHost, s));
        NEGF_HIP_TRY(hipStreamSynchronize(s));
        double a = 0.0;
        for (float v : h) a += v;
        *loss = a / (double)sites;
    }
    return NEGF_OK;
}

int Surrogate::adam(float lr, hipStream_t s)
{
    ++adam_t;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)adam_t), c2 = 1.f - std::pow(b2, (float)adam_t);
    hipLaunchKernelGGL(sg_adam_kernel, dim3((nparam + 255) / 256), dim3(256), 0, s, nparam, d_w.as<float>(),
                       d_g.as<float>(), d_m.as<float>(), d_v.as<float>(), lr, b1, b2, 1e-8f, c1, c2);
    NEGF_HIP_TRY(hipGetLastError());
    return pack(s);
}

}  // namespace negf

using namespace negf;

extern "C" {

int negf_surrogate_create(int N, unsigned long long seed, negf_surrogate** out)
{
    clear_error();
    if (N < 16 || N > NEGF_MAX_SITES || !out) {
        set_error("invalid surrogate arguments (N = %d)", N);
        return NEGF_EARG;
    }
    negf_surrogate* h = new negf_surrogate;
    const int rc = h->s.init(N, seed);
    if (rc) {
        delete h;
        return rc;
    }
    *out = h;
    return NEGF_OK;
}

int negf_surrogate_destroy(negf_surrogate* s)
{
    if (!s) return NEGF_EARG;
    delete s;
    return NEGF_OK;
}

int negf_surrogate_num_params(const negf_surrogate* s) { return s ? s->s.nparam : -1; }

int negf_surrogate_num_sites(const negf_surrogate* s) { return s ? s->s.N : -1; }

int negf_surrogate_get_params(negf_surrogate* s, float* w, double* norm)
{
    clear_error();
    if (!s) {
        set_error("null surrogate");
        return NEGF_EARG;
    }
    NEGF_HIP_TRY(hipStreamSynchronize(s->s.st));
    if (w) NEGF_HIP_TRY(hipMemcpy(w, s->s.d_w.p, sizeof(float) * s->s.nparam, hipMemcpyDeviceToHost));
    if (norm) {
        norm[0] = s->s.mean_Q;
        norm[1] = s->s.scale_Q;
    }
    return NEGF_OK;
}

int negf_surrogate_set_params(negf_surrogate* s, const float* w, const double* norm)
{
    clear_error();
    if (!s) {
        set_error("null surrogate");
        return NEGF_EARG;
    }
    if (norm && !(norm[1] > 0.0)) {
        set_error("surrogate output scale must be positive");
        return NEGF_EARG;
    }
    NEGF_HIP_TRY(hipStreamSynchronize(s->s.st));
    if (w) NEGF_HIP_TRY(hipMemcpy(s->s.d_w.p, w, sizeof(float) * s->s.nparam, hipMemcpyHostToDevice));
    if (norm) {
        s->s.mean_Q = norm[0];
        s->s.scale_Q = norm[1];
    }
    const int rc = s->s.pack(s->s.st);
    if (rc) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(s->s.st));
    return NEGF_OK;
}

int negf_surrogate_forward(negf_surrogate* s, int B, const double* d_U, const double* d_feat, double* d_Q,
                           void* stream)
{
    clear_error();
    if (!s || B <= 0 || !d_U || !d_Q) {
        set_error("invalid surrogate forward arguments");
        return NEGF_EARG;
    }
    hipStream_t st = stream ? (hipStream_t)stream : s->s.st;
    return s->s.evaluate(B, d_U, d_feat, d_Q, st);
}

int negf_surrogate_jvp(negf_surrogate* s, int B, const double* d_U, const double* d_feat, const double* d_V,
                       double* d_out, void* stream)
{
    clear_error();
    if (!s || B <= 0 || !d_U || !d_V || !d_out) {
        set_error("invalid surrogate tangent arguments");
        return NEGF_EARG;
    }
    hipStream_t st = stream ? (hipStream_t)stream : s->s.st;
    int rc = s->s.forward(B, d_U, d_feat, st);
    if (!rc) rc = s->s.jvp(B, d_V, d_out, st);
    return rc;
}

int negf_surrogate_gradient(negf_surrogate* s, int B, const double* d_U, const double* d_feat, const double* d_Q,
                            float* grad, double* loss)
{
    clear_error();
    if (!s || B <= 0 || !d_U || !d_Q) {
        set_error("invalid surrogate gradient arguments");
        return NEGF_EARG;
    }
    int rc = s->s.forward(B, d_U, d_feat, s->s.st);
    if (!rc) rc = s->s.backward(B, d_U, d_feat, d_Q, loss, s->s.st);
    if (rc) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(s->s.st));
    if (grad) NEGF_HIP_TRY(hipMemcpy(grad, s->s.d_g.p, sizeof(float) * s->s.nparam, hipMemcpyDeviceToHost));
    return NEGF_OK;
}

int negf_surrogate_fit_output_scale(negf_surrogate* s, int nsamples, const double* d_Q)
{
    clear_error();
    if (!s || nsamples <= 0 || !d_Q) {
        set_error("invalid surrogate scale arguments");
        return NEGF_EARG;
    }
    std::vector<double> h((size_t)nsamples * s->s.N);
    NEGF_HIP_TRY(hipMemcpy(h.data(), d_Q, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
    double a = 0.0;
    for (double v : h) a += v;
    const double mean = a / (double)h.size();
    double q = 0.0;
    for (double v : h) q += (v - mean) * (v - mean);
    s->s.mean_Q = mean;
    s->s.scale_Q = std::sqrt(q / (double)h.size());
    if (!(s->s.scale_Q > 0.0)) s->s.scale_Q = 1.0;
    return NEGF_OK;
}

// Adam on minibatches of nsamples device pairs (U, Q) (double [S][N]) with
// optional per-sample features (double [S]); seeded shuffle per epoch;
// learning rate linear from lr to lr_end.
int negf_surrogate_train(negf_surrogate* s, int nsamples, const double* d_U, const double* d_feat, const double* d_Q,
                         int epochs, int batch, double lr, double lr_end, unsigned long long seed, double* last_loss)
{
    clear_error();
    if (!s || nsamples <= 0 || !d_U || !d_Q || epochs <= 0 || batch <= 0 || batch > nsamples) {
        set_error("invalid surrogate training arguments");
        return NEGF_EARG;
    }
    Surrogate& m = s->s;
    const int N = m.N;
    int rc;
    if ((rc = m.d_bU.ensure(sizeof(double) * (size_t)batch * N))) return rc;
    if ((rc = m.d_bQ.ensure(sizeof(double) * (size_t)batch * N))) return rc;
    if ((rc = m.d_bF.ensure(sizeof(double) * (size_t)batch))) return rc;
    const int steps_per_epoch = nsamples / batch;
    if ((rc = m.d_idx.ensure(sizeof(int) * (size_t)steps_per_epoch * batch))) return rc;
    std::vector<int> order(nsamples);
    for (int i = 0; i < nsamples; ++i) order[i] = i;
    std::mt19937_64 rng(seed);
    const long long total_steps = (long long)steps_per_epoch * epochs;
    long long step = 0;
    double l = 0.0;
    const long long bs = (long long)batch * N;
    for (int ep = 0; ep < epochs; ++ep) {
        std::shuffle(order.begin(), order.end(), rng);
        NEGF_HIP_TRY(hipMemcpyAsync(m.d_idx.p, order.data(), sizeof(int) * (size_t)steps_per_epoch * batch,
                                    hipMemcpyHostToDevice, m.st));
        for (int k = 0; k < steps_per_epoch; ++k) {
            hipLaunchKernelGGL(sg_gather_kernel, dim3((unsigned)((bs + 255) / 256)), dim3(256), 0, m.st, N, batch,
                               m.d_idx.as<int>() + (size_t)k * batch, d_U, d_Q, d_feat, m.d_bU.as<double>(),
                               m.d_bQ.as<double>(), m.d_bF.as<double>());
            NEGF_HIP_TRY(hipGetLastError());
            const double* bF = d_feat ? m.d_bF.as<double>() : nullptr;
            if ((rc = m.forward(batch, m.d_bU.as<double>(), bF, m.st))) return rc;
            const bool want = (k == steps_per_epoch - 1) && last_loss;
            if ((rc = m.backward(batch, m.d_bU.as<double>(), bF, m.d_bQ.as<double>(), want ? &l : nullptr, m.st)))
                return rc;
            const double frac = total_steps > 1 ? (double)step / (double)(total_steps - 1) : 1.0;
            if ((rc = m.adam((float)(lr + (lr_end - lr) * frac), m.st))) return rc;
            ++step;
        }
        // the shuffled order is read by the gathers just queued
        NEGF_HIP_TRY(hipStreamSynchronize(m.st));
        if (last_loss) *last_loss = l;
    }
    NEGF_HIP_TRY(hipStreamSynchronize(m.st));
    return NEGF_OK;
}

}  // extern "C"
