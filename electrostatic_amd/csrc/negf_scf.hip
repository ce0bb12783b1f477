// negf_scf.hip -- Broyden modified-second update on the device and the
// self-consistent loop of one tube with a dense electrostatic stand-in.
//
// Broyden (Execute_Broyden_Modified_Second_Algorithm_Parallel
// Broyden_Second_Parallel.cpp:213-486, serial order :9-211): one workgroup of
// 1024 threads runs a whole update.  Every reduction has a fixed order
// (lane-strided partial sums, a fixed butterfly per wavefront, waves summed
// in index order), so results are identical from run to run.  The history
// dot products of one update are spread over the 16 wavefronts, one history
// column per wavefront at a time, so an update costs two block barriers per
// phase rather than two per history column.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "negf_internal.h"
#include "negf_material.h"
#include "surrogate.h"

namespace negf {

static constexpr int kBroydenThreads = 1024;
static constexpr int kWaves = kBroydenThreads / 64;

struct BroydenDev {
    double* n_in;
    double* n_prev;
    double* F;
    double* dF;
    double* Norm;
    double* sum_vec;
    double* V;          // [max_step + 1][S]: dF / |dF|^2 per update
    double* W;          // [max_step + 1][S]
    double* intermed;   // [max_step + 1] history dots V_it . dF past the LDS copy
    double* intermed2;  // [max_step + 1] history dots V_it . F past the LDS copy
    double* out;        // [0] max norm, [1] l2 norm, [2] |dF|^2
    double* PFp;        // previous preconditioned residual (preconditioned update only)
};

// Lane exchanges of the wavefront reductions: lane ^ 32 and ^ 16 by permlane swaps,
// ^ 8 and ^ 4 within a row of 16 by rotations (row_ror:8 is lane ^ 8; row_ror:4 reads
// lane - 4, which equals lane ^ 4's value once the values repeat every 8 lanes), ^ 2 and
// ^ 1 by quad permutations.  No LDS round trip, the same operands and order as a
// butterfly of ds_bpermute shuffles, hence the same bits.  A reduction takes
// about 110 instead of 700 cycles: broyden_scf_kernel of 400 sites 8.7 us against 9.3 us.
template <int D>
__device__ __forceinline__ double lane_xor(double v)
{
    if constexpr (D >= 16) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
        const bool up = (threadIdx.x & D) != 0;
        if constexpr (D == 32) {
            const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
            const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
            return __longlong_as_double(
                (long long)(((unsigned long long)(up ? h[0] : h[1]) << 32) | (up ? l[0] : l[1])));
        } else {
            const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
            const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
            return __longlong_as_double(
                (long long)(((unsigned long long)(up ? h[0] : h[1]) << 32) | (up ? l[0] : l[1])));
        }
    } else {
        constexpr int ctrl = D == 8 ? 0x128 : D == 4 ? 0x124 : D == 2 ? 0x4E : 0xB1;
        const long long b = __double_as_longlong(v);
        const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, ctrl, 0xF, 0xF, true);
        const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xF, 0xF, true);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
}

__device__ __forceinline__ double wave_sum(double v)
{
    v += lane_xor<32>(v);
    v += lane_xor<16>(v);
    v += lane_xor<8>(v);
    v += lane_xor<4>(v);
    v += lane_xor<2>(v);
    v += lane_xor<1>(v);
    return v;
}

__device__ __forceinline__ double wave_max(double v)
{
    v = fmax(v, lane_xor<32>(v));
    v = fmax(v, lane_xor<16>(v));
    v = fmax(v, lane_xor<8>(v));
    v = fmax(v, lane_xor<4>(v));
    v = fmax(v, lane_xor<2>(v));
    v = fmax(v, lane_xor<1>(v));
    return v;
}

// The history's dot products in one pass over V: a_it = V_it . dF and
// b_it = V_it . F for it in [1, m_hi], each summed lane-strided and then
// across the wavefront; wave w takes it = 1 + w, 1 + w + kWaves, ...  Entries
// below kHistLds go to LDS, the rest to intermed (a) and intermed2 (b).
static constexpr int kHistLds = 512;

__device__ void history_dots2(const BroydenDev& b, int S, int m_hi, int wave, int lane, double* ha, double* hb)
{
    for (int it = 1 + wave; it <= m_hi; it += kWaves) {
        const double* __restrict__ v = b.V + (size_t)it * S;
        double a = 0.0, c = 0.0;
#pragma unroll 4
        for (int s = lane; s < S; s += 64) {
            const double vs = v[s];
            a = fma(vs, b.dF[s], a);
            c = fma(vs, b.F[s], c);
        }
        a = wave_sum(a);
        c = wave_sum(c);
        if (lane == 0) {
            if (it < kHistLds) {
                ha[it] = a;
                hb[it] = c;
            } else {
                b.intermed[it] = a;
                b.intermed2[it] = c;
            }
        }
    }
}

// One Broyden update of one system by one workgroup of kBroydenThreads.
// PC: the mixing term fraction * F is replaced by a preconditioned residual
// PF = P F (P linear and fixed between history resets), and fraction * dF by
// PF - PF_previous; everything else is the reference update.
//
// The reference (Broyden_Parallel_General.cpp:106-170) forms
// sum_vec = sum_{it<=m} W_it (V_it . F) after appending V_m, W_m, which needs
// V_it . dF first (for W_m) and a second pass over V for V_it . F.  Both dot
// products of the old rows come from one pass here, and the new row's
// V_m . F is summed while V_m is written; the sums over it keep the
// reference's order (it = 1..m, the new row last).
template <bool PC>
__device__ void broyden_update(int S, int m, double fraction, int norm_type, const double* __restrict__ n_out,
                               const double* __restrict__ PF, const BroydenDev& b)
{
    __shared__ double red[3][kWaves];
    __shared__ double ha[kHistLds], hb[kHistLds];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;

    // norms and F, dF (:31-88)
    double nsum = 0.0, nmax = 0.0, den = 0.0;
    for (int s = tid; s < S; s += kBroydenThreads) {
        const double Fc = b.n_in[s] - n_out[s];
        double nrm;
        if (norm_type == 0) {
            nrm = fabs(Fc);
            nsum = fma(Fc, Fc, nsum);
        } else {
            nrm = fabs(Fc / (b.n_in[s] + n_out[s]));
            nsum = fma(nrm, nrm, nsum);
        }
        b.Norm[s] = nrm;
        nmax = fmax(nmax, nrm);
        const double d = Fc - b.F[s];
        b.dF[s] = d;
        b.F[s] = Fc;
        den = fma(d, d, den);
    }
    nsum = wave_sum(nsum);
    nmax = wave_max(nmax);
    den = wave_sum(den);
    if (lane == 0) {
        red[0][wave] = nsum;
        red[1][wave] = nmax;
        red[2][wave] = den;
    }
    __syncthreads();
    double norm_sum = 0.0, bnorm = 0.0, denom = 0.0;
    for (int w = 0; w < kWaves; ++w) {
        norm_sum += red[0][w];
        bnorm = fmax(bnorm, red[1][w]);
        denom += red[2][w];
    }
    if (tid == 0) {
        b.out[0] = bnorm;
        b.out[1] = sqrt(norm_sum);
        b.out[2] = denom;
    }

    double bm = 0.0;   // V_m . F
    if (m > 0) {
        history_dots2(b, S, m - 1, wave, lane, ha, hb);
        __syncthreads();
        // W_m = -fraction dF + (n_in - n_prev) - sum_{it<m} W_it (V_it . dF)
        // (:106-135); the same W_it loads give the old rows' part of sum_vec
        double vf = 0.0;
        for (int s = tid; s < S; s += kBroydenThreads) {
            double sa = 0.0, sb = 0.0;
            const int mL = min(m - 1, kHistLds - 1);
            int it = 1;
#pragma unroll 4
            for (; it <= mL; ++it) {
                const double w = b.W[(size_t)it * S + s];
                sa = fma(w, ha[it], sa);
                sb = fma(w, hb[it], sb);
            }
            for (; it <= m - 1; ++it) {
                const double w = b.W[(size_t)it * S + s];
                sa = fma(w, b.intermed[it], sa);
                sb = fma(w, b.intermed2[it], sb);
            }
            const double d = b.dF[s];
            const double pd = PC ? PF[s] - b.PFp[s] : fraction * d;
            const double vm = d / denom;
            b.V[(size_t)m * S + s] = vm;
            b.W[(size_t)m * S + s] = -pd + (b.n_in[s] - b.n_prev[s]) - sa;
            b.sum_vec[s] = sb;
            vf = fma(vm, b.F[s], vf);
        }
        vf = wave_sum(vf);
        if (lane == 0) red[0][wave] = vf;
        __syncthreads();
        for (int w = 0; w < kWaves; ++w) bm += red[0][w];
    }
    // sum_vec (:137-170) and the new input (:172-186), scalar = 1
    for (int s = tid; s < S; s += kBroydenThreads) {
        const double prev = b.n_in[s];
        const double sv = m > 0 ? fma(b.W[(size_t)m * S + s], bm, b.sum_vec[s]) : 0.0;
        if (m > 0) b.sum_vec[s] = sv;
        const double pf = PC ? PF[s] : fraction * b.F[s];
        if (PC) b.PFp[s] = PF[s];
        b.n_prev[s] = prev;
        b.n_in[s] = prev - pf - sv;
    }
}

// broyden_update for at most kBroydenThreads sites, thread s holding site s (q: its
// n_out): the same sums in the same order, with the residual and its change in
// registers and LDS and the first history rows requested before anything is waited
// for.  One workgroup is bound by the latency of its loads, one history pass after the
// other: 1024 sites, 26 updates, 15.0 us on average against 16.9 us; 400 sites 8.0 us
// against 8.7 us.
template <bool PC>
__device__ void broyden_update_small(int S, int m, double fraction, int norm_type, double q,
                                     const double* __restrict__ PF, const BroydenDev& b)
{
    constexpr int VK = kBroydenThreads / 64, WK = 16;
    __shared__ double red[3][kWaves];
    __shared__ double ha[kHistLds], hb[kHistLds];
    __shared__ double sF[kBroydenThreads], sD[kBroydenThreads];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const bool on = tid < S;
    const int h = m - 1;  // history rows 1 .. h
    double v[VK], w[WK];
    auto load_v = [&](int it) {  // row it of V, lane-strided (it is wave-uniform)
#pragma unroll
        for (int k = 0; k < VK; ++k) v[k] = lane + 64 * k < S ? b.V[(size_t)it * S + lane + 64 * k] : 0.0;
    };
    const double nin = on ? b.n_in[tid] : 0.0, Fold = on ? b.F[tid] : 0.0, nprev = on ? b.n_prev[tid] : 0.0;
    if (1 + wave <= h) load_v(1 + wave);
#pragma unroll
    for (int k = 0; k < WK; ++k) w[k] = on && 1 + k <= h ? b.W[(size_t)(1 + k) * S + tid] : 0.0;

    // norms and F, dF
    const double Fc = on ? nin - q : 0.0, d = on ? Fc - Fold : 0.0;
    double nrm = 0.0, nsum = 0.0;
    if (on) {
        if (norm_type == 0) {
            nrm = fabs(Fc);
            nsum = fma(Fc, Fc, nsum);
        } else {
            nrm = fabs(Fc / (nin + q));
            nsum = fma(nrm, nrm, nsum);
        }
        b.Norm[tid] = nrm;
        b.dF[tid] = d;
        b.F[tid] = Fc;
    }
    sF[tid] = Fc;
    sD[tid] = d;
    nsum = wave_sum(nsum);
    const double nmax = wave_max(fmax(0.0, nrm)), den = wave_sum(d * d);
    if (lane == 0) {
        red[0][wave] = nsum;
        red[1][wave] = nmax;
        red[2][wave] = den;
    }
    __syncthreads();
    double norm_sum = 0.0, bnorm = 0.0, denom = 0.0;
    for (int k = 0; k < kWaves; ++k) {
        norm_sum += red[0][k];
        bnorm = fmax(bnorm, red[1][k]);
        denom += red[2][k];
    }
    if (tid == 0) {
        b.out[0] = bnorm;
        b.out[1] = sqrt(norm_sum);
        b.out[2] = denom;
    }

    double sv = 0.0;
    const double pf = !on ? 0.0 : PC ? PF[tid] : fraction * Fc;
    if (m > 0) {
        for (int it = 1 + wave; it <= h; it += kWaves) {
            double a = 0.0, c = 0.0;
#pragma unroll
            for (int k = 0; k < VK; ++k)
                if (64 * k < S) {  // uniform
                    a = fma(v[k], sD[lane + 64 * k], a);
                    c = fma(v[k], sF[lane + 64 * k], c);
                }
            if (it + kWaves <= h) load_v(it + kWaves);
            a = wave_sum(a);
            c = wave_sum(c);
            if (lane == 0) {
                if (it < kHistLds) {
                    ha[it] = a;
                    hb[it] = c;
                } else {
                    b.intermed[it] = a;
                    b.intermed2[it] = c;
                }
            }
        }
        __syncthreads();
        double sa = 0.0, sb = 0.0, vf = 0.0, wm = 0.0;
        if (on) {
#pragma unroll
            for (int k = 0; k < WK; ++k)
                if (1 + k <= h) {  // uniform
                    sa = fma(w[k], ha[1 + k], sa);
                    sb = fma(w[k], hb[1 + k], sb);
                }
            int it = 1 + WK;
#pragma unroll 8
            for (; it <= min(h, kHistLds - 1); ++it) {
                const double x = b.W[(size_t)it * S + tid];
                sa = fma(x, ha[it], sa);
                sb = fma(x, hb[it], sb);
            }
            for (; it <= h; ++it) {
                const double x = b.W[(size_t)it * S + tid];
                sa = fma(x, b.intermed[it], sa);
                sb = fma(x, b.intermed2[it], sb);
            }
            const double pd = PC ? pf - b.PFp[tid] : fraction * d;
            const double vm = d / denom;
            wm = -pd + (nin - nprev) - sa;
            b.V[(size_t)m * S + tid] = vm;
            b.W[(size_t)m * S + tid] = wm;
            vf = fma(vm, Fc, vf);
        }
        vf = wave_sum(vf);
        if (lane == 0) red[0][wave] = vf;  // every thread read red[0] before the barrier above
        __syncthreads();
        double bm = 0.0;
        for (int k = 0; k < kWaves; ++k) bm += red[0][k];
        sv = fma(wm, bm, sb);
        if (on) b.sum_vec[tid] = sv;
    }
    if (on) {
        if (PC) b.PFp[tid] = pf;
        b.n_prev[tid] = nin;
        b.n_in[tid] = nin - pf - sv;
    }
}

__global__ __launch_bounds__(kBroydenThreads) void broyden_step_kernel(int S, int m, double fraction, int norm_type,
                                                                         const double* __restrict__ n_out,
                                                                         BroydenDev b)
{
    if (S <= kBroydenThreads)
        broyden_update_small<false>(S, m, fraction, norm_type, (int)threadIdx.x < S ? n_out[threadIdx.x] : 0.0,
                                    nullptr, b);
    else
        broyden_update<false>(S, m, fraction, norm_type, n_out, nullptr, b);
}

// U_i = U_ext_i - V_gate - sum_j K_ij n_j: one wavefront per row, lanes
// strided over j.
__global__ __launch_bounds__(256) void coulomb_potential_kernel(int N, const double* __restrict__ K,
                                                                const double* __restrict__ n,
                                                                const double* __restrict__ U_ext, double V_gate,
                                                                double* __restrict__ U)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= N) return;
    const double* __restrict__ k = K + (size_t)row * N;
    double acc = 0.0;
#pragma unroll 4
    for (int j = lane; j < N; j += 64) acc = fma(k[j], n[j], acc);
    acc = wave_sum(acc);
    if (lane == 0) U[row] = (U_ext ? U_ext[row] : 0.0) - V_gate - acc;
}

// ---------------------------------------------------------------- Broyden
class Broyden {
   public:
    ~Broyden()
    {
        for (DevBuf* d : {&d_state, &d_hist, &d_out, &d_nout}) d->release();
        h_out.release();
    }
    int init(int S_, double fraction_, int max_step_, int norm_type_)
    {
        S = S_;
        fraction = fraction_;
        max_step = max_step_;
        norm_type = norm_type_;
        int rc;
        if ((rc = d_state.ensure(sizeof(double) * 6 * (size_t)S))) return rc;
        if ((rc = d_hist.ensure(sizeof(double) * (2 * (size_t)(max_step + 1) * S + 2 * (max_step + 1))))) return rc;
        if ((rc = d_out.ensure(sizeof(double) * 4))) return rc;
        if ((rc = d_nout.ensure(sizeof(double) * (size_t)S))) return rc;
        if ((rc = h_out.ensure(sizeof(double) * 4))) return rc;
        return reset(0, 0.0, nullptr);
    }
    BroydenDev dev() const
    {
        BroydenDev b;
        double* st = d_state.as<double>();
        b.n_in = st;
        b.n_prev = st + S;
        b.F = st + 2 * (size_t)S;
        b.dF = st + 3 * (size_t)S;
        b.Norm = st + 4 * (size_t)S;
        b.sum_vec = st + 5 * (size_t)S;
        double* h = d_hist.as<double>();
        b.V = h;
        b.W = h + (size_t)(max_step + 1) * S;
        b.intermed = h + 2 * (size_t)(max_step + 1) * S;
        b.intermed2 = b.intermed + (max_step + 1);
        b.out = d_out.as<double>();
        b.PFp = nullptr;
        return b;
    }
    // Reset_Broyden_Parallel (Broyden_Parallel_General.cpp:250-355).
    int reset(int keep_n_in, double init_value, hipStream_t st)
    {
        BroydenDev b = dev();
        int rc;
        if (!keep_n_in && (rc = fill_device(b.n_in, S, init_value, st))) return rc;
        // the history needs no clearing: update m reads rows 1 .. m - 1, each written by
        // its own update since the reset, and row m after writing it
        if ((rc = fill_device(b.n_prev, 5LL * S, 0.0, st))) return rc;
        step = 1;
        return NEGF_OK;
    }
    // One update from the device output d_n_out; reads back the norms.
    int update(const double* d_n_out, double* max_norm, double* l2, hipStream_t st)
    {
        const int m = step - 1;
        if (m > max_step) {
            set_error("Broyden_Step %d exceeds Broyden_threshold_maxstep %d", step, max_step);
            return NEGF_ENONCONV;
        }
        hipLaunchKernelGGL(broyden_step_kernel, dim3(1), dim3(kBroydenThreads), 0, st, S, m, fraction, norm_type,
                           d_n_out, dev());
        NEGF_HIP_TRY(hipGetLastError());
        NEGF_HIP_TRY(hipMemcpyAsync(h_out.p, d_out.p, sizeof(double) * 3, hipMemcpyDeviceToHost, st));
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        const double* o = h_out.as<double>();
        if (max_norm) *max_norm = o[0];
        if (l2) *l2 = o[1];
        step += 1;
        if (!std::isfinite(o[0]) || !std::isfinite(o[1])) {
            set_error("Broyden: non-finite norm");
            return NEGF_ENAN;
        }
        return NEGF_OK;
    }

    int S = 0, max_step = 0, norm_type = 0, step = 1;
    double fraction = 0.1;
    DevBuf d_state, d_hist, d_out, d_nout;
    HostBuf h_out;
};

// ---------------------------------------------------------------- SCF
struct Scf {
    ~Scf()
    {
        if (st) (void)hipStreamSynchronize(st);
        for (DevBuf* d : {&d_K, &d_U, &d_Q, &d_Uext, &d_ctl}) d->release();
        if (h_back) (void)hipHostFree(h_back);
        if (st) (void)hipStreamDestroy(st);
    }
    Tube* tube = nullptr;
    negf_scf_params p{};
    Broyden br;
    std::vector<double> K;
    DevBuf d_K, d_U, d_Q, d_Uext;
    bool has_ext = false;
    hipStream_t st = nullptr;
    // Launched ahead: gate voltage, Broyden step and whether the loop still runs live on
    // the device (ScfCtl), and the Broyden kernel writes the norms and the plans' status
    // words straight into mapped, coherent host memory (ScfBack), so an iteration is
    // four launches that need nothing from the host.  The next one is launched before
    // the host looks at the present one's norm; the one behind the last finds the loop
    // stopped and changes nothing.  Measured per iteration (400 sites, 29 us of
    // kernels): 33 us, against 38 us as replays of a captured graph (13 us from one
    // replay to the next) and 53 us as replays that the host waits for one by one.
    // Off: every step of an iteration is waited for (negf_scf_use_graph).
    bool ahead = true;
    DevBuf d_ctl;
    void* h_back = nullptr;    // host address (two records: even and odd steps)
    void* d_back = nullptr;    // the same memory as the device sees it
};

struct ScfBack {
    double norm, l2;
    int status[2];
    int step;  // written last: the Broyden step that the record belongs to
};

// Wait until the n words at w, written by kernels on st into mapped host memory, hold
// want.  The stream's state is looked at now and then, so a failed launch ends the wait.
static int wait_words(const int* w, int n, int want, hipStream_t st)
{
    for (int i = 0; i < n; ++i)
        for (unsigned spin = 1; __atomic_load_n(w + i, __ATOMIC_ACQUIRE) != want; ++spin) {
            __builtin_ia32_pause();
            if (spin % 16384) continue;
            const hipError_t e = hipStreamQuery(st);
            if (e == hipErrorNotReady) continue;
            if (e == hipSuccess && __atomic_load_n(w + i, __ATOMIC_ACQUIRE) == want) break;
            set_error("SCF iteration ended without its record: %s", hipGetErrorString(e));
            return NEGF_EDEVICE;
        }
    return NEGF_OK;
}
struct ScfCtl {
    double V;
    int step;    // Broyden step of the next iteration
    int active;  // 0: the loop has ended (converged, or an error that the host reports)
};

// Dense stand-in for the Poisson solve + gather (not in the reference):
// K_ij [V per e] = ke/eps_r (1/sqrt(d^2 + R^2) - 1/sqrt(d^2 + R_img^2)),
// d = axial distance of rings i, j in nm, ke = q/(4 pi eps0) * 1e9 V nm.
static void coulomb_kernel(const std::vector<double>& ptd, const negf_scf_params& p, std::vector<double>& K)
{
    const double q = 1.602176634e-19, eps0 = 8.8541878128e-12, pi = 3.14159265358979323846;
    const double ke = q / (4.0 * pi * eps0) * 1.0e9;
    const size_t N = ptd.size();
    K.resize(N * N);
    for (size_t i = 0; i < N; ++i)
        for (size_t j = 0; j < N; ++j) {
            const double d = ptd[i] - ptd[j];
            const double d2 = d * d;
            K[i * N + j] = ke / p.eps_r *
                           (1.0 / std::sqrt(d2 + p.R_ring_nm * p.R_ring_nm) -
                            1.0 / std::sqrt(d2 + p.R_image_nm * p.R_image_nm));
        }
}

// ---------------------------------------------------------------- batched SCF
// Many equal tubes coupled to their own charge through one shared dense
// kernel K (N x N): every iteration is a GEMM U_t = U_ext,t - V_t - K n_t for
// all tubes, one batched NEGF solve, and one Broyden workgroup per tube.

// Partial products Yp[z][t][i] = sum_{j in chunk z} A[i][j] X[t][j]
// (A row-major M x K, rows lda apart; X rows ldx apart; T rows) on
// v_mfma_f64_16x16x4f64, chunk z = [z kchunk, (z + 1) kchunk); Yp[z] is
// T x M.  A workgroup of 4 wavefronts computes a 32 (i) x 32 (t) tile, one
// 16 x 16 quadrant per wavefront, over 32-wide j blocks staged in LDS; the
// next block's global loads are issued before the present block's MFMAs.
// Lane l supplies A[i0 + l % 16][j + l / 16] and X[t0 + l % 16][j + l / 16];
// result register v of lane l is the entry (i = l / 16 + 4 v, t = l % 16).
// The caller sums the chunks in order.  With live (a device count) nothing is done
// once it is 0 or less.
typedef __attribute__((ext_vector_type(4))) double d4;
__global__ __launch_bounds__(256) void mfma_dgemm_kernel(int M, int K, int T, const double* __restrict__ A,
                                                         size_t lda, const double* __restrict__ X, size_t ldx,
                                                         int kchunk, double* __restrict__ Yp,
                                                         const int* __restrict__ live)
{
    if (live && *live <= 0) return;
    __shared__ double As[32][33];
    __shared__ double Xs[32][33];
    const int i0 = blockIdx.x * 32, t0 = blockIdx.y * 32;
    const int jb = blockIdx.z * kchunk, je = min(K, jb + kchunk);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int qi = w >> 1, qt = w & 1;
    double ra[4], rx[4];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = tid + 256 * q;
            const int r = e >> 5, c = e & 31;
            const int i = i0 + r, t = t0 + r, j = j0 + c;
            ra[q] = (i < M && j < je) ? A[(size_t)i * lda + j] : 0.0;
            rx[q] = (t < T && j < je) ? X[(size_t)t * ldx + j] : 0.0;
        }
    };
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    fetch(jb);
    for (int j0 = jb; j0 < je; j0 += 32) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = tid + 256 * q;
            As[e >> 5][e & 31] = ra[q];
            Xs[e >> 5][e & 31] = rx[q];
        }
        __syncthreads();
        if (j0 + 32 < je) fetch(j0 + 32);
#pragma unroll
        for (int k0 = 0; k0 < 32; k0 += 4) {
            const double a = As[qi * 16 + (lane & 15)][k0 + (lane >> 4)];
            const double x = Xs[qt * 16 + (lane & 15)][k0 + (lane >> 4)];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    double* Y = Yp + (size_t)blockIdx.z * T * M;
    const int t = t0 + qt * 16 + (lane & 15);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = i0 + qi * 16 + (lane >> 4) + 4 * v;
        if (i < M && t < T) Y[(size_t)t * M + i] = acc[v];
    }
}

// K-split of a GEMM with M output rows and inner length K: enough
// workgroups to cover the chip (about 1024), chunks a multiple of 32 wide
static int gemm_splits(int M, int K, int T)
{
    const int tiles = ((M + 31) / 32) * ((T + 31) / 32);
    int z = std::max(1, std::min(8, 1024 / std::max(tiles, 1)));
    while (z > 1 && (K + 32 * z - 1) / (32 * z) < 4) --z;  // keep >= 4 blocks per chunk
    return z;
}

static int gemm_chunk(int K, int z) { return ((K + z - 1) / z + 31) / 32 * 32; }

// Yp[z] (T x M) = A (M x K, rows lda apart) X^T over chunk z of the inner index
static void launch_dgemm(int M, int K, int T, int z, const double* A, size_t lda, const double* X, size_t ldx,
                         double* Yp, hipStream_t st, const int* live = nullptr)
{
    dim3 g((M + 31) / 32, (T + 31) / 32, z);
    hipLaunchKernelGGL(mfma_dgemm_kernel, g, dim3(256), 0, st, M, K, T, A, lda, X, ldx, gemm_chunk(K, z), Yp, live);
}

// Y = sum of the z partial products, in chunk order
__device__ __forceinline__ double sum_parts(const double* __restrict__ P, int z, long long NT, long long q)
{
    double a = P[q];
    for (int k = 1; k < z; ++k) a += P[k * NT + q];
    return a;
}

// U_t = U_ext,t - V_t - KN_t, scattered into each tube's potential and
// contact potentials; also kept in Uall for the caller.
__global__ void batch_potential_kernel(int N, int T, const double* __restrict__ Uext, const double* __restrict__ V,
                                       const double* __restrict__ KN, int nz, double* const* __restrict__ dU,
                                       double* const* __restrict__ dUc, double* __restrict__ Uall,
                                       const int* __restrict__ live)
{
    if (*live <= 0) return;
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long NT = (long long)N * T;
    if (q >= NT) return;
    const int t = (int)(q / N), i = (int)(q - (long long)t * N);
    const double u = (Uext ? Uext[q] : 0.0) - V[t] - sum_parts(KN, nz, NT, q);
    Uall[q] = u;
    dU[t][i] = u;
    if (i == 0) dUc[t][0] = u;
    if (i == N - 1) dUc[t][1] = u;
}

// The charge of a batch's tubes before its last two steps: tube t's equilibrium
// charge in nrows[t] partial rows (row r of site s at part[off[t] + r S + s]), and
// the arrays that batch_combine_kernel reads.
struct ChargeRows {
    const double* part = nullptr;  // nullptr: Q is formed already
    const long long* off;
    const int* nrows;
    double* eq;
    const double *neq, *rho0;
};

// Doubles of a read-back record: 4 per tube (max norm, l2 norm, |dF|^2, step-limit
// flag), the plans' two status words and per tube the count of iterations, written last.
__host__ __device__ constexpr size_t rec_stride(int T) { return 4 * (size_t)T + 1 + ((size_t)T + 1) / 2; }

// Where the iteration's outcome goes: the host's two read-back records, used in turn,
// and the kept U and Q.
struct TrackOut {
    const double* U;
    double *Uo, *Qo;
    double* back;
    const int *st_eq, *st_neq;
    double max_norm;
};

// The end of a batched iteration, one workgroup per tube: with cr.part the tube's
// charge from the partial rows (summed in order from 0.0, as the plan's own row sum of
// at most 16 rows, into eq; Q = (eq + noneq) - rho0), one Broyden update, and the
// tube's record.  A tube whose max norm reached max_norm keeps its U and Q (Uo, Qo) and
// leaves the active set, as does one at its step limit; the host applies the same
// tests to the same values, so its bookkeeping follows without copies.  A residual that
// is not finite stops every tube from the next iteration on (the host reports it).  The
// counters live on the device so that the launch is identical every iteration: steps[t]
// the Broyden step, steps[T + t] the iteration, steps[2T] the first iteration that is not
// to run (0: none), steps[2T + 1] the tubes still active (0 or less: the loop has
// ended, and the potential stays too).  Row sum, charge, update and record in one launch instead of four: 32
// tubes x 1024 sites, 16.6 us against 3.9 + 2.9 + 14.8 + 3.9.
// SMALL (at most kBroydenThreads sites) and the general update are kernels of their own: as
// one with a branch the general one runs at half the speed (104 registers instead of
// 53); 3 tubes x 6000 / 2048 / 1200 sites 265 / 81 / 54 us an iteration, now 204 / 68 / 52.
template <bool PC, bool SMALL>
__global__ __launch_bounds__(kBroydenThreads) void broyden_batch_kernel(int S, int T, int max_step, double fraction,
                                                                          int norm_type, ChargeRows cr, double* n_out_all,
                                                                          const double* __restrict__ PF,
                                                                          BroydenDev base, size_t state_stride,
                                                                          size_t hist_stride, int* steps, int* active,
                                                                          TrackOut tr)
{
    __shared__ int keep;
    const int t = blockIdx.x;
    const int tid = threadIdx.x;
    const int it = steps[T + t], halt = steps[2 * T];
    double* rec = tr.back + (size_t)(it & 1) * rec_stride(T);
    int* rec_it = reinterpret_cast<int*>(rec + 4 * T + 1) + t;
    const bool on = active[t] != 0 && !(halt > 0 && halt <= it);
    __syncthreads();  // every thread has read the counter and the flag
    if (tid == 0) {
        steps[T + t] = it + 1;
        if (t == 0) {
            int* st = reinterpret_cast<int*>(rec + 4 * T);
            st[0] = *tr.st_eq;
            st[1] = tr.st_neq ? *tr.st_neq : 0;
        }
        if (!on) {
            __threadfence_system();
            __hip_atomic_store(rec_it, it + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    if (!on) return;
    const size_t o = (size_t)t * S;
    double* n_out = n_out_all + o;
    double q = 0.0;  // this thread's last entry of Q: the only one up to kBroydenThreads sites
    if (!PC && cr.part) {
        const double* part = cr.part + cr.off[t];
        const int R = cr.nrows[t];
        for (int s = tid; s < S; s += kBroydenThreads) {
            double e = 0.0;
#pragma unroll 4
            for (int r = 0; r < R; ++r) e += part[(size_t)r * S + s];
            cr.eq[o + s] = e;
            q = (e + cr.neq[o + s]) - cr.rho0[o + s];
            n_out[s] = q;
        }
    } else if (tid < S) {
        q = n_out[tid];
    }
    const int m = steps[t] - 1;
    BroydenDev b;
    b.n_in = base.n_in + t * state_stride;
    b.n_prev = base.n_prev + t * state_stride;
    b.F = base.F + t * state_stride;
    b.dF = base.dF + t * state_stride;
    b.Norm = base.Norm + t * state_stride;
    b.sum_vec = base.sum_vec + t * state_stride;
    b.V = base.V + t * hist_stride;
    b.W = base.W + t * hist_stride;
    b.intermed = base.intermed + t * hist_stride;
    b.intermed2 = base.intermed2 + t * hist_stride;
    b.out = base.out + (size_t)t * 4;
    b.PFp = PC ? base.PFp + t * state_stride : nullptr;
    const bool limit = m > max_step;
    if (!limit) {  // uniform
        if constexpr (SMALL)
            broyden_update_small<PC>(S, m, fraction, norm_type, q, PC ? PF + o : nullptr, b);
        else
            broyden_update<PC>(S, m, fraction, norm_type, n_out, PC ? PF + o : nullptr, b);
    }
    if (tid == 0) {  // b.out[0..2] were written by this thread
        if (!limit) steps[t] = m + 2;
        const double nrm = b.out[0];
        // the max norm drops a NaN (it is a chain of fmax), |dF|^2 keeps it
        const bool finite = isfinite(nrm) && isfinite(b.out[2]);
        b.out[3] = limit ? 1.0 : 0.0;  // step limit reached
        for (int k = 0; k < 3; ++k) rec[4 * t + k] = b.out[k];
        rec[4 * t + 3] = limit ? 1.0 : 0.0;
        keep = !limit && finite && nrm <= tr.max_norm;
        if (limit || keep) {
            active[t] = 0;
            atomicSub(&steps[2 * T + 1], 1);
        } else if (!finite) {
            steps[2 * T] = it + 1;
            atomicSub(&steps[2 * T + 1], T + 1);
        }
        __threadfence_system();
        __hip_atomic_store(rec_it, it + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    if (!keep) return;
    for (int i = tid; i < S; i += kBroydenThreads) {
        tr.Uo[o + i] = tr.U[o + i];
        tr.Qo[o + i] = n_out[i];
    }
}

// R[t][s] = n_in,t[s] - Q[t][s] (the reference's F = n_in - n_out)
__global__ void batch_residual_kernel(int N, int T, const double* __restrict__ n_in, size_t stride,
                                      const double* __restrict__ Q, double* __restrict__ R)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)N * T) return;
    const int t = (int)(q / N), i = (int)(q - (long long)t * N);
    R[q] = n_in[(size_t)t * stride + i] - Q[q];
}

// Mode-space factor of the preconditioner's correction:
// Y[t][k] = (sum of the z partial products) * c_t lam_k / (1 + c_t lam_k)
__global__ void batch_modescale_kernel(int R, int T, const double* __restrict__ lam, const double* __restrict__ c,
                                       const double* __restrict__ parts, int nz, double* __restrict__ Y)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long RT = (long long)R * T;
    if (q >= RT) return;
    const int t = (int)(q / R), k = (int)(q - (long long)t * R);
    const double cl = c[t] * lam[k];
    Y[q] = sum_parts(parts, nz, RT, q) * (cl / (1.0 + cl));
}

// X = Rv - (sum of the z partial products)
__global__ void batch_minus_parts_kernel(long long NT, const double* __restrict__ Rv,
                                         const double* __restrict__ parts, int nz, double* __restrict__ X)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < NT) X[q] = Rv[q] - sum_parts(parts, nz, NT, q);
}

// c_t = max(0, mean_s J[t][s]) for the tubes in use: the site-averaged
// response dQ/dU . 1 (capacitance per site, e per eV); one workgroup per tube
__global__ __launch_bounds__(256) void batch_rowmean_kernel(int N, const double* __restrict__ J,
                                                            double* __restrict__ c)
{
    __shared__ double red[4];
    const int t = blockIdx.x;
    double a = 0.0;
    for (int s = threadIdx.x; s < N; s += 256) a += J[(size_t)t * N + s];
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double m = (red[0] + red[1] + red[2] + red[3]) / N;
        c[t] = m > 0.0 ? m : 0.0;
    }
}

// n_in,t -= P R_t (a preconditioned step without history, for the seed)
// One seed step n_in -= beta P (n_in - Q_surrogate)
__global__ void batch_seed_step_kernel(int N, int T, double* __restrict__ n_in, size_t stride,
                                       const double* __restrict__ PR, double beta)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)N * T) return;
    const int t = (int)(q / N), i = (int)(q - (long long)t * N);
    n_in[(size_t)t * stride + i] -= beta * PR[q];
}

__global__ __launch_bounds__(256) void batch_clear_state_kernel(int n, int T, double* __restrict__ p, size_t stride)
{
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    if (q >= (long long)n * T) return;
    const size_t t = (size_t)(q / n);
    p[t * stride + ((size_t)q - t * n)] = 0.0;
}

// The tubes' input charges between their Broyden states (state t at p + t stride) and a
// dense array [T][n]: with PUT into the states, else out of them.  One launch and one
// copy instead of a synchronous copy per tube (32 tubes: 300 us).
template <bool PUT>
__global__ __launch_bounds__(256) void batch_charge_rows_kernel(int n, int T, double* __restrict__ p,
                                                                size_t stride, double* __restrict__ dense)
{
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    if (q >= (long long)n * T) return;
    const size_t t = (size_t)(q / n), i = (size_t)q - t * n;
    if (PUT)
        p[t * stride + i] = dense[q];
    else
        dense[q] = p[t * stride + i];
}

class BatchScf {
   public:
    ~BatchScf()
    {
        if (st) {
            (void)hipStreamSynchronize(st);
            (void)hipStreamDestroy(st);
        }
        if (h_back) (void)hipHostFree(h_back);
    }
    int init(negf_batch* b, negf_tube* const* tubes, int T_, const negf_scf_params& prm)
    {
        batch = b;
        T = T_;
        p = prm;
        N = tubes[0]->t.N;
        this->tubes.assign(tubes, tubes + T_);
        for (int t = 0; t < T; ++t) {
            if (tubes[t]->t.N != N) {
                set_error("batched SCF needs tubes of equal length (shared electrostatic kernel)");
                return NEGF_EARG;
            }
            hU.push_back(tubes[t]->t.d_U.as<double>());
            hUc.push_back(tubes[t]->t.d_Uc());
        }
        coulomb_kernel(tubes[0]->t.ptd, p, K);
        M = p.Broyden_threshold_maxstep;
        state_stride = 7 * (size_t)N;
        hist_stride = 2 * (size_t)(M + 1) * N + 2 * (M + 1);
        int rc;
        NEGF_HIP_TRY(hipStreamCreate(&st));
        if ((rc = d_K.ensure(sizeof(double) * K.size()))) return rc;
        if ((rc = d_Uext.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_V.ensure(sizeof(double) * T))) return rc;
        nz = gemm_splits(N, N, T);
        if ((rc = d_KN.ensure(sizeof(double) * N * T * nz))) return rc;
        if ((rc = d_U.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_Q.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_Uo.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_Qo.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_ptrU.ensure(sizeof(double*) * T))) return rc;
        if ((rc = d_ptrUc.ensure(sizeof(double*) * T))) return rc;
        if ((rc = d_state.ensure(sizeof(double) * state_stride * T))) return rc;
        if ((rc = d_hist.ensure(sizeof(double) * hist_stride * T))) return rc;
        if ((rc = d_out.ensure(sizeof(double) * 4 * T))) return rc;
        if ((rc = d_steps.ensure(sizeof(int) * (2 * T + 2)))) return rc;
        if ((rc = d_active.ensure(sizeof(int) * T))) return rc;
        {
            hipError_t eh = hipHostMalloc(&h_back, 2 * sizeof(double) * rec_stride(T),
                                          hipHostMallocMapped | hipHostMallocCoherent);
            if (eh == hipSuccess) eh = hipHostGetDevicePointer(&d_back, h_back, 0);
            if (eh != hipSuccess) {
                set_error("mapped host buffer for the batched SCF read-back: %s", hipGetErrorString(eh));
                return NEGF_EALLOC;
            }
        }
        NEGF_HIP_TRY(hipMemcpy(d_K.p, K.data(), sizeof(double) * K.size(), hipMemcpyHostToDevice));
        NEGF_HIP_TRY(hipMemcpy(d_ptrU.p, hU.data(), sizeof(double*) * T, hipMemcpyHostToDevice));
        NEGF_HIP_TRY(hipMemcpy(d_ptrUc.p, hUc.data(), sizeof(double*) * T, hipMemcpyHostToDevice));
        if ((rc = fill_device(d_Uext.as<double>(), (long long)N * T, 0.0, st))) return rc;
        if ((rc = fill_device(d_state.as<double>(), (long long)(state_stride * T), 0.0, st))) return rc;
        for (int t = 0; t < T; ++t)
            if ((rc = fill_device(d_state.as<double>() + t * state_stride, N, p.NS_initial_deposit_value, st)))
                return rc;
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        return NEGF_OK;
    }
    // Reset_Broyden_Parallel of every tube, n_in kept.  The history rows need no
    // clearing (Broyden::reset).
    int clear_history()
    {
        hipLaunchKernelGGL(batch_clear_state_kernel, dim3((unsigned)((6LL * N * T + 255) / 256)), dim3(256), 0, st, 6 * N, T,
                           d_state.as<double>() + N, state_stride);
        NEGF_HIP_TRY(hipGetLastError());
        return NEGF_OK;
    }
    BroydenDev base() const
    {
        BroydenDev b;
        double* s0 = d_state.as<double>();
        b.n_in = s0;
        b.n_prev = s0 + N;
        b.F = s0 + 2 * (size_t)N;
        b.dF = s0 + 3 * (size_t)N;
        b.Norm = s0 + 4 * (size_t)N;
        b.sum_vec = s0 + 5 * (size_t)N;
        double* h = d_hist.as<double>();
        b.V = h;
        b.W = h + (size_t)(M + 1) * N;
        b.intermed = h + 2 * (size_t)(M + 1) * N;
        b.intermed2 = b.intermed + (M + 1);
        b.out = d_out.as<double>();
        b.PFp = s0 + 6 * (size_t)N;
        return b;
    }
    int enqueue_iteration()
    {
        int rc = enqueue_potential();
        if (rc) return rc;
        // the batch leaves its last two steps to the Broyden launch where its own row sum
        // is the in-order one (at most 16 rows)
        ChargeRows cr;
        BatchRows br;
        const bool fuse = batch_rows(batch, &br);
        rc = batch_enqueue(batch, d_Q.as<double>(), st, d_active.as<int>(), !fuse);
        if (rc) return rc;
        if (fuse) cr = ChargeRows{br.part, br.off, br.nrows, br.eq, br.neq, br.rho0};
        return enqueue_broyden<false>(cr, nullptr);
    }
    template <bool PC>
    int enqueue_broyden(const ChargeRows& cr, const double* PF)
    {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(T), dim3(kBroydenThreads), 0, st, N, T, M, p.Broyden_fraction,
                               p.Broyden_norm_type, cr, d_Q.as<double>(), PF, base(), state_stride, hist_stride,
                               d_steps.as<int>(), d_active.as<int>(), track_out());
        };
        if (N <= kBroydenThreads)
            launch(broyden_batch_kernel<PC, true>);
        else
            launch(broyden_batch_kernel<PC, false>);
        NEGF_HIP_TRY(hipGetLastError());
        return NEGF_OK;
    }
    TrackOut track_out() const
    {
        TrackOut tr;
        tr.U = d_U.as<const double>();
        tr.Uo = d_Uo.as<double>();
        tr.Qo = d_Qo.as<double>();
        tr.back = static_cast<double*>(d_back);
        tr.st_eq = tr.st_neq = nullptr;
        batch_status_words(batch, &tr.st_eq, &tr.st_neq);
        tr.max_norm = p.Broyden_max_norm;
        return tr;
    }
    // Host part of iteration it: when a tube's adaptive correction falls due
    // (flag_adaptive_integration_limits), its integrand is sampled at this
    // iteration's potential, so the potential is written first, as in
    // Solve_NEGF (NEGF_Common.cpp:1314-1337); then the batch's plans are
    // brought up to date.
    int prepare_iteration(int it)
    {
        int rc;
        if (adaptive_due(it)) {
            if ((rc = enqueue_potential())) return rc;
            NEGF_HIP_TRY(hipStreamSynchronize(st));
        }
        bool rebuilt = false;
        return batch_prepare(batch, it, &rebuilt);
    }
    bool adaptive_due(int it) const
    {
        for (const negf_tube* t : tubes)
            if (t->t.p.flag_adaptive_integration_limits && it % t->t.p.integrand_correction_interval == 0) return true;
        return false;
    }

    double* record(int it) const { return static_cast<double*>(h_back) + (size_t)(it & 1) * rec_stride(T); }
    // Wait for iteration it's read-back record, which its Broyden kernel
    // writes; from it, fold nonzero plan status words into the batch's
    // sticky root flag, stop on a non-finite norm, and mirror the device's
    // retirement of converged tubes (which already kept their U and Q).
    struct LoopState {
        std::vector<int> active, keep, done_it;
        std::vector<double> fin;
        int remaining = 0;
        bool overflow = false;
    };
    int after_iteration(int it, LoopState& ls)
    {
        int rc;
        const double* o = record(it);
        const int* bs = reinterpret_cast<const int*>(o + 4 * T);
        if ((rc = wait_words(bs + 2, T, it + 1, st))) return rc;
        if (bs[0] | bs[1]) {
            // the status words are read and cleared: not under a running iteration
            NEGF_HIP_TRY(hipStreamSynchronize(st));
            if ((rc = batch_poll_status(batch))) return rc;
        }
        for (int t = 0; t < T; ++t) {
            ls.keep[t] = 0;
            if (!ls.active[t]) continue;
            if (o[4 * t + 3] != 0.0) {
                ls.overflow = true;
                ls.active[t] = 0;
                --ls.remaining;
                continue;
            }
            const double nrm = o[4 * t];
            if (!std::isfinite(nrm) || !std::isfinite(o[4 * t + 2])) {
                set_error("batched SCF: non-finite Broyden norm for tube %d at iteration %d", t, it + 1);
                return NEGF_ENAN;
            }
            if (nrm <= p.Broyden_max_norm) {  // the Broyden kernel kept U, Q and cleared the flag
                ls.keep[t] = 1;
                ls.active[t] = 0;
                ls.done_it[t] = it + 1;
                ls.fin[t] = nrm;
                --ls.remaining;
            }
        }
        return NEGF_OK;
    }
    int finish_run(int it, const LoopState& ls, double* U_out, double* Q_out, int* iters, double* norms,
                   int* total_iters)
    {
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        if (U_out) NEGF_HIP_TRY(hipMemcpy(U_out, d_Uo.p, sizeof(double) * N * T, hipMemcpyDeviceToHost));
        if (Q_out) NEGF_HIP_TRY(hipMemcpy(Q_out, d_Qo.p, sizeof(double) * N * T, hipMemcpyDeviceToHost));
        if (iters) std::copy(ls.done_it.begin(), ls.done_it.end(), iters);
        if (norms) std::copy(ls.fin.begin(), ls.fin.end(), norms);
        if (total_iters) *total_iters = it;
        if (ls.overflow) {
            set_error("Broyden_Step has exceeded the Broyden_Threshold_MaxStep for some tube");
            return NEGF_ENONCONV;
        }
        return NEGF_OK;
    }
    int start_run(const double* V, LoopState& ls)
    {
        NEGF_HIP_TRY(hipMemcpyAsync(d_V.p, V, sizeof(double) * T, hipMemcpyHostToDevice, st));
        std::vector<int> steps(2 * T + 2, 0);  // Broyden steps 1, iterations 0, no halt, T tubes
        std::fill(steps.begin(), steps.begin() + T, 1);
        steps[2 * T + 1] = T;
        ls.active.assign(T, 1);
        ls.keep.assign(T, 0);
        ls.done_it.assign(T, -1);
        ls.fin.assign(T, 0.0);
        ls.remaining = T;
        ls.overflow = false;
        NEGF_HIP_TRY(hipMemcpyAsync(d_steps.p, steps.data(), sizeof(int) * steps.size(), hipMemcpyHostToDevice, st));
        NEGF_HIP_TRY(hipMemcpyAsync(d_active.p, ls.active.data(), sizeof(int) * T, hipMemcpyHostToDevice, st));
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        return NEGF_OK;
    }

    // Iteration it onto the stream.
    template <class F>
    int launch_iteration(int it, F enqueue)
    {
        int rc;
        if ((rc = prepare_iteration(it))) return rc;
        int* w = reinterpret_cast<int*>(record(it) + 4 * T + 1);
        for (int t = 0; t < T; ++t) __atomic_store_n(w + t, 0, __ATOMIC_RELEASE);
        return enqueue();
    }
    // Iteration it may be launched before the host has seen the one before: it needs
    // nothing from the host, and the GPU does not wait for it.  Once the last tube has
    // left the active set such an iteration changes nothing.  Measured (32 tubes x 1024
    // sites, 54 us of kernels an iteration): 2049 us a run, 2226 us with the iterations
    // as replays of a captured graph (13 us from one replay to the next).
    bool runs_ahead(int it) const { return ahead && it <= M + 1 && !adaptive_due(it); }

    // Run every tube to Broyden_Norm <= Broyden_max_norm (or its step
    // limit); per-tube iteration counts and final norms.
    int run(const double* V, double* U_out, double* Q_out, int* iters, double* norms, int* total_iters)
    {
        int rc, it = 0;
        LoopState ls;
        if ((rc = start_run(V, ls))) return rc;
        auto next = [&] { return enqueue_iteration(); };
        if ((rc = iterate(ls, &it, [](int) { return NEGF_OK; }, next, -1))) return drain(rc);
        return finish_run(it, ls, U_out, Q_out, iters, norms, total_iters);
    }
    // The loop of a run: before(it) on the host, then iteration it, and the next one ahead
    // of it unless that is number hold.  *it counts the iterations.
    template <class B, class F>
    int iterate(LoopState& ls, int* count, B before, F enqueue, int hold)
    {
        int rc, launched = 0;
        int& it = *count;
        while (ls.remaining > 0) {
            if (it > M + 1) {
                ls.overflow = true;
                break;
            }
            if ((rc = before(it))) return rc;
            if (launched == it) {
                if ((rc = launch_iteration(it, enqueue))) return rc;
                ++launched;
            }
            if (it + 1 != hold && runs_ahead(it + 1)) {
                if ((rc = launch_iteration(it + 1, enqueue))) return rc;
                ++launched;
            }
            if ((rc = after_iteration(it, ls))) return rc;
            ++it;
        }
        return NEGF_OK;
    }
    // A run that ends by an error: the iteration launched ahead still writes the batch's
    // rows, the status words and the record, so it is waited for before the caller goes on.
    int drain(int rc)
    {
        (void)hipStreamSynchronize(st);
        return rc;
    }

    // ---- surrogate-seeded, preconditioned iteration
    // P_t = Z diag(1 / (1 + c_t lam)) Z^T = I - Z diag(c_t lam / (1 + c_t lam)) Z^T,
    // applied with the modes of lam_k >= kPcModeCut * max lam only: a dropped
    // mode's factor differs from 1 by c_t lam_k / (1 + c_t lam_k) < c_t
    // kPcModeCut max lam, and P only sets the mixing, not the fixed point.
    static constexpr double kPcModeCut = 1e-2;
    int set_preconditioner(const double* Z, const double* lam)
    {
        int rc;
        double lmax = 0.0;
        for (int k = 0; k < N; ++k) lmax = std::max(lmax, lam[k]);
        std::vector<int> keep;
        for (int k = 0; k < N; ++k)
            if (lam[k] > 0.0 && lam[k] >= kPcModeCut * lmax) keep.push_back(k);
        R_pc = std::max<int>(1, (int)keep.size());
        const size_t NR = (size_t)N * R_pc;
        if ((rc = d_Z.ensure(sizeof(double) * NR))) return rc;
        if ((rc = d_Zt.ensure(sizeof(double) * NR))) return rc;
        if ((rc = d_lam.ensure(sizeof(double) * R_pc))) return rc;
        if ((rc = d_c.ensure(sizeof(double) * T))) return rc;
        if ((rc = d_R.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_Rh.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_PF.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_ones.ensure(sizeof(double) * N * T))) return rc;
        if ((rc = d_J.ensure(sizeof(double) * N * T))) return rc;
        z_pc1 = gemm_splits(R_pc, N, T);
        z_pc2 = gemm_splits(N, R_pc, T);
        const size_t kn = std::max({(size_t)N * T * nz, (size_t)R_pc * T * z_pc1, (size_t)N * T * z_pc2});
        if ((rc = d_KN.ensure(sizeof(double) * kn))) return rc;
        // Zr: N x R (row i: the kept modes' entries at site i); Zrt: R x N
        std::vector<double> zr(NR, 0.0), zrt(NR, 0.0), lr(R_pc, 0.0);
        for (int q = 0; q < (int)keep.size(); ++q) {
            const int k = keep[q];
            lr[q] = lam[k];
            for (int i = 0; i < N; ++i) {
                zr[(size_t)i * R_pc + q] = Z[(size_t)i * N + k];
                zrt[(size_t)q * N + i] = Z[(size_t)i * N + k];
            }
        }
        NEGF_HIP_TRY(hipMemcpy(d_Z.p, zr.data(), sizeof(double) * NR, hipMemcpyHostToDevice));
        NEGF_HIP_TRY(hipMemcpy(d_Zt.p, zrt.data(), sizeof(double) * NR, hipMemcpyHostToDevice));
        NEGF_HIP_TRY(hipMemcpy(d_lam.p, lr.data(), sizeof(double) * R_pc, hipMemcpyHostToDevice));
        if ((rc = fill_device(d_ones.as<double>(), (long long)N * T, 1.0, st))) return rc;
        if ((rc = fill_device(d_c.as<double>(), T, 0.0, st))) return rc;
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        has_pc = true;
        return NEGF_OK;
    }
    // U_t = U_ext,t - V_t - K n_in,t into the tubes and d_U
    int enqueue_potential()
    {
        launch_dgemm(N, N, T, nz, d_K.as<double>(), (size_t)N, base().n_in, state_stride, d_KN.as<double>(), st, live());
        const long long NT = (long long)N * T;
        hipLaunchKernelGGL(batch_potential_kernel, dim3((unsigned)((NT + 255) / 256)), dim3(256), 0, st, N, T,
                           d_Uext.as<double>(), d_V.as<double>(), d_KN.as<double>(), nz,
                           d_ptrU.as<double*>(), d_ptrUc.as<double*>(), d_U.as<double>(), live());
        NEGF_HIP_TRY(hipGetLastError());
        return NEGF_OK;
    }
    const int* live() const { return d_steps.as<const int>() + 2 * T + 1; }
    // d_PF = P (n_in - Q) from the charge Q (T x N): R = n_in - Q,
    // Y = Zr^T R, Y_k *= c_t lam_k / (1 + c_t lam_k), PF = R - Zr Y
    int enqueue_precondition(const double* Q)
    {
        const long long NT = (long long)N * T, RT = (long long)R_pc * T;
        const dim3 g((unsigned)((NT + 255) / 256));
        hipLaunchKernelGGL(batch_residual_kernel, g, dim3(256), 0, st, N, T, base().n_in, state_stride, Q,
                           d_R.as<double>());
        launch_dgemm(R_pc, N, T, z_pc1, d_Zt.as<double>(), (size_t)N, d_R.as<double>(), (size_t)N,
                     d_KN.as<double>(), st);
        hipLaunchKernelGGL(batch_modescale_kernel, dim3((unsigned)((RT + 255) / 256)), dim3(256), 0, st, R_pc, T,
                           d_lam.as<double>(), d_c.as<double>(), d_KN.as<double>(), z_pc1, d_Rh.as<double>());
        launch_dgemm(N, R_pc, T, z_pc2, d_Z.as<double>(), (size_t)R_pc, d_Rh.as<double>(), (size_t)R_pc,
                     d_KN.as<double>(), st);
        hipLaunchKernelGGL(batch_minus_parts_kernel, g, dim3(256), 0, st, NT, d_R.as<double>(), d_KN.as<double>(),
                           z_pc2, d_PF.as<double>());
        NEGF_HIP_TRY(hipGetLastError());
        return NEGF_OK;
    }
    // c_t from the surrogate's tangent dQ/dU . 1 at the present d_U
    int enqueue_capacitance()
    {
        int rc = sg->forward(T, d_U.as<double>(), has_feat ? d_feat.as<double>() : nullptr, st);
        if (!rc) rc = sg->jvp(T, d_ones.as<double>(), d_J.as<double>(), st);
        if (rc) return rc;
        hipLaunchKernelGGL(batch_rowmean_kernel, dim3(T), dim3(256), 0, st, N, d_J.as<double>(), d_c.as<double>());
        NEGF_HIP_TRY(hipGetLastError());
        return NEGF_OK;
    }
    int enqueue_iteration_pc()
    {
        int rc = enqueue_potential();
        if (!rc) rc = batch_enqueue(batch, d_Q.as<double>(), st, d_active.as<int>());
        if (!rc) rc = enqueue_precondition(d_Q.as<double>());
        if (rc) return rc;
        return enqueue_broyden<true>(ChargeRows(), d_PF.as<const double>());
    }
    // Seed steps are half steps: with full steps the scalar capacitance
    // overshoots on the high-gate tubes, whose seed then oscillates (128
    // tubes x 2048 sites: 3 full steps leave a tube unconverged after 300
    // exact iterations; 6 half steps need 23 against 29 after 6 full ones).
    static constexpr double kSeedStep = 0.5;
    // Seeded, preconditioned run: seed_iters preconditioned steps on the
    // surrogate charge (a fixed-point iteration of the surrogate SCF), then
    // the Broyden loop on the exact NEGF charge with the mixing term P F.  The
    // capacitances come from the surrogate at the start, half way through
    // the seed, at the seed, and (with a fresh history) at iteration
    // refresh_iter of the exact loop if refresh_iter > 0.
    int run_pc(const double* V, int seed_iters, int refresh_iter, double* U_out, double* Q_out, int* iters,
               double* norms, int* total_iters, double* cap)
    {
        int rc;
        LoopState ls;
        if ((rc = start_run(V, ls))) return rc;
        if ((rc = enqueue_potential())) return rc;
        if ((rc = enqueue_capacitance())) return rc;
        const long long NT = (long long)N * T;
        for (int k = 0; k < seed_iters; ++k) {
            // the capacitances follow the seed once, half way
            if (k > 0 && k == seed_iters / 2 && (rc = enqueue_capacitance())) return rc;
            if ((rc = sg->forward(T, d_U.as<double>(), has_feat ? d_feat.as<double>() : nullptr, st))) return rc;
            if ((rc = sg->output(T, d_Q.as<double>(), st))) return rc;
            if ((rc = enqueue_precondition(d_Q.as<double>()))) return rc;
            hipLaunchKernelGGL(batch_seed_step_kernel, dim3((unsigned)((NT + 255) / 256)), dim3(256), 0, st, N, T,
                               base().n_in, state_stride, d_PF.as<double>(), kSeedStep);
            NEGF_HIP_TRY(hipGetLastError());
            if ((rc = enqueue_potential())) return rc;
        }
        if (seed_iters > 0 && (rc = enqueue_capacitance())) return rc;
        NEGF_HIP_TRY(hipStreamSynchronize(st));
        auto refresh = [&](int it) {
            if (it == 0 || it != refresh_iter) return (int)NEGF_OK;
            // new capacitances at the present potential; fresh history, n_in kept
            if (int e = enqueue_capacitance()) return e;
            std::vector<int> steps(T, 1);
            NEGF_HIP_TRY(hipMemcpyAsync(d_steps.p, steps.data(), sizeof(int) * T, hipMemcpyHostToDevice, st));
            NEGF_HIP_TRY(hipStreamSynchronize(st));
            return (int)NEGF_OK;
        };
        auto next = [&] { return enqueue_iteration_pc(); };
        int it = 0;
        if ((rc = iterate(ls, &it, refresh, next, refresh_iter))) return drain(rc);
        rc = finish_run(it, ls, U_out, Q_out, iters, norms, total_iters);
        if (cap) NEGF_HIP_TRY(hipMemcpy(cap, d_c.p, sizeof(double) * T, hipMemcpyDeviceToHost));
        return rc;
    }

    Surrogate* sg = nullptr;
    bool has_pc = false, has_feat = false;
    DevBuf d_Z, d_Zt, d_lam, d_c, d_R, d_Rh, d_PF, d_ones, d_J, d_feat;

    negf_batch* batch = nullptr;
    std::vector<negf_tube*> tubes;
    int T = 0, N = 0, M = 0;
    int nz = 1;  // K-split of the GEMMs (partials in d_KN)
    int R_pc = 0, z_pc1 = 1, z_pc2 = 1;   // preconditioner modes and its GEMMs' K-splits
    negf_scf_params p{};
    std::vector<double> K;
    std::vector<double*> hU, hUc;
    size_t state_stride = 0, hist_stride = 0;
    DevBuf d_K, d_Uext, d_V, d_KN, d_U, d_Q, d_Uo, d_Qo, d_ptrU, d_ptrUc, d_state, d_hist, d_out, d_steps,
        d_active;
    void* h_back = nullptr;   // mapped read-back record (host address)
    void* d_back = nullptr;   // the same memory as the device sees it
    bool has_ext = false;
    bool ahead = true;  // launch iterations ahead of the host's tests
    hipStream_t st = nullptr;
};

// The potential of one SCF iteration written where the loop and the tube
// read it: U_i = U_ext_i - V - sum_j K_ij n_j (the sum as in
// coulomb_potential_kernel) into U and tU, the contact potentials U_0 and
// U_{N-1} into tUc.  V is read from the device, with the flag that says whether the
// loop still runs: an iteration launched ahead needs nothing from the host.
__global__ __launch_bounds__(256) void scf_potential_kernel(int N, const double* __restrict__ K,
                                                            const double* __restrict__ n,
                                                            const double* __restrict__ U_ext,
                                                            const ScfCtl* __restrict__ ctl, double* __restrict__ U,
                                                            double* __restrict__ tU, double* __restrict__ tUc)
{
    if (!ctl->active) return;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= N) return;
    const double* __restrict__ k = K + (size_t)row * N;
    double acc = 0.0;
#pragma unroll 4
    for (int j = lane; j < N; j += 64) acc = fma(k[j], n[j], acc);
    acc = wave_sum(acc);
    if (lane == 0) {
        const double u = (U_ext ? U_ext[row] : 0.0) - ctl->V - acc;
        U[row] = u;
        tU[row] = u;
        if (row == 0) tUc[0] = u;
        if (row == N - 1) tUc[1] = u;
    }
}

static void scf_enqueue_potential(Scf& s, hipStream_t q)
{
    Tube& t = *s.tube;
    hipLaunchKernelGGL(scf_potential_kernel, dim3((t.N + 3) / 4), dim3(256), 0, q, t.N, s.d_K.as<double>(),
                       s.br.dev().n_in, s.has_ext ? s.d_Uext.as<double>() : nullptr, s.d_ctl.as<ScfCtl>(),
                       s.d_U.as<double>(), t.d_U.as<double>(), t.d_Uc());
}

// With part: the tube's equilibrium charge from the plan's partial rows
// (rows r = 0..R-1 of site s at part[r S + s], summed in order from 0.0 as
// the plan's own row sum of at most 16 rows does) into eq, its charge
// Q = (eq + noneq) - rho0 (as combine_charge_kernel) into n_out; without,
// n_out holds Q already.  Then one Broyden update with the step counter on
// the device (the host checks the step limit before each launch), then the
// norms and the plans' status words to the host's read-back record.  Each
// thread forms the Q entries that it reads first in the update.
__global__ __launch_bounds__(kBroydenThreads) void broyden_scf_kernel(int S, double fraction, int norm_type,
                                                                        const double* __restrict__ part, int R,
                                                                        double* __restrict__ eq,
                                                                        const double* __restrict__ neq,
                                                                        const double* __restrict__ rho0,
                                                                        double* n_out, BroydenDev b,
                                                                        ScfCtl* ctl, double max_norm,
                                                                        const int* __restrict__ st_eq,
                                                                        const int* __restrict__ st_neq,
                                                                        ScfBack* __restrict__ back)
{
    if (!ctl->active) return;
    double q = 0.0;  // this thread's last entry of Q: the only one up to kBroydenThreads sites
    if (part) {
        for (int s = threadIdx.x; s < S; s += kBroydenThreads) {
            double e = 0.0;
#pragma unroll 4
            for (int r = 0; r < R; ++r) e += part[(size_t)r * S + s];
            eq[s] = e;
            q = (e + (neq ? neq[s] : 0.0)) - rho0[s];
            n_out[s] = q;
        }
    } else if ((int)threadIdx.x < S) {
        q = n_out[threadIdx.x];
    }
    const int m = ctl->step - 1;
    if (S <= kBroydenThreads)
        broyden_update_small<false>(S, m, fraction, norm_type, q, nullptr, b);
    else
        broyden_update<false>(S, m, fraction, norm_type, n_out, nullptr, b);
    if (threadIdx.x == 0) {   // b.out[0..1] were written by this thread
        const double norm = b.out[0], l2 = b.out[1];
        const int s0 = *st_eq, s1 = st_neq ? *st_neq : 0;
        ctl->step = m + 2;
        // the tests of the host loop: go on while the norm is above max_norm, stop on
        // a norm that is not finite and on a status word that reports an error
        if (!(norm > max_norm) || !isfinite(norm) || !isfinite(l2) || ((s0 | s1) & 2)) ctl->active = 0;
        back += m & 1;
        back->norm = norm;
        back->l2 = l2;
        back->status[0] = s0;
        back->status[1] = s1;
        __threadfence_system();
        __hip_atomic_store(&back->step, m + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Potential, solve, Broyden update and read-back: nothing on the host.
static int scf_enqueue_iteration(Scf& s, hipStream_t q)
{
    Tube& t = *s.tube;
    scf_enqueue_potential(s, q);
    NEGF_HIP_TRY(hipGetLastError());
    // the row sum and the charge go into the Broyden kernel when the plan's
    // own row sum is the in-order one (at most 16 rows)
    const double* part = nullptr;
    int R = 0;
    const bool fuse = t.eq_rows(&part, &R) && R <= 16;
    if (!fuse) part = nullptr;
    int rc = t.enqueue_solve(s.d_Q.as<double>(), q, !fuse, &s.d_ctl.as<ScfCtl>()->active);
    if (rc) return rc;
    hipLaunchKernelGGL(broyden_scf_kernel, dim3(1), dim3(kBroydenThreads), 0, q, s.br.S, s.br.fraction,
                       s.br.norm_type, part, R, t.d_eq.as<double>(),
                       t.neq_status() ? t.d_neq.as<const double>() : nullptr, t.d_rho0.as<const double>(),
                       s.d_Q.as<double>(), s.br.dev(), s.d_ctl.as<ScfCtl>(), s.p.Broyden_max_norm, t.eq_status(),
                       t.neq_status(), static_cast<ScfBack*>(s.d_back));
    NEGF_HIP_TRY(hipGetLastError());
    return NEGF_OK;
}

static bool scf_adaptive_due(const Scf& s, int it)
{
    const Tube& t = *s.tube;
    return t.p.flag_adaptive_integration_limits && it % t.p.integrand_correction_interval == 0;
}

// Launch iteration it (Broyden step step): the host part of the solve first
// (with an adaptive correction due, the integrand is sampled at this
// iteration's potential, enqueued and finished beforehand), then its kernels.
static int scf_launch_iteration(Scf& s, int it, int step)
{
    Tube& t = *s.tube;
    int rc;
    if (scf_adaptive_due(s, it)) {
        scf_enqueue_potential(s, s.st);
        NEGF_HIP_TRY(hipGetLastError());
        NEGF_HIP_TRY(hipStreamSynchronize(s.st));
    }
    if ((rc = t.prepare(it))) return rc;
    ScfBack* back = static_cast<ScfBack*>(s.h_back) + ((step - 1) & 1);
    __atomic_store_n(&back->step, 0, __ATOMIC_RELEASE);  // steps count from 1
    return scf_enqueue_iteration(s, s.st);
}

// Wait for the iteration of the present Broyden step and take its record.
static int scf_collect_iteration(Scf& s, double* norm, double* l2)
{
    const ScfBack* back = static_cast<const ScfBack*>(s.h_back) + ((s.br.step - 1) & 1);
    int rc;
    if ((rc = wait_words(&back->step, 1, s.br.step, s.st))) return rc;
    if (back->status[0] | back->status[1]) {
        // the status words are read and cleared: not under a running iteration
        NEGF_HIP_TRY(hipStreamSynchronize(s.st));
        if ((rc = s.tube->check_status())) return rc;
    }
    const double o[2] = {back->norm, back->l2};
    *norm = o[0];
    *l2 = o[1];
    s.br.step += 1;
    if (!std::isfinite(o[0]) || !std::isfinite(o[1])) {
        set_error("Broyden: non-finite norm");
        return NEGF_ENAN;
    }
    return NEGF_OK;
}

}  // namespace negf

using namespace negf;

struct negf_broyden {
    Broyden b;
    hipStream_t st = nullptr;
};
struct negf_scf {
    Scf s;
};

extern "C" {

int negf_broyden_create(int S, double fraction, int max_step, int norm_type, negf_broyden** out)
{
    clear_error();
    if (!out || S <= 0 || max_step < 0 || (norm_type != 0 && norm_type != 1)) {
        set_error("invalid Broyden arguments");
        return NEGF_EARG;
    }
    negf_broyden* h = new negf_broyden;
    hipError_t e = hipStreamCreate(&h->st);
    if (e != hipSuccess) {
        set_error("hipStreamCreate: %s", hipGetErrorString(e));
        delete h;
        return NEGF_EDEVICE;
    }
    int rc = h->b.init(S, fraction, max_step, norm_type);
    if (rc == NEGF_OK) rc = hipStreamSynchronize(h->st) == hipSuccess ? NEGF_OK : NEGF_EDEVICE;
    if (rc) {
        (void)hipStreamDestroy(h->st);
        delete h;
        return rc;
    }
    *out = h;
    return NEGF_OK;
}

int negf_broyden_destroy(negf_broyden* b)
{
    if (!b) return NEGF_EARG;
    (void)hipStreamSynchronize(b->st);
    (void)hipStreamDestroy(b->st);
    delete b;
    return NEGF_OK;
}

int negf_broyden_set_nin(negf_broyden* b, const double* n_in)
{
    clear_error();
    if (!b || !n_in) {
        set_error("null argument");
        return NEGF_EARG;
    }
    NEGF_HIP_TRY(hipStreamSynchronize(b->st));
    NEGF_HIP_TRY(hipMemcpy(b->b.dev().n_in, n_in, sizeof(double) * b->b.S, hipMemcpyHostToDevice));
    return NEGF_OK;
}

int negf_broyden_get_nin(const negf_broyden* b, double* n_in)
{
    clear_error();
    if (!b || !n_in) {
        set_error("null argument");
        return NEGF_EARG;
    }
    NEGF_HIP_TRY(hipStreamSynchronize(b->st));
    NEGF_HIP_TRY(hipMemcpy(n_in, b->b.dev().n_in, sizeof(double) * b->b.S, hipMemcpyDeviceToHost));
    return NEGF_OK;
}

int negf_broyden_step(negf_broyden* b, const double* n_out, double* max_norm, double* l2, double* norm_per_site)
{
    clear_error();
    if (!b || !n_out) {
        set_error("null argument");
        return NEGF_EARG;
    }
    NEGF_HIP_TRY(hipMemcpyAsync(b->b.d_nout.p, n_out, sizeof(double) * b->b.S, hipMemcpyHostToDevice, b->st));
    int rc = b->b.update(b->b.d_nout.as<double>(), max_norm, l2, b->st);
    if (rc) return rc;
    if (norm_per_site)
        NEGF_HIP_TRY(hipMemcpy(norm_per_site, b->b.dev().Norm, sizeof(double) * b->b.S, hipMemcpyDeviceToHost));
    return NEGF_OK;
}

int negf_broyden_step_device(negf_broyden* b, const double* d_n_out, double* max_norm, double* l2, void* stream)
{
    clear_error();
    if (!b || !d_n_out) {
        set_error("null argument");
        return NEGF_EARG;
    }
    hipStream_t st = stream ? (hipStream_t)stream : b->st;
    return b->b.update(d_n_out, max_norm, l2, st);
}

const double* negf_broyden_device_nin(const negf_broyden* b) { return b ? b->b.dev().n_in : nullptr; }

int negf_broyden_reset(negf_broyden* b, int keep_n_in, double init_value)
{
    clear_error();
    if (!b) {
        set_error("null argument");
        return NEGF_EARG;
    }
    int rc = b->b.reset(keep_n_in, init_value, b->st);
    if (rc) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(b->st));
    return NEGF_OK;
}

int negf_broyden_get_step(const negf_broyden* b) { return b ? b->b.step : -1; }

int negf_scf_create(negf_tube* t, const negf_scf_params* p, negf_scf** out)
{
    clear_error();
    if (!t || !p || !out || p->eps_r <= 0 || p->Broyden_max_norm <= 0 || p->Broyden_threshold_maxstep < 0) {
        set_error("invalid SCF arguments");
        return NEGF_EARG;
    }
    negf_scf* h = new negf_scf;
    Scf& s = h->s;
    s.tube = &t->t;
    s.p = *p;
    const int N = s.tube->N;
    int rc = NEGF_OK;
    hipError_t e = hipStreamCreate(&s.st);
    if (e != hipSuccess) {
        set_error("hipStreamCreate: %s", hipGetErrorString(e));
        delete h;
        return NEGF_EDEVICE;
    }
    coulomb_kernel(s.tube->ptd, s.p, s.K);
    if (!rc) rc = s.d_K.ensure(sizeof(double) * (size_t)N * N);
    if (!rc) rc = s.d_U.ensure(sizeof(double) * N);
    if (!rc) rc = s.d_Q.ensure(sizeof(double) * N);
    if (!rc) rc = s.br.init(N, p->Broyden_fraction, p->Broyden_threshold_maxstep, p->Broyden_norm_type);
    if (!rc) rc = s.d_ctl.ensure(sizeof(ScfCtl));
    if (!rc) {
        hipError_t eh = hipHostMalloc(&s.h_back, 2 * sizeof(ScfBack), hipHostMallocMapped | hipHostMallocCoherent);
        if (eh == hipSuccess) eh = hipHostGetDevicePointer(&s.d_back, s.h_back, 0);
        if (eh != hipSuccess) {
            set_error("mapped host buffer for the SCF read-back: %s", hipGetErrorString(eh));
            rc = NEGF_EALLOC;
        }
    }
    if (!rc) {
        // Set_Broyden_Parallel: n_in starts at the initial deposit value
        rc = s.br.reset(0, p->NS_initial_deposit_value, s.st);
    }
    if (!rc && hipMemcpy(s.d_K.p, s.K.data(), sizeof(double) * s.K.size(), hipMemcpyHostToDevice) != hipSuccess) {
        set_error("hipMemcpy of the electrostatic kernel failed");
        rc = NEGF_EDEVICE;
    }
    if (!rc && hipStreamSynchronize(s.st) != hipSuccess) rc = NEGF_EDEVICE;
    if (rc) {
        delete h;
        return rc;
    }
    *out = h;
    return NEGF_OK;
}

int negf_scf_destroy(negf_scf* s)
{
    if (!s) return NEGF_EARG;
    delete s;
    return NEGF_OK;
}

int negf_scf_kernel(const negf_scf* s, double* K)
{
    clear_error();
    if (!s || !K) {
        set_error("null argument");
        return NEGF_EARG;
    }
    std::copy(s->s.K.begin(), s->s.K.end(), K);
    return NEGF_OK;
}

int negf_scf_use_graph(negf_scf* h, int on)
{
    clear_error();
    if (!h) {
        set_error("null argument");
        return NEGF_EARG;
    }
    h->s.ahead = on != 0;
    return NEGF_OK;
}

int negf_scf_set_external_potential(negf_scf* h, const double* U_ext)
{
    clear_error();
    if (!h) {
        set_error("null argument");
        return NEGF_EARG;
    }
    Scf& s = h->s;
    if (!U_ext) {
        s.has_ext = false;
        return NEGF_OK;
    }
    int rc = s.d_Uext.ensure(sizeof(double) * s.tube->N);
    if (rc) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(s.st));
    NEGF_HIP_TRY(hipMemcpy(s.d_Uext.p, U_ext, sizeof(double) * s.tube->N, hipMemcpyHostToDevice));
    s.has_ext = true;
    return NEGF_OK;
}

// c_TransportSolver::Solve (Transport.cpp:359-539): iterate electrostatics ->
// NEGF -> Broyden until Broyden_Norm <= Broyden_max_norm, then
// Reset_ForNextBiasStep.
int negf_scf_bias_point(negf_scf* h, double V_gate, double* U_out, double* Q_out, int* iters, double* final_norm)
{
    clear_error();
    if (!h || !U_out || !Q_out) {
        set_error("null argument");
        return NEGF_EARG;
    }
    Scf& s = h->s;
    Tube& t = *s.tube;
    const int N = t.N;
    double norm = 1.0, l2 = 0.0;
    int it = 0, rc = NEGF_OK;
    int launched = 0;  // iterations launched ahead
    if (s.ahead) {
        const ScfCtl ctl = {V_gate, s.br.step, 1};
        NEGF_HIP_TRY(hipStreamSynchronize(s.st));
        NEGF_HIP_TRY(hipMemcpy(s.d_ctl.p, &ctl, sizeof(ctl), hipMemcpyHostToDevice));
    }
    do {
        if (s.br.step > s.p.Broyden_threshold_maxstep) {
            set_error("Broyden_Step has exceeded the Broyden_Threshold_MaxStep");
            rc = NEGF_ENONCONV;
            break;
        }
        if (s.ahead) {
            if (launched == it) {
                if ((rc = scf_launch_iteration(s, it, s.br.step))) break;
                ++launched;
            }
            // the next one follows without waiting, where it needs nothing from the host
            if (launched == it + 1 && s.br.step + 1 <= s.p.Broyden_threshold_maxstep && !scf_adaptive_due(s, it + 1)) {
                if ((rc = scf_launch_iteration(s, it + 1, s.br.step + 1))) break;
                ++launched;
            }
            if ((rc = scf_collect_iteration(s, &norm, &l2))) break;
            ++it;
            continue;
        }
        hipLaunchKernelGGL(coulomb_potential_kernel, dim3((N + 3) / 4), dim3(256), 0, s.st, N, s.d_K.as<double>(),
                           s.br.dev().n_in, s.has_ext ? s.d_Uext.as<double>() : nullptr, V_gate,
                           s.d_U.as<double>());
        NEGF_HIP_TRY(hipGetLastError());
        if ((rc = t.set_potential_device(s.d_U.as<double>(), s.st))) break;
        if ((rc = t.solve(it, s.d_Q.as<double>(), s.st))) break;
        if ((rc = s.br.update(s.d_Q.as<double>(), &norm, &l2, s.st))) break;
        if ((rc = t.check_status())) break;
        ++it;
    } while (norm > s.p.Broyden_max_norm);
    NEGF_HIP_TRY(hipStreamSynchronize(s.st));
    NEGF_HIP_TRY(hipMemcpy(U_out, s.d_U.p, sizeof(double) * N, hipMemcpyDeviceToHost));
    NEGF_HIP_TRY(hipMemcpy(Q_out, s.d_Q.p, sizeof(double) * N, hipMemcpyDeviceToHost));
    if (iters) *iters = it;
    if (final_norm) *final_norm = norm;
    if (rc) return rc;
    // Reset_ForNextBiasStep
    if ((rc = s.br.reset(s.p.reset_with_previous_charge_distribution, s.p.NS_initial_deposit_value, s.st))) return rc;
    NEGF_HIP_TRY(hipStreamSynchronize(s.st));
    return NEGF_OK;
}

struct negf_batch_scf {
    BatchScf s;
};

int negf_batch_scf_create(negf_batch* b, negf_tube* const* tubes, int ntubes, const negf_scf_params* p,
                          negf_batch_scf** out)
{
    clear_error();
    if (!b || !tubes || ntubes <= 0 || !p || !out || p->eps_r <= 0 || p->Broyden_max_norm <= 0 ||
        p->Broyden_threshold_maxstep < 0) {
        set_error("invalid batched SCF arguments");
        return NEGF_EARG;
    }
    negf_batch_scf* h = new negf_batch_scf;
    int rc = h->s.init(b, tubes, ntubes, *p);
    if (rc) {
        delete h;
        return rc;
    }
    *out = h;
    return NEGF_OK;
}

int negf_batch_scf_destroy(negf_batch_scf* s)
{
    if (!s) return NEGF_EARG;
    delete s;
    return NEGF_OK;
}

int negf_batch_scf_set_external_potential(negf_batch_scf* s, const double* U_ext)
{
    clear_error();
    if (!s) {
        set_error("null argument");
        return NEGF_EARG;
    }
    // The iterations read d_Uext by address: cleared means zeros.
    BatchScf& b = s->s;
    const long long NT = (long long)b.N * b.T;
    NEGF_HIP_TRY(hipStreamSynchronize(b.st));
    if (!U_ext) {
        int rc = fill_device(b.d_Uext.as<double>(), NT, 0.0, b.st);
        if (rc) return rc;
        NEGF_HIP_TRY(hipStreamSynchronize(b.st));
        b.has_ext = false;
        return NEGF_OK;
    }
    for (long long i = 0; i < NT; ++i)
        if (!std::isfinite(U_ext[i])) {
            set_error("U_ext[%lld] is not finite", i);
            return NEGF_EARG;
        }
    NEGF_HIP_TRY(hipMemcpy(b.d_Uext.p, U_ext, sizeof(double) * NT, hipMemcpyHostToDevice));
    b.has_ext = true;
    return NEGF_OK;
}

int negf_batch_scf_set_input_charge(negf_batch_scf* s, const double* n_in)
{
    clear_error();
    if (!s || !n_in) {
        set_error("null argument");
        return NEGF_EARG;
    }
    BatchScf& b = s->s;
    NEGF_HIP_TRY(hipStreamSynchronize(b.st));
    NEGF_HIP_TRY(hipMemcpy(b.d_KN.p, n_in, sizeof(double) * b.N * b.T, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(batch_charge_rows_kernel<true>, dim3((unsigned)(((long long)b.N * b.T + 255) / 256)),
                       dim3(256), 0, b.st, b.N, b.T, b.d_state.as<double>(), b.state_stride, b.d_KN.as<double>());
    NEGF_HIP_TRY(hipGetLastError());
    return NEGF_OK;
}

int negf_batch_scf_get_input_charge(const negf_batch_scf* s, double* n_in)
{
    clear_error();
    if (!s || !n_in) {
        set_error("null argument");
        return NEGF_EARG;
    }
    const BatchScf& b = s->s;
    hipLaunchKernelGGL(batch_charge_rows_kernel<false>, dim3((unsigned)(((long long)b.N * b.T + 255) / 256)),
                       dim3(256), 0, b.st, b.N, b.T, b.d_state.as<double>(), b.state_stride, b.d_KN.as<double>());
    NEGF_HIP_TRY(hipGetLastError());
    NEGF_HIP_TRY(hipStreamSynchronize(b.st));
    NEGF_HIP_TRY(hipMemcpy(n_in, b.d_KN.p, sizeof(double) * b.N * b.T, hipMemcpyDeviceToHost));
    return NEGF_OK;
}

int negf_batch_scf_use_graph(negf_batch_scf* s, int on)
{
    if (!s) return NEGF_EARG;
    s->s.ahead = on != 0;
    return NEGF_OK;
}

int negf_batch_scf_get_kernel(const negf_batch_scf* s, double* K)
{
    clear_error();
    if (!s || !K) {
        set_error("null argument");
        return NEGF_EARG;
    }
    std::copy(s->s.K.begin(), s->s.K.end(), K);
    return NEGF_OK;
}

int negf_batch_scf_set_preconditioner(negf_batch_scf* s, const double* Z, const double* lam)
{
    clear_error();
    if (!s || !Z || !lam) {
        set_error("null argument");
        return NEGF_EARG;
    }
    return s->s.set_preconditioner(Z, lam);
}

int negf_batch_scf_set_surrogate(negf_batch_scf* s, negf_surrogate* sg, const double* feat)
{
    clear_error();
    if (!s || !sg) {
        set_error("null argument");
        return NEGF_EARG;
    }
    BatchScf& b = s->s;
    if (sg->s.N != b.N) {
        set_error("surrogate has %d sites, the tubes %d", sg->s.N, b.N);
        return NEGF_EARG;
    }
    b.sg = &sg->s;
    b.has_feat = feat != nullptr;
    if (feat) {
        int rc = b.d_feat.ensure(sizeof(double) * b.T);
        if (rc) return rc;
        NEGF_HIP_TRY(hipMemcpy(b.d_feat.p, feat, sizeof(double) * b.T, hipMemcpyHostToDevice));
    }
    return NEGF_OK;
}

int negf_batch_scf_run_surrogate(negf_batch_scf* s, const double* V_gate, int seed_iters, int refresh_iter,
                                 double* U_out, double* Q_out, int* iters, double* final_norms,
                                 int* total_iterations, double* capacitance)
{
    clear_error();
    if (!s || !V_gate || seed_iters < 0) {
        set_error("invalid arguments");
        return NEGF_EARG;
    }
    BatchScf& b = s->s;
    if (!b.sg || !b.has_pc) {
        set_error("set a surrogate and a preconditioner basis first");
        return NEGF_EARG;
    }
    int rc = b.clear_history();
    if (rc) return rc;
    return b.run_pc(V_gate, seed_iters, refresh_iter, U_out, Q_out, iters, final_norms, total_iterations,
                    capacitance);
}

int negf_batch_scf_run(negf_batch_scf* s, const double* V_gate, double* U_out, double* Q_out, int* iters,
                       double* final_norms, int* total_iterations)
{
    clear_error();
    if (!s || !V_gate) {
        set_error("null argument");
        return NEGF_EARG;
    }
    // each run starts a fresh Broyden history (Reset_Broyden_Parallel), keeping n_in
    BatchScf& b = s->s;
    int rc = b.clear_history();
    if (rc) return rc;
    return b.run(V_gate, U_out, Q_out, iters, final_norms, total_iterations);
}

}  // extern "C"
