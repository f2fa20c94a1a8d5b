// score.hip -- per-segment line prologue, sinc^2 reduction and BH+Elwert
// bremsstrahlung on gfx950.
//
// Algorithms follow PyRITE's batched incoherent line route and brem reducer
// (src/pyrite/montecarlo/spectrum/cxr/_batched.py:461-728, cxr/_fused.py,
// cxr/_recoil.py:35-76, cxr_jit_kernel.py:32-613, brem_jit_kernel.py:76-153,
// segment_escape.py:286-300).  Precision policy (MI355X-first):
//  * the prologue (resonance root, couplings, amplitudes, weights) runs in FP64:
//    it is once per line, and keeping the resonance energy E_r and the sinc slope
//    a in FP64 keeps the phase a(E - E_r) exact to ~1e-11 turns;
//  * a reduction cell is [sin(pi u) / (pi u)]^2, u = a(E - E_r)/pi.  In general u is
//    formed in FP64, reduced to r = u - rint(u) in FP64, and the cell taken in FP32
//    (polynomial sine, hardware reciprocal).  On a uniform grid the sines of lines
//    without a bin in their central half period |u| < 1/2 are stepped from bin to
//    bin in FP64 and divided in FP32 by the distance in bins.  Cells are summed in
//    FP32 over groups of 4 lines (all terms are positive) and in FP64 beyond;
//  * the brem cell is FP32 (as the reference's), its sums FP64; of large inputs the
//    cross section is taken from FP32 polynomials that are fitted in FP64.
// Reductions never use atomics: each workgroup writes a partial spectrum and a
// second pass adds the partials in a fixed order, so results are bitwise
// reproducible for a fixed launch shape.
#include <type_traits>
#include <math.h>

#include <mutex>

#include "hr_common.hpp"
#include "line_core.hpp"
#include "math64.hpp"
#include "row_sum.hpp"

namespace hr {
namespace {

using namespace line;

constexpr double kReCm2 = 7.9407877e-26;   // brem.py:63
constexpr double kMc2 = 510.99895;

// Lines of one (segment j, direction d) pair: emit(g, E_r, a, w) for every
// reflection g (w = 0 and E_r = a = 0 for a rejected pair).
template <class Emit>
__device__ __forceinline__ void segment_lines(const hr_line_args &p, int64_t j, int d, Emit &&emit) {
    const double nx = p.n_hat[3 * d], ny = p.n_hat[3 * d + 1], nz = p.n_hat[3 * d + 2];
    const double dir_w = p.dir_weight[d] * p.scale * (p.row_weight ? (double)p.row_weight[j] : 1.0);
    const SegKin k = seg_kin(p.r_mid[3 * j + 2], p.v_hat[3 * j], p.v_hat[3 * j + 1], p.v_hat[3 * j + 2], p.L[j],
                             p.E[j], nx, ny, nz, p.thickness);
    const GridGuess guess = grid_guess(p.E_tab, p.n_tab);
    for (int g = 0; g < p.n_g; ++g) {
        const LineCore o = line_core(p, k, nx, ny, nz, d, g, guess);
        double w = 0.0, a_width = 0.0, Er = 0.0;
        if (o.keep) {
            double A2 = 0.0;
#pragma unroll
            for (int pol = 0; pol < 2; ++pol) A2 += o.A_re[pol] * o.A_re[pol] + o.A_im[pol] * o.A_im[pol];
            // _batched.py:702-728 + _fused.py:267-281, one piece, fraction 1
            const double T_abs = mean_transmission(k.path0 * o.mu, k.path1 * o.mu);
            constexpr double kPref = kAlpha / (4.0 * kPi * kPi * kHbarc);
            const double pref = kPref * o.omega * (k.t_L * k.t_L) * T_abs;
            const double wt = pref * A2 * p.wm[g];
            if (isfinite(wt) && wt > 0.0) {
                w = wt * dir_w;
                a_width = o.slope * k.t_L * (1.0 / (2.0 * kHbarc));
                Er = o.E_res;
            }
        }
        emit(g, Er, a_width, w);
    }
}

// One (segment, direction) pair per thread: writes its n_g lines.
__global__ void __launch_bounds__(256) cxr_lines_kernel(hr_line_args p) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = p.n_seg * (int64_t)p.n_dir;
    if (tid >= total) return;
    const int64_t j = tid % p.n_seg;
    const int d = (int)(tid / p.n_seg);
    const int64_t out0 = ((int64_t)d * p.n_seg + j) * p.n_g;
    segment_lines(p, j, d, [&](int g, double Er, double a_width, double w) {
        p.E_r[out0 + g] = Er;
        p.a[out0 + g] = a_width;
        p.w[out0 + g] = (float)w;
    });
}

// sin(pi r)/pi for |r| <= 1/2 as r P(r^2): an odd polynomial of degree 9 fitted
// to sin(pi r) for minimax relative error on [0, 1/2] (Lawson's iteration of
// weighted least squares on Chebyshev-clustered nodes, fit error 5.3e-9), its
// coefficients divided by pi and rounded to FP32.
constexpr float kSinPiOverPi[5] = {1.0f, -1.6449331045150757f, 0.8117124438285828f, -0.19042645394802094f,
                                   0.024688366800546646f};

// [sin(pi u)/(pi u)]^2 from r = u - rint(u) (|r| <= 1/2) and u in FP32:
// x = r P(r^2) / u with one hardware reciprocal (v_rcp_f32, 1 ulp); maximum
// relative error 5.4e-7 over |u| <= 5e4.  |x| <= 1 in exact arithmetic (the
// central period has u == r, elsewhere |u| >= 1/2), so fminf(x, 1) only trims
// rounding, and at u == 0 (r == 0) it turns 0 * inf = NaN into the limit 1,
// where the reference substitutes x = 1e-20.
__device__ __forceinline__ float sinc_poly(float r) {
    const float r2 = r * r;
    float s = kSinPiOverPi[4];
    s = fmaf(s, r2, kSinPiOverPi[3]);
    s = fmaf(s, r2, kSinPiOverPi[2]);
    s = fmaf(s, r2, kSinPiOverPi[1]);
    return fmaf(s, r2, kSinPiOverPi[0]);
}
__device__ __forceinline__ float sinc2_cell(float r, float uf) {
    const float x = fminf(r * __builtin_amdgcn_rcpf(uf) * sinc_poly(r), 1.0f);
    return x * x;
}

// The same for finite u with r / u = 1 exact where r == u, so that the central half
// period carries the polynomial's rounding alone (root mean square error of a cell
// there 4.9e-8 against 7.4e-8).
__device__ __forceinline__ float sinc2_near(float r, float uf) {
    const float x = (r == uf ? 1.0f : r * __builtin_amdgcn_rcpf(uf)) * sinc_poly(r);
    return x * x;
}

constexpr int kRedThreads = 256;
constexpr int kSincGroup = 4;   // cells summed in FP32 before each FP64 add (all terms >= 0)

// ---- dense sum over a uniform grid E_k = E0 + k dE
//
// A line's profile is w sin^2(pi u)/(pi u)^2 with u = u0 + k du, so along a run of
// bins sin(pi u) obeys s[k+1] = 2 cos(pi du) s[k] - s[k-1]: one FP64 FMA per
// cell instead of a phase, its reduction and a polynomial.  A wave owns a window
// of 64 BINS bins, BINS consecutive ones per lane; per line each lane takes one
// sine and cosine at the middle of its run and steps outward both ways (at most
// BINS/2 steps: the sines stay within 1e-13).  The divisor is the distance in
// bins, d = (k - n) + u(n)/du with n the bin nearest the centre, so it is exact to
// FP32 rounding there; 1/(pi du) rides on the sines.  The weight multiplies the
// square on its own and FP32 groups end with every eighth line of the input, so that
// weighted copies add up to the unweighted sum (a weight of 2 is twice the line).
//
// VALU bound: about 30 SIMD cycles per cell (FP64, conversions and selects issue
// in 4, plain FP32 in 2, the reciprocal in 8) against 52 of a cell with its own
// phase.  2.7e6 lines of 5 MeV electrons (1.47e6 live) on 1024 bins of 48 eV: 600 us
// with a phase per cell, 451 so (about 43 cycles: staging, the lines taken cell by
// cell, FP64 sums and waves of uneven work make the rest).  Lines wider than a bin
// are all taken cell by cell: 1e6 of them on 1024 bins 523 us before, 513 so.
constexpr int kSincWaves = 4;     // waves per block, each with its own lines
constexpr int kSincBlock = 64 * kSincWaves;
constexpr int kSincChunk = 64;    // lines a wave stages at a time (one per lane)

// Mean relative error of v_rcp_f32, all mantissas with the density of a logarithm
// (measured; its root mean square is 2.8e-8).  Left in, it would be 1.3e-8 of a sum
// of many lines.
constexpr double kRcpMean = -6.4e-9;

// sin(pi r)/r and cos(pi r) on |r| <= 1/2 in r^2 (Chebyshev interpolation of
// each; errors 1.6e-13 and 2.0e-15).
constexpr double kSinR[7] = {3.141592653589635, -5.167712779987959, 2.550164035906745, -0.5992644339357286, 0.08214479467064854,
          -0.007364005472115722, 0.0004474920849077101};
constexpr double kCosR[8] = {0.9999999999999981, -4.934802200543686, 4.058712126333295, -1.3352627661817635, 0.23533058831317874,
          -0.025806531975921563, 0.0019278700526981333, -0.0001004164642205389};

template <int N>
__device__ __forceinline__ double horner(const double (&c)[N], double z) {
    double p = c[N - 1];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) p = fma(p, z, c[i]);
    return p;
}

// A staged live line.
struct alignas(16) SincLine {
    double u0, du;    // u = u0 + k du, turns of pi
    double cd, sd;    // cos, sin of pi du
    double q;         // 1 / (pi du), the reciprocal's mean error taken off
    float nf, f, w;   // n - bin0 for the integer n nearest the centre; u(n)/du; w
    int direct;       // no recurrence: see the staging
};

template <int BINS>
__global__ void __launch_bounds__(kSincBlock, 4) sincsq_uniform_kernel(
    const double *__restrict__ E_r, const double *__restrict__ a, const float *__restrict__ w, int64_t n_lines,
    int per, double E0, double dE, int64_t n_E, double *__restrict__ partial) {
    static_assert(BINS % 4 == 0 && BINS >= 4, "runs are stepped outward from their middle");
    constexpr int kWindow = 64 * BINS, kMid = BINS / 2;
    __shared__ SincLine s_line[kSincWaves][kSincChunk];
    __shared__ double s_sum[kWindow];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t bin0 = (int64_t)blockIdx.y * kWindow;
    const int run0 = lane * BINS;                           // first bin of the lane's run, from bin0
    const double kb = (double)(bin0 + run0 + kMid);         // its middle
    const float run0f = (float)run0;
    SincLine *lines = s_line[wave];
    double acc[BINS];
#pragma unroll
    for (int m = 0; m < BINS; ++m) acc[m] = 0.0;
    const double inv_pi = 1.0 / kPi, inv_dE = 1.0 / dE;
    const double first = (double)bin0, last = (double)((bin0 + kWindow < n_E ? bin0 + kWindow : n_E) - 1);
    // the coefficients in scalar registers, from which an FMA reads them directly
    double sin_r[7], cos_r[8];
#pragma unroll
    for (int i = 0; i < 7; ++i) {
        sin_r[i] = kSinR[i];
        asm volatile("" : "+s"(sin_r[i]));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        cos_r[i] = kCosR[i];
        asm volatile("" : "+s"(cos_r[i]));
    }
    const int64_t n_chunks = (n_lines + per - 1) / per;
    for (int64_t c = (int64_t)blockIdx.x * kSincWaves + wave; c < n_chunks; c += (int64_t)gridDim.x * kSincWaves) {
        const int64_t l = c * per + lane;
        // the weight is read first: a zero-weight line (a rejected resonance)
        // costs nothing else, and the live ones are packed to the front
        const float wl = (lane < per && l < n_lines) ? w[l] : 0.0f;
        const uint64_t live = __ballot(wl != 0.0f);
        const int n_live = __popcll(live);
        if (n_live == 0) continue;
        __builtin_amdgcn_wave_barrier();
        if (wl != 0.0f) {
            SincLine o;
            const double al = fabs(a[l]) * inv_pi, er = E_r[l];
            o.u0 = al * (E0 - er);
            o.du = al * dE;
            sincospi(o.du - 2.0 * rint(0.5 * o.du), &o.sd, &o.cd);
            const double inv_du = rcp_nr(o.du);
            o.q = inv_pi * (1.0 - kRcpMean) * inv_du;
            const double n = rint((er - E0) * inv_dE), u = fma(n, o.du, o.u0);
            o.nf = (float)(n - (double)bin0);
            o.f = (float)(u * inv_du);
            o.w = wl;
            // A line with a bin of this window in its central half period takes every
            // cell on its own: there sine and distance vanish together, and the two
            // rounded apart would leave 1.05e-7 a cell (root mean square) where one
            // rounding for both leaves 4.9e-8; elsewhere the stepped cell has 1.05e-7
            // and the one with a phase 1.2e-7.  Lines narrower than a bin, du >> 1,
            // are 1 in du of these (5 % of the lines of 5 MeV electrons on 48 eV bins);
            // those wider than one are all of them.  So are steps too small to divide by.
            const double nearest = fma(fmin(fmax(n, first), last), o.du, o.u0);
            o.direct = !(fabs(o.du) >= 1.0e-250) || !(fabs(nearest) >= 0.5);
            if (!isfinite(fma(first, o.du, o.u0)) || !isfinite(fma(last, o.du, o.u0))) {  // a profile of 1
                o.u0 = 0.0;
                o.du = 0.0;
                o.direct = 1;
            }
            lines[__popcll(live & ((1ULL << lane) - 1ULL))] = o;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint64_t left = live;  // from the eighth line that `stop` belongs to on
        for (int j0 = 0, stop = 0; j0 < n_live;) {
            for (; stop <= j0; left >>= 8) stop += __popcll(left & 0xff);
            float g[BINS];
#pragma unroll
            for (int m = 0; m < BINS; ++m) g[m] = 0.0f;
            const int j1 = j0 + kSincGroup < stop ? j0 + kSincGroup : stop;
#pragma unroll 2
            for (int j = j0; j < j1; ++j) {
                const SincLine &o = lines[j];
                if (__builtin_amdgcn_readfirstlane(o.direct)) {
                    double k = kb - kMid;
                    asm volatile("" : "+v"(k));  // keeps the run's bins out of registers outside this branch
#pragma unroll
                    for (int m = 0; m < BINS; ++m) {
                        const double u = fma(k + m, o.du, o.u0);
                        g[m] = fmaf(o.w, sinc2_near((float)(u - rint(u)), (float)u), g[m]);
                    }
                    continue;
                }
                const double cd = o.cd, c2 = 2.0 * cd, q = o.q;
                const float wl = o.w;
                const double u = fma(kb, o.du, o.u0), r = u - rint(u), z = r * r;
                const double S = (q * r) * horner(sin_r, z), C = q * horner(cos_r, z);
                const float base = run0f - o.nf, f = o.f;
                double up = S, lo = fma(S, cd, -C * o.sd);  // sines at the middle and one bin before
                double up_p = lo, lo_p = up;
#pragma unroll
                for (int i = 0; i < kMid; ++i) {
                    const int mu = kMid + i, ml = kMid - 1 - i;
                    const float xu = (float)up * __builtin_amdgcn_rcpf((base + (float)mu) + f);
                    const float xl = (float)lo * __builtin_amdgcn_rcpf((base + (float)ml) + f);
                    g[mu] = fmaf(wl * xu, xu, g[mu]);
                    g[ml] = fmaf(wl * xl, xl, g[ml]);
                    const double un = fma(c2, up, -up_p), ln = fma(c2, lo, -lo_p);
                    up_p = up;
                    up = un;
                    lo_p = lo;
                    lo = ln;
                }
            }
#pragma unroll
            for (int m = 0; m < BINS; ++m) acc[m] += (double)g[m];
            j0 = j1;
        }
    }
    // the block's partial row: its waves added in order
    for (int v = 0; v < kSincWaves; ++v) {
        if (wave == v) {
#pragma unroll
            for (int m = 0; m < BINS; ++m) s_sum[run0 + m] = v == 0 ? acc[m] : s_sum[run0 + m] + acc[m];
        }
        __syncthreads();
    }
    double *out = partial + (int64_t)blockIdx.x * n_E;
    for (int k = threadIdx.x; k < kWindow && bin0 + k < n_E; k += kSincBlock) out[bin0 + k] = s_sum[k];
}

// General grid: x = a (E_k - E_r) formed in FP64 per cell (E_grid null: the
// degenerate uniform grid E0 + k dE whose step is zero or not finite).  A wave
// evaluates as many of a thread's bins as reach the grid (777 bins: 13 of 16 runs
// of 64), and a block's lines are short tiles from all over the input, since lines
// without weight come in runs.  Bound by vector instructions, 22 a cell, some 60 SIMD
// cycles by their issue (65 measured where most lines live, 114 where a third does).
// The call before (four bins each, 256 lines in a row) and now: 150,000 live
// lines of 320,000 x 777 bins 130 -> 98 us, x 300 128 -> 49, x 1,024 129 -> 111, 38,000
// of 80,000 x 201 bins 75 -> 26, of 1,200 x 777 51 -> 22 (53 with a block to 256 lines).
constexpr int kGeneralTile = 64;
template <int BINS>
__global__ void __launch_bounds__(kRedThreads) sincsq_general_kernel(
    const double *__restrict__ E_r, const double *__restrict__ a, const float *__restrict__ w,
    int64_t n_lines, const double *__restrict__ E_grid, double E0, double dE, int64_t n_E,
    double *__restrict__ partial) {
    __shared__ double s_er[kGeneralTile];
    __shared__ double s_a[kGeneralTile];
    __shared__ float s_w[kGeneralTile];
    const int t = threadIdx.x;
    const int64_t bin0 = (int64_t)blockIdx.y * kRedThreads * BINS;
    double acc[BINS], Ek[BINS];
#pragma unroll
    for (int m = 0; m < BINS; ++m) {
        acc[m] = 0.0;
        const int64_t k = bin0 + t + (int64_t)m * kRedThreads;
        Ek[m] = k < n_E ? (E_grid ? E_grid[k] : E0 + (double)k * dE) : 0.0;
    }
    int runs = 0;  // of the wave's bins
#pragma unroll
    for (int m = 0; m < BINS; ++m) runs += bin0 + (t & ~63) + (int64_t)m * kRedThreads < n_E;
    runs = __builtin_amdgcn_readfirstlane(runs);
    auto lines = [&](auto count) {
        constexpr int N = decltype(count)::value;
        for (int q0 = 0; q0 < kGeneralTile; q0 += kSincGroup) {
            float g[N];
#pragma unroll
            for (int m = 0; m < N; ++m) g[m] = 0.0f;
            for (int q = q0; q < q0 + kSincGroup; ++q) {
                const float wq = s_w[q];
                if (wq == 0.0f) continue;
                const double er = s_er[q], aq = s_a[q];
#pragma unroll
                for (int m = 0; m < N; ++m) {
                    const double u = aq * (Ek[m] - er);
                    const float r = (float)(u - rint(u));
                    g[m] = fmaf(wq, sinc2_cell(r, (float)u), g[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < N; ++m) acc[m] += (double)g[m];
        }
    };
    const double inv_pi = 1.0 / kPi;
    const int64_t n_tiles = (n_lines + kGeneralTile - 1) / kGeneralTile;
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        if (t < kGeneralTile) {
            const int64_t l = tile * kGeneralTile + t;
            const float wl = l < n_lines ? w[l] : 0.0f;  // zero-weight lines: E_r and a not fetched
            s_w[t] = wl;
            s_er[t] = wl != 0.0f ? E_r[l] : 0.0;
            s_a[t] = wl != 0.0f ? a[l] * inv_pi : 0.0;
        }
        __syncthreads();
        static_assert(BINS == 4, "the cases below");
        switch (runs) {
        case 4: lines(std::integral_constant<int, 4>{}); break;
        case 3: lines(std::integral_constant<int, 3>{}); break;
        case 2: lines(std::integral_constant<int, 2>{}); break;
        case 1: lines(std::integral_constant<int, 1>{}); break;
        default: break;
        }
        __syncthreads();
    }
    double *out = partial + (int64_t)blockIdx.x * n_E;
#pragma unroll
    for (int m = 0; m < BINS; ++m) {
        const int64_t k = bin0 + t + (int64_t)m * kRedThreads;
        if (k < n_E) out[k] = acc[m];
    }
}

constexpr float kMc2f = 510.99895f;
constexpr float kInvMc2f = (float)(1.0 / 510.99895);
constexpr double kLog2e = 1.4426950408889634;

// Hardware single-instruction forms (v_rcp_f32, v_sqrt_f32, v_exp_f32): about
// 1 ulp each, against the multi-instruction correctly rounded sequences.
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
constexpr float kLn2f = 0.69314718055994531f;
constexpr double kLn2d = 0.6931471805599453;

// BH+Elwert brem over segment tiles (brem.py:396-423, brem_jit_kernel.py:76-153).
//
// A cell is A g(T, k) e(path, mu_k): the segment's length and weight, the Born
// cross section with its Elwert factors, which depend on the energy and the bin
// alone, and the mean escape.  The kernel is bound by vector instructions, 39 a
// cell.  g is smooth in T away from the spectral tip, so rows of one energy class,
// an eighth of an octave, can take it as a polynomial of degree 6 per bin, through
// seven Chebyshev points of the class evaluated in FP64: 22 instructions a cell.
// The nearest singularity is T = k: a class c +- h with (c - k) >= 8 h interpolates
// to 16^-7 = 4e-9 of g; closer classes (energies below about twice the bin's)
// evaluate every cell.
//
// So the rows are first ordered by class, those that add nothing dropped (a stable
// counting sort: the order, and with it the sum, is fixed), and the polynomials of
// the classes that occur are laid out, 30 us in three launches, where there is enough
// to gain (brem_plan).  Before (one order, four tiles of 128 rows to a block) and now, us:
// 150,000 rows of 0.5..5 MeV x 1,024 bins 234 -> 143 (222 unordered), 150,001 of
// 5 keV..10 MeV x 2,000 with a quarter dead 271 -> 230 (268), 1e6 of 5 keV..5 MeV x
// 1,024 990 -> 720 (976); below the limit 60,000 x 1,024 93 -> 79 (82 ordered),
// 150,000 x 300 125 -> 87 (103), 20,000 x 1,024 92 -> 48.
constexpr int kBremStage = 128;  // rows staged at a time
constexpr int kBremDeg = 6, kBremNodes = kBremDeg + 1;
constexpr double kBremReach = 8.0;
constexpr int64_t kBremSortCells = 100'000'000, kBremSortRows = 20'480, kBremSortBins = 65'536;

// Chebyshev points x_i = cos(pi (2i + 1)/14) of [-1, 1] and, row j, the weights of
// the values there in coefficient j of the polynomial through them.
__constant__ const double kNode[kBremNodes] = {0.97492791218182361, 0.78183148246802981, 0.43388373911755812, 0.0,
                                               -0.43388373911755812, -0.78183148246802981, -0.97492791218182361};
__constant__ const double kNodeWeight[kBremNodes][kBremNodes] = {
    {0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0},
    {0.22824347439014988, -0.79747338888240381, 2.0765213965723364, 0.0, -2.0765213965723364, 0.79747338888240381,
     -0.22824347439014988},
    {0.23411318061389407, -1.0200067492357776, 4.7858935686218833, -8.0, 4.7858935686218833, -1.0200067492357776,
     0.23411318061389407},
    {-1.5858139578511551, 5.0751495106189253, -5.5818117994536827, 0.0, 5.5818117994536827, -5.0751495106189253,
     1.5858139578511551},
    {-1.6265961185809208, 6.4913598702856729, -12.864763751704752, 16.0, -12.864763751704752, 6.4913598702856729,
     -1.6265961185809208},
    {1.9834685216802656, -4.4568133128311934, 3.5740867769967075, 0.0, -3.5740867769967075, 4.4568133128311934,
     -1.9834685216802656},
    {2.0344771104577316, -5.7004781884227062, 8.2374296493935458, -9.1428571428571423, 8.2374296493935458,
     -5.7004781884227062, 2.0344771104577316}};

// Energy class of a row: eight to an octave from 1/4 keV up (the exponent and top
// three mantissa bits), the last for rows that add nothing.
constexpr int kBremClasses = 128;
constexpr uint32_t kBremClass0 = 0x3e800000u >> 20;

// Centre and half width of a class, and whether its rows may take polynomials up
// to photon energy k_hi (the first and last classes are open ended).
struct BremBand {
    double c, h;
    __device__ __forceinline__ explicit BremBand(int cls) {
        const double lo = __uint_as_float((kBremClass0 + cls) << 20), hi = __uint_as_float((kBremClass0 + cls + 1) << 20);
        c = 0.5 * (lo + hi);
        h = 0.5 * (hi - lo);
    }
    __device__ __forceinline__ static bool closed(int cls) { return cls > 0 && cls < kBremClasses - 2; }
    __device__ __forceinline__ bool reaches(double k) const { return c - k >= kBremReach * h; }
};

__device__ __forceinline__ int brem_class(float T, float L, float w) {
    if ((double)w * (double)L == 0.0) return kBremClasses - 1;
    const int c = (int)(__float_as_uint(fmaxf(T, 0.25f)) >> 20) - (int)kBremClass0;
    return c < 0 ? 0 : (c > kBremClasses - 2 ? kBremClasses - 2 : c);
}

// The wave's class counts (kScatter false), or its rows written where `at` says
// the next row of each class goes: rows [b per, (b + 1) per) of wave b.
template <bool kScatter>
__device__ __forceinline__ void brem_order(const hr_brem_args &p, int64_t per, int64_t b, uint32_t *s_at,
                                           uint32_t *__restrict__ order) {
    const int lane = threadIdx.x;
    const int64_t end = (b + 1) * per < p.n_seg ? (b + 1) * per : p.n_seg;
    for (int64_t j0 = b * per; j0 < end; j0 += 64) {
        const int64_t j = j0 + lane;
        const bool in = j < end;
        const int c = in ? brem_class(p.E_keV[j], p.L[j], p.row_weight ? p.row_weight[j] : 1.0f) : 0;
        uint64_t same = __ballot(in);  // the lanes of this lane's class
#pragma unroll
        for (int bit = 0; bit < 7; ++bit) {
            const uint64_t set = __ballot((c >> bit) & 1);
            same &= ((c >> bit) & 1) ? set : ~set;
        }
        const uint32_t rank = (uint32_t)__popcll(same & ((1ULL << lane) - 1ULL));
        const uint32_t at = in ? s_at[c] : 0u;
        __syncthreads();
        if (in && kScatter) order[at + rank] = (uint32_t)j;
        if (in && rank == 0) s_at[c] = at + (uint32_t)__popcll(same);
        __syncthreads();
    }
}

// counts[class][wave]
__global__ void __launch_bounds__(64) brem_count_kernel(hr_brem_args p, int64_t per, uint32_t *__restrict__ counts) {
    __shared__ uint32_t s_at[kBremClasses];
    for (int c = threadIdx.x; c < kBremClasses; c += 64) s_at[c] = 0u;
    __syncthreads();
    brem_order<false>(p, per, blockIdx.x, s_at, nullptr);
    for (int c = threadIdx.x; c < kBremClasses; c += 64) counts[c * (int64_t)gridDim.x + blockIdx.x] = s_at[c];
}

// Exclusive sums over the waves of each class, and the classes' totals.  One wave per class.
__global__ void __launch_bounds__(64) brem_scan_kernel(uint32_t *__restrict__ counts, int64_t waves,
                                                       uint32_t *__restrict__ totals) {
    uint32_t *C = counts + blockIdx.x * waves;
    const int lane = threadIdx.x;
    uint32_t sum = 0;
    for (int64_t i0 = 0; i0 < waves; i0 += 64) {
        const uint32_t v = i0 + lane < waves ? C[i0 + lane] : 0u;
        uint32_t incl = v;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const uint32_t up = __shfl_up(incl, d);
            incl += lane >= d ? up : 0u;
        }
        if (i0 + lane < waves) C[i0 + lane] = sum + incl - v;
        sum += __shfl(incl, 63);
    }
    if (lane == 0) totals[blockIdx.x] = sum;
}

// Exclusive sums of f(total) over the classes, by one wave; the whole sum in [kBremClasses].
template <class F>
__device__ __forceinline__ void brem_class_sums(const uint32_t *__restrict__ totals, uint32_t *out, F f) {
    const int lane = __lane_id();
    const uint32_t a = f(totals[2 * lane]), b = f(totals[2 * lane + 1]);
    uint32_t incl = a + b;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const uint32_t up = __shfl_up(incl, d);
        incl += lane >= d ? up : 0u;
    }
    out[2 * lane] = incl - a - b;
    out[2 * lane + 1] = incl - b;
    if (lane == 63) out[kBremClasses] = incl;
}

// The first `waves` blocks write the rows in class order; the others, eight bins of
// one class each, lay out the polynomials of g in the place of T within its class,
// poly[class][power][bin], for the classes that occur and the bins they reach: one
// lane per node and bin.
constexpr int kBremPolyBins = 8;
__global__ void __launch_bounds__(64) brem_lay_kernel(hr_brem_args p, int64_t per, int64_t waves,
                                                      const uint32_t *__restrict__ counts,
                                                      const uint32_t *__restrict__ totals,
                                                      uint32_t *__restrict__ order, float *__restrict__ poly) {
    __shared__ uint32_t s_at[kBremClasses + 1];
    const int lane = threadIdx.x;
    if (blockIdx.x < waves) {
        brem_class_sums(totals, s_at, [](uint32_t n) { return n; });
        __syncthreads();
        for (int c = lane; c < kBremClasses; c += 64) s_at[c] += counts[c * waves + blockIdx.x];
        __syncthreads();
        brem_order<true>(p, per, blockIdx.x, s_at, order);
        return;
    }
    const int64_t groups = (p.n_E + kBremPolyBins - 1) / kBremPolyBins, at = blockIdx.x - waves;
    const int cls = (int)(at / groups);
    const int node = lane / kBremPolyBins;
    const int64_t k = at % groups * kBremPolyBins + lane % kBremPolyBins;
    if (!BremBand::closed(cls) || totals[cls] == 0) return;
    const BremBand band(cls);
    const double kev = k < p.n_E ? p.E_grid_eV[k] * 1.0e-3 : 0.0;
    double v = 0.0;
    if (kev > 0.0 && band.reaches(kev) && node < kBremNodes) {
        const double T = band.c + band.h * kNode[node], Tf = T - kev, Tm = Tf + 2.0 * kMc2;
        const double pi_ = sqrt_nr(T * (T + 2.0 * kMc2)) * (1.0 / kMc2);
        const double inv_bi = (1.0 + T * (1.0 / kMc2)) * rcp_nr(pi_);
        const double TT = Tf * Tm, rs = rsqrt_nr(TT), spf = pi_ + TT * rs * (1.0 / kMc2);
        const double rcp_bf = rs * (kMc2 + Tf);
        const double born = ln(spf * spf * (kMc2 * kMc2) * rcp_nr(kev * (T + Tm)));
        double sum = 0.0;
        for (int el = 0; el < p.n_el; ++el) {
            // n (16/3) alpha r_e^2 Z^2 beta_i (1 - exp(-2 pi Z alpha/beta_i)) / (1 - exp(-2 pi Z alpha/beta_f))
            const double z = 2.0 * kPi * kAlpha * p.Z[el];
            sum += p.n_cm3[el] * p.Z[el] * p.Z[el] * (1.0 - exp_any(-z * inv_bi)) * rcp_nr(1.0 - exp_any(-z * rcp_bf));
        }
        const double front = (16.0 / 3.0) * kAlpha * kReCm2 * rcp_nr(pi_ * pi_ * inv_bi * (kev * 1.0e3));
        v = front * born * rcp_bf * sum;
    }
    double coef = 0.0;
#pragma unroll
    for (int i = 0; i < kBremNodes; ++i)
        coef += kNodeWeight[node < kBremNodes ? node : 0][i] * __shfl(v, i * kBremPolyBins + lane % kBremPolyBins);
    if (k < p.n_E && node < kBremNodes) poly[((int64_t)cls * kBremNodes + node) * p.n_E + k] = (float)coef;
}

// The rows of a tile: `rows` rows of one class where the rows are in class order,
// of all rows as they lie where not.
struct BremOrder {
    const uint32_t *order, *totals;  // rows in class order; rows of each class
    const float *poly;
};

struct BremTile {
    int64_t r0, r1;
    int cls;    // -1 without the order
    bool band;  // rows that take the polynomials in this window of bins
};

struct BremShared {
    uint32_t tile[kBremClasses + 1], first[kBremClasses + 1];  // of each class: first tile, first row
    float k_max[kRedThreads / 64];
};

// Tile blockIdx.x of the window whose bins end at k_hi [keV] (this thread's bins;
// the block's are joined here).
template <bool kOrdered>
__device__ __forceinline__ BremTile brem_tile(const hr_brem_args &p, int64_t rows, const BremOrder &o, float k_hi,
                                              BremShared &sh) {
    const int t = threadIdx.x;
    const int64_t tile = blockIdx.x;
    if (!kOrdered) {
        const int64_t r0 = tile * rows;
        return {r0, r0 + rows < p.n_seg ? r0 + rows : p.n_seg, -1, false};
    }
    if (t < 64) brem_class_sums(o.totals, sh.first, [](uint32_t n) { return n; });
    else if (t < 128)
        brem_class_sums(o.totals, sh.tile, [rows](uint32_t n) { return (uint32_t)((n + rows - 1) / rows); });
#pragma unroll
    for (int d = 32; d > 0; d /= 2) k_hi = fmaxf(k_hi, __shfl_xor(k_hi, d));
    if ((t & 63) == 0) sh.k_max[t >> 6] = k_hi;
    __syncthreads();
    k_hi = fmaxf(fmaxf(sh.k_max[0], sh.k_max[1]), fmaxf(sh.k_max[2], sh.k_max[3]));
    if (tile >= (int64_t)sh.tile[kBremClasses - 1]) return {0, 0, -1, false};
    int lo = 0, hi = kBremClasses - 2;  // the last class that starts by this tile holds it
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int64_t)sh.tile[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    const int64_t r0 = (int64_t)sh.first[lo] + (tile - sh.tile[lo]) * rows, end = sh.first[lo + 1];
    return {r0, r0 + rows < end ? r0 + rows : end, lo, BremBand::closed(lo) && BremBand(lo).reaches((double)k_hi)};
}

// Length of segment j with its weight, and the shorter and longer of its escape paths:
// from its two ends along n_hat (segment_escape.py:190-211).
struct BremRow {
    double wL, plo, phi;
    __device__ __forceinline__ BremRow(const hr_brem_args &p, int64_t j) {
        const double L = (double)p.L[j], half = 0.5 * L;
        wL = (p.row_weight ? (double)p.row_weight[j] : 1.0) * L;
        const double rz = p.r_mid[3 * j + 2], vz = p.v_hat[3 * j + 2];
        const double p0 = slab_path(rz - half * vz, p.thickness, p.n_hat[2]);
        const double p1 = slab_path(rz + half * vz, p.thickness, p.n_hat[2]);
        plo = fmin(p0, p1);
        phi = fmax(p0, p1);
    }
};

constexpr int kBremGroup = 8;  // cells summed in FP32 (positive terms: rounding below 5e-7) before each FP64 add

// Tile blockIdx.x of window blockIdx.y, to its partial row; thread t owns bins
// t + kRedThreads m of the window.
// NEL: element count of the composition (1..4), a template parameter so the
// per-element loop unrolls with its constants in registers.
template <int BINS, int NEL, bool kOrdered>
__global__ void __launch_bounds__(kRedThreads, kOrdered && NEL == 4 ? 3 : 4) brem_kernel(hr_brem_args p, int64_t rows, BremOrder o,
                                                              double *__restrict__ partial) {
    // per staged segment: kinetic energy (its place in the class), momentum (length
    // times weight, 1e-8 L w), the shorter and longer escape paths, their mean and
    // difference; of rows evaluated cell by cell also the per-element prefactors and
    // whether any of them is nonzero
    __shared__ float s_T[kBremStage], s_pi[kBremStage], s_plo[kBremStage], s_phi[kBremStage], s_pmid[kBremStage],
        s_dp[kBremStage];
    __shared__ float s_pref[kBremStage * 4];
    __shared__ int s_live[kBremStage];
    __shared__ BremShared sh;
    const int t = threadIdx.x;
    const int64_t bin0 = (int64_t)blockIdx.y * kRedThreads * BINS;
    constexpr int n_el = NEL;
    double acc[BINS];
    // per-bin constants: k [keV], k / m^2 [1/keV], ln 2 / k [1/eV], mu, mu log2(e)
    float keV[BINS], k_m2[BINS], ln2_inv_k[BINS], mu[BINS], mu2[BINS];
    float k_hi = 0.0f;
#pragma unroll
    for (int m = 0; m < BINS; ++m) {
        acc[m] = 0.0;
        const int64_t k = bin0 + t + (int64_t)m * kRedThreads;
        const double kev = k < p.n_E ? p.E_grid_eV[k] : 0.0;
        keV[m] = (float)(kev * 1.0e-3);
        k_m2[m] = (float)(kev * 1.0e-3 / (kMc2 * kMc2));
        ln2_inv_k[m] = (float)(kLn2d / fmax(kev, 1.0e-30));
        mu[m] = kev > 0.0 ? p.mu[k] : 0.0f;  // no cell otherwise
        mu2[m] = (float)((double)mu[m] * kLog2e);
        k_hi = fmaxf(k_hi, keV[m] * (1.0f + 1.0e-6f));
    }
    const BremTile tile = brem_tile<kOrdered>(p, rows, o, k_hi, sh);
    float g[BINS][kBremNodes];
    double c = 0.0, inv_h = 0.0;
    if (kOrdered && tile.band) {
        const BremBand band(tile.cls);
        c = band.c;
        inv_h = 1.0 / band.h;
#pragma unroll
        for (int m = 0; m < BINS; ++m) {
            const int64_t k = bin0 + t + (int64_t)m * kRedThreads;
#pragma unroll
            for (int i = 0; i < kBremNodes; ++i)
                g[m][i] = k < p.n_E ? o.poly[((int64_t)tile.cls * kBremNodes + i) * p.n_E + k] : 0.0f;
        }
    }
    float zi2[4];
    for (int el = 0; el < 4; ++el)  // exp(-2 pi Z alpha / beta) = exp2(-(2 pi Z alpha log2 e) / beta)
        zi2[el] = el < n_el ? (float)(2.0 * kPi * p.Z[el] * kAlpha * kLog2e) : 0.0f;
    for (int64_t s0 = tile.r0; s0 < tile.r1; s0 += kBremStage) {
        const int cnt = (int)(tile.r1 - s0 < kBremStage ? tile.r1 - s0 : kBremStage);
        __syncthreads();
        if (t < cnt) {
            const int64_t j = kOrdered ? (int64_t)o.order[s0 + t] : s0 + t;
            const BremRow row(p, j);
            const float T = p.E_keV[j];
            s_plo[t] = (float)row.plo;
            s_phi[t] = (float)row.phi;
            s_pmid[t] = (float)(0.5 * (row.plo + row.phi));
            s_dp[t] = (float)(row.phi - row.plo);
            if (kOrdered && tile.band) {
                s_T[t] = (float)(((double)T - c) * inv_h);
                s_pi[t] = (float)(row.wL * 1.0e-8);
            } else {
                const float pi_ = sqrtf(T * (T + 2.0f * (float)kMc2)) / (float)kMc2;
                const float bi = pi_ / (1.0f + T / (float)kMc2);
                s_T[t] = T;
                s_pi[t] = pi_;
                int live = 0;
                for (int el = 0; el < n_el; ++el) {
                    // n L 1e-8 (16/3) alpha r_e^2 Z^2 beta_i (1 - exp(-2 pi Z alpha/beta_i)) / p_i^2
                    const double den_i = 1.0 - exp(-2.0 * kPi * p.Z[el] * kAlpha / (double)bi);
                    const float pref =
                        (float)(row.wL * p.n_cm3[el] * 1.0e-8 * (16.0 / 3.0) * kAlpha * kReCm2 * p.Z[el] * p.Z[el] *
                                (double)bi * den_i / ((double)pi_ * (double)pi_));
                    s_pref[t * 4 + el] = pref;
                    live |= pref != 0.0f;
                }
                s_live[t] = live;
            }
        }
        __syncthreads();
        float part[BINS];
#pragma unroll
        for (int m = 0; m < BINS; ++m) part[m] = 0.0f;
        for (int q = 0; q < cnt; ++q) {
            if ((q & (kBremGroup - 1)) == 0 && q > 0) {
#pragma unroll
                for (int m = 0; m < BINS; ++m) {
                    acc[m] += (double)part[m];
                    part[m] = 0.0f;
                }
            }
            const float plo = s_plo[q], phi = s_phi[q], pmid = s_pmid[q], dp = s_dp[q];
            if (kOrdered && tile.band) {
                const float x = s_T[q], wL = s_pi[q];
#pragma unroll
                for (int m = 0; m < BINS; ++m) {
                    float v = g[m][kBremDeg];
#pragma unroll
                    for (int i = kBremDeg - 1; i >= 0; --i) v = fmaf(v, x, g[m][i]);
                    v *= wL;
                    const float d = dp * mu[m];  // the escape as below
                    if (d > 1.0f) {
                        v *= fast_rcp(d);
                        part[m] = fmaf(v, fast_exp2(-plo * mu2[m]) - fast_exp2(-phi * mu2[m]), part[m]);
                    } else {
                        const float x2 = 0.25f * d * d;
                        v *= fmaf(x2, fmaf(x2, fmaf(x2, 1.0f / 5040, 1.0f / 120), 1.0f / 6), 1.0f);
                        part[m] = fmaf(v, fast_exp2(-pmid * mu2[m]), part[m]);
                    }
                }
                continue;
            }
            // a zero-weight row (a copy that does not carry this tally) adds nothing
            if (!s_live[q]) continue;
            const float T = s_T[q], pi_ = s_pi[q];
#pragma unroll
            for (int m = 0; m < BINS; ++m) {
                const float Tf = T - keV[m];
                if (!(Tf > 1.0e-6f) || !(keV[m] > 0.0f)) continue;
                const float Tm = Tf + 2.0f * kMc2f;
                // p_f m = sqrt(T_f (T_f + 2m)) and 1/beta_f = (m + T_f) / (p_f m), from one v_rsq_f32
                const float TT = Tf * Tm;
                const float rs = fast_rsq(TT);
                const float pf = TT * rs * kInvMc2f;
                const float rcp_bf = rs * (kMc2f + Tf);
                // ln((p_i + p_f)^2 m^2 / (k (T_i + T_f + 2m))) = ln((p_i + p_f)/(p_i - p_f)): the
                // difference form has no cancellation for k << T_i; the argument is >= 1 up to
                // rounding (no denormal path in the hardware log2); ln 2 / k is folded per bin
                const float spf = pi_ + pf;
                const float born_k = fast_log2(spf * spf * fast_rcp(k_m2[m] * (T + Tm))) * ln2_inv_k[m];
                // Elwert factors sum_el pref_el / (1 - exp(-2 pi Z_el alpha / beta_f)) as one
                // fraction num / den
                float num = s_pref[q * 4];
                float den = 1.0f - fast_exp2(-zi2[0] * rcp_bf);
#pragma unroll
                for (int el = 1; el < n_el; ++el) {
                    const float d_el = 1.0f - fast_exp2(-zi2[el] * rcp_bf);
                    num = fmaf(num, d_el, s_pref[q * 4 + el] * den);
                    den *= d_el;
                }
                // segment-mean escape (exp(-p_lo mu) - exp(-p_hi mu)) / d, d = (p_hi - p_lo) mu;
                // for d <= 1 as exp(-p_mid mu) sinh(d/2)/(d/2), the series truncated after
                // (d/2)^6 / 7! (remainder < 3e-8 relative)
                const float d = dp * mu[m];
                float esc;
                if (d > 1.0f) {
                    esc = fast_exp2(-plo * mu2[m]) - fast_exp2(-phi * mu2[m]);
                    den *= d;
                } else {
                    const float x2 = 0.25f * d * d;
                    const float shc = fmaf(x2, fmaf(x2, fmaf(x2, 1.0f / 5040, 1.0f / 120), 1.0f / 6), 1.0f);
                    esc = fast_exp2(-pmid * mu2[m]) * shc;
                }
                part[m] = fmaf(num * born_k * rcp_bf * esc, fast_rcp(den), part[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < BINS; ++m) acc[m] += (double)part[m];
    }
    double *out = partial + (int64_t)blockIdx.x * p.n_E;
#pragma unroll
    for (int m = 0; m < BINS; ++m) {
        const int64_t k = bin0 + t + (int64_t)m * kRedThreads;
        if (k < p.n_E) out[k] = acc[m];
    }
}

// ---- support-windowed reduction with the cycle-averaged far tail
// (spectrum/cxr/_node_window.py:86-250 NodeTail / row_window_plan,
// :454-522 _sincsq_window_reduce).  A line deposits its exact sinc^2 on the
// bins within |a (E - E_r)| <= x_c (minus the tail there) and three tail
// moments (m2, m3, m4) = w (1, 2 eps, 3 eps^2) / (2 a^2) at its node; a second
// pass adds sum_node m2/x^2 + m3/x^3 + m4/x^4 everywhere.  Broad windows (a
// quarter of the grid or more) and nodes outside [-n, 2n) are summed exactly
// over the whole grid.  Per-direction spectra and in-grid moments live in LDS
// (FP64 atomics); out-of-grid moments go to global memory.
// Threads per window workgroup (one workgroup per CU: the spectrum and moments
// fill its LDS); a tuning build may set HR_WINDOW_THREADS.
#ifndef HR_WINDOW_THREADS
#define HR_WINDOW_THREADS 1024
#endif
constexpr int kWinThreads = HR_WINDOW_THREADS;
constexpr int kWinMaxBins = 4096;

struct WindowItem {
    double Er, a, w;
};

struct WindowShared {
    double spec[kWinMaxBins];
    double dep[3][kWinMaxBins];
    WindowItem queue[kWinThreads / 64][64];  // each wave's lines of longer windows
};
static_assert(sizeof(WindowShared) <= 160 * 1024, "window LDS");

__device__ __forceinline__ double tail_value(double m2, double m3, double m4, double x) {
    const double inv = rcp_nr(x);
    return (m2 + (m3 + m4 * inv) * inv) * inv * inv;
}

// Exact cell of the dense reducer at u = a (E - E_r) / pi (FP64 phase, FP32 profile).
__device__ __forceinline__ double sincsq_cell(double u) {
    return (double)sinc2_cell((float)(u - rint(u)), (float)u);
}

struct WindowGrid {
    int64_t n;
    double E0, dE, x_c, inv_dE;
};

// Where a line deposits: bins [lo, hi] exactly, the tail moments at its node
// where `conv` (a window of less than a quarter of the grid, node in reach).
struct WindowPlan {
    double Er, al, m2, m3, m4;  // al = a/pi
    int64_t node, lo, hi;
    bool conv;
};

__device__ __forceinline__ WindowPlan window_plan(const WindowGrid &G, double Er, double a) {
    const int64_t n = G.n;
    WindowPlan P;
    P.Er = Er;
    P.al = a * (1.0 / kPi);
    // quotients rounded as divisions: they decide the line's node and reach
    const double inv_a = rcp_nr(a);
    const double nd = rint(div_by(Er - G.E0, G.dE, G.inv_dE));
    const double eps = Er - (G.E0 + nd * G.dE);
    double R = ceil(div_by(fabs(eps) + div_by(G.x_c, a, inv_a), G.dE, G.inv_dE));
    R = fmin(R, 4503599627370496.0);
    P.node = (int64_t)nd;
    P.lo = 0;
    P.hi = n - 1;
    P.conv = false;
    if (P.node + n >= 0 && P.node + n < 3 * n) {
        const int64_t RR = (int64_t)R;
        const int64_t l = P.node - RR < 0 ? 0 : P.node - RR;
        const int64_t h = P.node + RR > n - 1 ? n - 1 : P.node + RR;
        if ((double)(h - l + 1) < 0.25 * (double)n) {
            P.lo = l;
            P.hi = h;
            P.conv = true;
        }
    }
    P.m2 = 0.5 * inv_a * inv_a;
    P.m3 = 2.0 * eps * P.m2;
    P.m4 = 3.0 * eps * eps * P.m2;
    return P;
}

// Bins lo + first, lo + first + step, ... of a line's window.
__device__ __forceinline__ void window_cells(WindowShared &sh, const WindowGrid &G, const WindowPlan &P, double w,
                                             int first, int step) {
    for (int64_t e = P.lo + first; e <= P.hi; e += step) {
        double v = sincsq_cell(P.al * ((G.E0 + (double)e * G.dE) - P.Er));
        if (P.conv && e != P.node) v -= tail_value(P.m2, P.m3, P.m4, (double)(e - P.node) * G.dE);
        atomicAdd(&sh.spec[e], w * v);
    }
}

__device__ __forceinline__ void window_moments(WindowShared &sh, double *__restrict__ dep_far, const WindowGrid &G,
                                               const WindowPlan &P, double w) {
    const int64_t n = G.n, node = P.node;
    if (node >= 0 && node < n) {
        atomicAdd(&sh.dep[0][node], w * P.m2);
        atomicAdd(&sh.dep[1][node], w * P.m3);
        atomicAdd(&sh.dep[2][node], w * P.m4);
    } else {
        const int64_t L = 3 * n;
        atomicAdd(&dep_far[node + n], w * P.m2);
        atomicAdd(&dep_far[L + node + n], w * P.m3);
        atomicAdd(&dep_far[2 * L + node + n], w * P.m4);
    }
}

// Deposits one line per lane (w == 0: none); every lane of the wave takes part.
// A window's length goes as 1/L: most lines cover a few bins, one in hundreds the
// whole grid, and a lane that walked its own held the other 63 up (12,007
// segments x 64 reflections x 64 rays: 5.6 to 35 ms by the draw of lengths, 1.9
// to 2.1 so).  Windows of up to kOwnCells bins stay with their lane; longer ones
// go through the wave's queue, four at a time to 16 lanes each, and those above
// kGroupCells to the whole wave.
constexpr int kOwnCells = 8, kGroupCells = 128, kGroupLanes = 16;

__device__ __forceinline__ void window_deposit(WindowShared &sh, double *__restrict__ dep_far,
                                               const WindowGrid &G, double Er, double a, float wf) {
    const int lane = __lane_id();
    WindowItem *queue = sh.queue[threadIdx.x >> 6];
    const double w = (double)wf;
    const bool live = wf != 0.0f && a > 0.0;
    int64_t cells = 0;
    if (live) {
        const WindowPlan P = window_plan(G, Er, a);
        cells = P.hi - P.lo + 1;
        if (P.conv) window_moments(sh, dep_far, G, P, w);
        if (cells <= kOwnCells) window_cells(sh, G, P, w, 0, 1);
    }
    const uint64_t queued = __ballot(cells > kOwnCells);
    if (queued == 0) return;
    uint64_t wide = __ballot(cells > kGroupCells);
    const int n = __popcll(queued);
    __builtin_amdgcn_wave_barrier();
    if (cells > kOwnCells) queue[__popcll(queued & ((1ULL << lane) - 1ULL))] = WindowItem{Er, a, w};
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int i = lane / kGroupLanes; i < n; i += 64 / kGroupLanes) {
        const WindowItem it = queue[i];
        const WindowPlan P = window_plan(G, it.Er, it.a);
        if (P.hi - P.lo + 1 <= kGroupCells) window_cells(sh, G, P, it.w, lane % kGroupLanes, kGroupLanes);
    }
    while (wide != 0) {
        const int l = __ffsll((unsigned long long)wide) - 1;
        wide &= wide - 1;
        const WindowItem it = queue[__popcll(queued & ((1ULL << l) - 1ULL))];
        window_cells(sh, G, window_plan(G, it.Er, it.a), it.w, lane, 64);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void window_zero(WindowShared &sh, int64_t n) {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        sh.spec[i] = 0.0;
        sh.dep[0][i] = 0.0;
        sh.dep[1][i] = 0.0;
        sh.dep[2][i] = 0.0;
    }
}

// Block partial: [spec | m2 | m3 | m4] over the grid.
__device__ __forceinline__ void window_flush(const WindowShared &sh, int64_t n, double *__restrict__ out) {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        out[i] = sh.spec[i];
        out[n + i] = sh.dep[0][i];
        out[2 * n + i] = sh.dep[1][i];
        out[3 * n + i] = sh.dep[2][i];
    }
}

// Segments [chunk share) x direction blockIdx.y: prologue fused with the window deposit.
__global__ void __launch_bounds__(kWinThreads) window_lines_kernel(hr_line_args p, WindowGrid G,
                                                                   double *__restrict__ partial,
                                                                   double *__restrict__ dep_far) {
    __shared__ WindowShared sh;
    const int d = blockIdx.y;
    window_zero(sh, G.n);
    __syncthreads();
    const int64_t per = (p.n_seg + gridDim.x - 1) / gridDim.x;
    const int64_t j0 = (int64_t)blockIdx.x * per;
    const int64_t j1 = j0 + per < p.n_seg ? j0 + per : p.n_seg;
    double *far = dep_far + (int64_t)d * 9 * G.n;
    // whole waves: the lanes past the end carry the last segment without weight
    for (int64_t jw = j0 + (threadIdx.x & ~63); jw < j1; jw += blockDim.x) {
        const int64_t j = jw + (threadIdx.x & 63);
        segment_lines(p, j < j1 ? j : j1 - 1, d, [&](int, double Er, double a_width, double w64) {
            // the line weight the dense route stores
            window_deposit(sh, far, G, Er, a_width, j < j1 ? (float)w64 : 0.0f);
        });
    }
    __syncthreads();
    window_flush(sh, G.n, partial + ((int64_t)d * gridDim.x + blockIdx.x) * 4 * G.n);
}

// Given lines (one target): the windowed counterpart of hr_sincsq_reduce.
__global__ void __launch_bounds__(kWinThreads) window_given_kernel(const double *__restrict__ E_r,
                                                                   const double *__restrict__ a,
                                                                   const float *__restrict__ w, int64_t n_lines,
                                                                   WindowGrid G, double *__restrict__ partial,
                                                                   double *__restrict__ dep_far) {
    __shared__ WindowShared sh;
    window_zero(sh, G.n);
    __syncthreads();
    for (int64_t lw = (int64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63); lw < n_lines;
         lw += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = lw + (threadIdx.x & 63);
        const float wf = l < n_lines ? w[l] : 0.0f;
        window_deposit(sh, dep_far, G, wf != 0.0f ? E_r[l] : 0.0, wf != 0.0f ? a[l] : 0.0, wf);
    }
    __syncthreads();
    window_flush(sh, G.n, partial + (int64_t)blockIdx.x * 4 * G.n);
}

// Sum the block partials of each direction in a fixed order; spectra to spec,
// in-grid moments to the node slots [n, 2n) of the moment array.
__global__ void __launch_bounds__(256) window_sum_kernel(const double *__restrict__ partial, int64_t n_blocks,
                                                         int64_t n, int n_dir, double *__restrict__ spec,
                                                         double *__restrict__ dep) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n_dir * 4 * n) return;
    const int64_t d = i / (4 * n), r = i % (4 * n);
    double s = 0.0;
    for (int64_t b = 0; b < n_blocks; ++b) s += partial[(d * n_blocks + b) * 4 * n + r];
    const int64_t part = r / n, e = r % n;
    if (part == 0) spec[d * n + e] = s;
    else dep[d * 9 * n + (part - 1) * 3 * n + n + e] = s;
}

// out[d][e] += spec[d][e] + sum_q tail(dep[d][.][q], (e - (q - n)) dE) over node slots q in [q_lo, q_hi).
// FP64-bound: four operations a cell.  A block covers kConvTile bins, four
// neighbours to a lane, and its four waves a quarter of each tile of nodes: the
// reciprocals of a lane's bins slide along with the nodes, so that four nodes
// cost 4 reads of reciprocals (kept by index mod 4: no bank conflict) and 8 of
// moments for 16 cells, where one bin a thread read 4 values for each and was
// bound by LDS (64 directions x 4,096 bins: 488 us, 220 so).
constexpr int kConvTile = 256, kConvWaves = 4;
__global__ void __launch_bounds__(64 * kConvWaves) window_tail_kernel(const double *__restrict__ spec,
                                                                      const double *__restrict__ dep, int64_t n,
                                                                      double dE, int64_t q_lo, int64_t q_hi,
                                                                      double *__restrict__ out) {
    static_assert(kConvTile == 64 * kConvWaves && kConvWaves == 4, "four bins to a lane, a node to a thread");
    __shared__ double4 s_m[kConvTile];
    // reciprocal of bin x node offset o = (e0 - q0 + n) + k - 255 at [k % 4][k / 4]
    __shared__ double s_inv[4][2 * kConvTile / 4];
    __shared__ double s_sum[kConvWaves][kConvTile];
    const int d = blockIdx.y;
    const int64_t e0 = (int64_t)blockIdx.x * kConvTile;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const double *D = dep + (int64_t)d * 9 * n;
    const int64_t L = 3 * n;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t q0 = q_lo; q0 < q_hi; q0 += kConvTile) {
        const int64_t q = q0 + t;
        const bool in = q < q_hi;
        __syncthreads();
        s_m[t] = in ? make_double4(D[q], D[L + q], D[2 * L + q], 0.0) : make_double4(0.0, 0.0, 0.0, 0.0);
        for (int k = t; k < 2 * kConvTile; k += kConvTile) {
            const int64_t o = (e0 - q0 + n) + (int64_t)(k - (kConvTile - 1));
            s_inv[k & 3][k >> 2] = o == 0 ? 0.0 : rcp_nr((double)o * dE);
        }
        __syncthreads();
        // bin e0 + 4 lane + m against node q0 + 4 i + r: k = 4 (lane - i + 63) + (m - r + 3)
        const int i0 = wave * (kConvTile / 4 / kConvWaves);
        double v[7];
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] = s_inv[k][lane - i0 + 64];
#pragma unroll 2
        for (int i = i0; i < i0 + kConvTile / 4 / kConvWaves; ++i) {
#pragma unroll
            for (int k = 0; k < 3; ++k) v[k + 4] = v[k];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = s_inv[k][lane - i + 63];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double4 M = s_m[4 * i + r];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const double inv = v[m - r + 3];
                    acc[m] = fma(fma(fma(M.z, inv, M.y), inv, M.x), inv * inv, acc[m]);
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) s_sum[wave][4 * lane + m] = acc[m];
    __syncthreads();
    const int64_t e = e0 + t;
    if (e >= n) return;
    double sum = 0.0;
    for (int w = 0; w < kConvWaves; ++w) sum += s_sum[w][t];
    out[(int64_t)d * n + e] += spec[(int64_t)d * n + e] + sum;
}

__global__ void fill_zero_kernel(double *__restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Workspace bytes for gx partial rows of n_E bins.
size_t partial_bytes(int64_t gx, int64_t n_E) { return (size_t)gx * (size_t)n_E * sizeof(double); }

// Blocks along the line axis: enough to fill the chip several times over, but
// never more than there are line tiles.
int64_t line_blocks(int cu, int64_t n_tiles, int64_t bin_tiles) {
    int64_t want = (int64_t)cu * 8 / (bin_tiles > 0 ? bin_tiles : 1);
    if (want < 1) want = 1;
    return n_tiles < want ? (n_tiles > 0 ? n_tiles : 1) : want;
}

constexpr int kDenseBins = 4;  // bins per thread of the dense reducers

// Launch shape and workspace bytes of the general reduction of n_lines lines on
// n_E bins, for the current device.
struct DensePlan {
    int64_t gx = 0, bin_tiles = 0;
    size_t bytes = 0;
};
hr_status dense_plan(int64_t n_lines, int64_t n_E, DensePlan &P) {
    int cu = 0;
    hr_status st = device_cu(cu);
    if (st != HR_OK) return st;
    P.bin_tiles = (n_E + kRedThreads * kDenseBins - 1) / (kRedThreads * kDenseBins);
    const int64_t n_tiles = (n_lines + kGeneralTile - 1) / kGeneralTile;
    P.gx = line_blocks(cu, n_tiles, P.bin_tiles);
    P.bytes = (n_lines == 0 || n_E == 0) ? 0 : partial_bytes(P.gx, n_E);
    return HR_OK;
}

// Launch shape and workspace of the brem reduction: bins per thread to the grid
// (a 201-bin grid takes one, not four), tiles of a power of two rows, at least 32,
// that make up to 16 blocks per CU (rows below the bins' energies cost less than
// others, direct ones more), and the class order where it pays: from 1e8 cells, whose
// direct evaluation takes 120 us, and from 160 rows a class on, since a class of a bin
// costs as much as the polynomial saves in some 150 rows (20,480 rows x 4,883 bins of
// 5 keV..10 MeV 141 us against 122 cell by cell, 163 with the tiles before; of
// 0.5..5 MeV 124 against 137; 2,048 x 48,829 458 and 341 against 130).  The
// polynomials and the classes' own rows take 4.6 kB a bin, 300 MB at kBremSortBins,
// beyond which rows stay as they lie in the 32 MB of the direct route.
constexpr int kBremWaves = 512;  // of the sort, at most
struct BremPlan {
    int bins = 4;
    int64_t rows = 32, gx = 1, windows = 1, waves = 0, per = 0;  // waves: of the sort, 0 none
    size_t partials = 0, bytes = 0;
};
hr_status brem_plan(int64_t n_seg, int64_t n_E, BremPlan &P) {
    int cu = 0;
    hr_status st = device_cu(cu);
    if (st != HR_OK) return st;
    P.bins = n_E <= kRedThreads ? 1 : (n_E <= 2 * kRedThreads ? 2 : 4);
    P.windows = (n_E + kRedThreads * P.bins - 1) / (kRedThreads * P.bins);
    int64_t room = 16 * (int64_t)cu / (P.windows > 0 ? P.windows : 1);
    room = room < 1 ? 1 : room;
    while (n_seg > room * P.rows) P.rows *= 2;
    P.gx = (n_seg + P.rows - 1) / P.rows;
    // sizes at their bounds, so that a workspace serves fewer rows too
    const bool some = n_seg > 0 && n_E > 0;
    int64_t rows_max = (n_seg + 31) / 32 < room ? (n_seg + 31) / 32 : room;
    // row indices of the order are 32-bit
    if (some && n_seg >= kBremSortRows && n_seg <= INT32_MAX && n_E <= kBremSortBins &&
        n_seg >= kBremSortCells / n_E) {
        P.per = (n_seg + kBremWaves - 1) / kBremWaves;
        P.per = P.per < 256 ? 256 : (P.per + 63) / 64 * 64;
        P.waves = (n_seg + P.per - 1) / P.per;
        P.gx += kBremClasses - 1;  // every class may end in a tile of its own
        rows_max += kBremClasses - 1;
    }
    P.partials = some ? partial_bytes(rows_max, n_E) : 0;
    P.bytes = P.partials;
    if (P.waves > 0) {
        // [partial rows | order | counts | totals | polynomials]
        P.bytes += (size_t)(n_seg + (kBremWaves + 1) * kBremClasses) * sizeof(uint32_t) +
                   (size_t)kBremClasses * kBremNodes * (size_t)n_E * sizeof(float);
    }
    return HR_OK;
}

// Launch shape of the uniform-grid reduction.  The window of 64 `bins` bins is
// the smallest cover of the grid in windows of 256 to 1024 bins, a window's
// fixed cost per line counted as three bins per lane (the sine and cosine at the
// middle of each run).  Four blocks of four waves share a CU; a wave takes chunks
// of `per` lines, 64 where that leaves every resident wave four, fewer on small
// inputs so that all of them work.  Dead lines come in runs, so where chunks
// abound four times the resident blocks are launched to even the waves out
// (2.7e6 lines on 1024 bins: 464 us resident, 451 so, and 9 more in the row sum).
struct SincPlan {
    int bins = 16, per = kSincChunk;
    int64_t gx = 1, windows = 1;
    size_t bytes = 0;
};
hr_status sinc_plan(int64_t n_lines, int64_t n_E, SincPlan &P) {
    int cu = 0;
    hr_status st = device_cu(cu);
    if (st != HR_OK) return st;
    int64_t best = INT64_MAX;
    for (int b = 16; b >= 4; b -= 4) {
        const int64_t win = (n_E + 64 * b - 1) / (64 * b), cost = win * (b + 3);
        if (cost < best) {
            best = cost;
            P.bins = b;
            P.windows = win;
        }
    }
    const int64_t resident = 4 * (int64_t)cu, windows = P.windows > 0 ? P.windows : 1;
    int64_t room = resident < windows ? 1 : resident / windows;
    while (P.per > 8 && n_lines < room * kSincWaves * P.per * 4) P.per /= 2;
    // (a grid of more windows than blocks keeps one row: four would pass the bound of
    // hr_sincsq_reduce_static)
    if (P.per == kSincChunk) room = 4 * resident < windows ? 1 : 4 * resident / windows;
    const int64_t chunks = (n_lines + P.per - 1) / P.per;
    const int64_t want = (chunks + kSincWaves - 1) / kSincWaves;
    P.gx = want < room ? (want > 0 ? want : 1) : room;
    P.bytes = (n_lines == 0 || n_E == 0) ? 0 : partial_bytes(P.gx, n_E);
    return HR_OK;
}

// Whether the recurrence runs: a uniform grid with a step (every other grid
// takes the general reducer).
bool sinc_recurs(const hr_sincsq_args &p) { return p.uniform && p.dE != 0.0 && isfinite(p.dE) && isfinite(p.E0); }

// Workspace bytes of hr_sincsq_reduce.
hr_status sinc_bytes(const hr_sincsq_args &p, size_t &bytes) {
    if (sinc_recurs(p)) {
        SincPlan P;
        hr_status st = sinc_plan(p.n_lines, p.n_E, P);
        bytes = P.bytes;
        return st;
    }
    DensePlan P;
    hr_status st = dense_plan(p.n_lines, p.n_E, P);
    bytes = P.bytes;
    return st;
}

// Blocks of the standalone windowed reduction and its workspace bytes:
// [partials blocks*4*n | spec n | node moments 9n].
int64_t window_reduce_blocks(int cu, int64_t n_lines) {
    int64_t blocks = (n_lines + kWinThreads - 1) / kWinThreads;
    return blocks < 2 * (int64_t)cu ? blocks : 2 * (int64_t)cu;
}

// Line-axis chunks per direction of the fused pixel route (about two resident
// blocks per CU in total; one block fills a CU's LDS).
int64_t window_chunks(int cu, int64_t n_seg, int32_t n_dir) {
    int64_t chunks = (2 * (int64_t)cu + n_dir - 1) / n_dir;
    const int64_t max_chunks = (n_seg + kWinThreads - 1) / kWinThreads;
    chunks = chunks < max_chunks ? chunks : max_chunks;
    return chunks < 1 ? 1 : chunks;
}

}  // namespace
}  // namespace hr

extern "C" hr_status hr_cxr_lines(const hr_line_args *args, void *stream) {
    HR_TRACE("hr_cxr_lines");
    using namespace hr;
    HR_REQUIRE(args != nullptr, "hr_cxr_lines: null args");
    const hr_line_args &p = *args;
    HR_REQUIRE(p.n_seg >= 0 && p.n_dir >= 1 && p.n_g >= 1 && p.n_tab >= 2 && p.n_mu >= 1,
               "hr_cxr_lines: bad sizes (n_seg=%lld n_dir=%d n_g=%d n_tab=%lld n_mu=%d)",
               (long long)p.n_seg, p.n_dir, p.n_g, (long long)p.n_tab, p.n_mu);
    if (p.n_seg == 0) return HR_OK;
    HR_REQUIRE(p.r_mid && p.v_hat && p.L && p.E && p.n_hat && p.dir_weight && p.g && p.wm && p.row &&
                   p.e_s && p.e_p && p.E_tab && p.delta_tab && p.chi_re && p.chi_im && p.u_re && p.u_im &&
                   p.log_mu && p.E_r && p.a && p.w,
               "hr_cxr_lines: null pointer");
    const int64_t total = p.n_seg * (int64_t)p.n_dir;
    const int block = 256;
    const int64_t grid = (total + block - 1) / block;
    HR_REQUIRE(grid < (1LL << 31), "hr_cxr_lines: %lld segment-direction pairs exceed one launch",
               (long long)total);
    hipLaunchKernelGGL(cxr_lines_kernel, dim3((unsigned)grid), dim3(block), 0, (hipStream_t)stream, p);
    HR_CHECK_HIP(hipGetLastError());
    return HR_OK;
}

extern "C" hr_status hr_sincsq_reduce(const hr_sincsq_args *args, void *stream) {
    HR_TRACE("hr_sincsq_reduce");
    using namespace hr;
    HR_REQUIRE(args != nullptr, "hr_sincsq_reduce: null args");
    const hr_sincsq_args &p = *args;
    HR_REQUIRE(p.n_lines >= 0 && p.n_E >= 0, "hr_sincsq_reduce: negative size");
    if (p.n_lines == 0 || p.n_E == 0) return HR_OK;
    HR_REQUIRE(p.E_r && p.a && p.w && p.out, "hr_sincsq_reduce: null pointer");
    HR_REQUIRE(p.uniform || p.E_grid, "hr_sincsq_reduce: a non-uniform grid needs E_grid");
    hipStream_t s = (hipStream_t)stream;
    void *ws = p.ws.ptr;
    if (sinc_recurs(p)) {
        SincPlan P;
        hr_status st = sinc_plan(p.n_lines, p.n_E, P);
        if (st != HR_OK) return st;
        HR_REQUIRE_WS(p.ws, P.bytes, "hr_sincsq_reduce");
        HR_REQUIRE(P.windows <= 65535, "hr_sincsq_reduce: %lld bins exceed one launch", (long long)p.n_E);
        const dim3 grid((unsigned)P.gx, (unsigned)P.windows), block(kSincBlock);
#define HR_SINC(B)                                                                                              \
    hipLaunchKernelGGL(sincsq_uniform_kernel<B>, grid, block, 0, s, p.E_r, p.a, p.w, p.n_lines, P.per, p.E0,   \
                       p.dE, p.n_E, (double *)ws)
        switch (P.bins) {
        case 4: HR_SINC(4); break;
        case 8: HR_SINC(8); break;
        case 12: HR_SINC(12); break;
        default: HR_SINC(16); break;
        }
#undef HR_SINC
        HR_CHECK_HIP(hipGetLastError());
        return row_sum((const double *)ws, P.gx, p.n_E, p.out, s);
    }
    DensePlan P;
    hr_status st = dense_plan(p.n_lines, p.n_E, P);
    if (st != HR_OK) return st;
    HR_REQUIRE_WS(p.ws, P.bytes, "hr_sincsq_reduce");
    const dim3 grid((unsigned)P.gx, (unsigned)P.bin_tiles);
    hipLaunchKernelGGL(sincsq_general_kernel<kDenseBins>, grid, dim3(kRedThreads), 0, s, p.E_r, p.a, p.w, p.n_lines,
                       p.uniform ? nullptr : p.E_grid, p.E0, p.dE, p.n_E, (double *)ws);
    HR_CHECK_HIP(hipGetLastError());
    return row_sum((const double *)ws, P.gx, p.n_E, p.out, s);
}

// Scratch of hr_sincsq_reduce_static: the partial spectra of one call live in
// this file-scope device array instead of a caller workspace.  Each device
// holds its own copy at its own address, found once per device with
// hipGetSymbolAddress; host code uses that address, never the symbol itself.
static __device__ __align__(256) unsigned char scratch[HR_SINCSQ_STATIC_SCRATCH_BYTES];

namespace hr {
namespace {
std::mutex g_scratch_mu;
void *g_scratch_ptr[64];

hr_status static_scratch(void **out) {
    int dev = 0;
    HR_CHECK_HIP(hipGetDevice(&dev));
    HR_REQUIRE(dev >= 0 && dev < 64, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        HR_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        HR_REQUIRE(p != nullptr && ((uintptr_t)p & 255u) == 0, "static scratch at %p is null or misaligned", p);
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return HR_OK;
}
}  // namespace
}  // namespace hr

extern "C" hr_status hr_sincsq_reduce_static(const hr_sincsq_args *args, void *stream) {
    HR_TRACE("hr_sincsq_reduce_static");
    using namespace hr;
    HR_REQUIRE(args != nullptr, "hr_sincsq_reduce_static: null args");
    HR_REQUIRE(args->n_lines >= 0 && args->n_E >= 0, "hr_sincsq_reduce_static: negative size");
    if (args->n_lines == 0 || args->n_E == 0) return HR_OK;
    // the sizes taken are those whose general-grid partials (and 64 more rows) fit, whatever the grid
    DensePlan P;
    size_t need = 0;
    hr_status st = dense_plan(args->n_lines, args->n_E, P);
    if (st == HR_OK) st = sinc_bytes(*args, need);
    if (st != HR_OK) return st;
    const size_t limit = partial_bytes(P.gx + (P.gx < 64 ? P.gx : 64), args->n_E);
    if (need < limit) need = limit;
    HR_REQUIRE(need <= (size_t)HR_SINCSQ_STATIC_SCRATCH_BYTES,
               "hr_sincsq_reduce_static: %lld bins need %zu bytes of partials, more than the %zu-byte static "
               "scratch (use hr_sincsq_reduce with a workspace)",
               (long long)args->n_E, need, (size_t)HR_SINCSQ_STATIC_SCRATCH_BYTES);
    void *ptr = nullptr;
    st = static_scratch(&ptr);
    if (st != HR_OK) return st;
    hr_sincsq_args q = *args;
    q.ws.ptr = ptr;
    q.ws.bytes = (size_t)HR_SINCSQ_STATIC_SCRATCH_BYTES;
    return hr_sincsq_reduce(&q, stream);
}

extern "C" hr_status hr_sincsq_workspace_bytes(const hr_sincsq_args *args, size_t *bytes) {
    using namespace hr;
    HR_REQUIRE(args != nullptr && bytes != nullptr, "hr_sincsq_workspace_bytes: null argument");
    HR_REQUIRE(args->n_lines >= 0 && args->n_E >= 0, "hr_sincsq_workspace_bytes: negative size");
    return sinc_bytes(*args, *bytes);
}

extern "C" hr_status hr_brem_workspace_bytes(const hr_brem_args *args, size_t *bytes) {
    using namespace hr;
    HR_REQUIRE(args != nullptr && bytes != nullptr, "hr_brem_workspace_bytes: null argument");
    HR_REQUIRE(args->n_seg >= 0 && args->n_E >= 0, "hr_brem_workspace_bytes: negative size");
    BremPlan P;
    hr_status st = brem_plan(args->n_seg, args->n_E, P);
    if (st != HR_OK) return st;
    *bytes = P.bytes;
    return HR_OK;
}

extern "C" hr_status hr_brem_reduce(const hr_brem_args *args, void *stream) {
    HR_TRACE("hr_brem_reduce");
    using namespace hr;
    HR_REQUIRE(args != nullptr, "hr_brem_reduce: null args");
    const hr_brem_args &p = *args;
    HR_REQUIRE(p.n_seg >= 0 && p.n_E >= 0, "hr_brem_reduce: negative size");
    HR_REQUIRE(p.n_el >= 1 && p.n_el <= 4, "hr_brem_reduce: 1..4 elements supported, got %d", p.n_el);
    if (p.n_seg == 0 || p.n_E == 0) return HR_OK;
    HR_REQUIRE(p.r_mid && p.v_hat && p.L && p.E_keV && p.E_grid_eV && p.mu && p.out,
               "hr_brem_reduce: null pointer");
    BremPlan P;
    hr_status st = brem_plan(p.n_seg, p.n_E, P);
    if (st != HR_OK) return st;
    HR_REQUIRE_WS(p.ws, P.bytes, "hr_brem_reduce");
    hipStream_t s = (hipStream_t)stream;
    double *ws = (double *)p.ws.ptr;
    BremOrder o{};
    if (P.waves > 0) {
        uint32_t *order = (uint32_t *)((char *)p.ws.ptr + P.partials), *counts = order + p.n_seg;
        uint32_t *totals = counts + P.waves * kBremClasses;
        float *poly = (float *)(totals + kBremClasses);
        o = BremOrder{order, totals, poly};
        hipLaunchKernelGGL(brem_count_kernel, dim3((unsigned)P.waves), dim3(64), 0, s, p, P.per, counts);
        HR_CHECK_HIP(hipGetLastError());
        hipLaunchKernelGGL(brem_scan_kernel, dim3(kBremClasses), dim3(64), 0, s, counts, P.waves, totals);
        HR_CHECK_HIP(hipGetLastError());
        const int64_t groups = (p.n_E + kBremPolyBins - 1) / kBremPolyBins;
        hipLaunchKernelGGL(brem_lay_kernel, dim3((unsigned)(P.waves + groups * kBremClasses)), dim3(64), 0, s, p, P.per,
                           P.waves, counts, totals, order, poly);
        HR_CHECK_HIP(hipGetLastError());
    }
    const dim3 grid((unsigned)P.gx, (unsigned)P.windows);
#define HR_BREM(B, NEL)                                                                                             \
    if (P.waves > 0)                                                                                                \
        hipLaunchKernelGGL((brem_kernel<B, NEL, true>), grid, dim3(kRedThreads), 0, s, p, P.rows, o, ws);           \
    else                                                                                                            \
        hipLaunchKernelGGL((brem_kernel<B, NEL, false>), grid, dim3(kRedThreads), 0, s, p, P.rows, o, ws)
#define HR_BREM_EL(B)                    \
    switch (p.n_el) {                    \
    case 1: HR_BREM(B, 1); break;        \
    case 2: HR_BREM(B, 2); break;        \
    case 3: HR_BREM(B, 3); break;        \
    default: HR_BREM(B, 4); break;       \
    }
    switch (P.bins) {
    case 1: HR_BREM_EL(1); break;
    case 2: HR_BREM_EL(2); break;
    default: HR_BREM_EL(4); break;
    }
#undef HR_BREM_EL
#undef HR_BREM
    HR_CHECK_HIP(hipGetLastError());
    return row_sum(ws, P.gx, p.n_E, p.out, s);
}

namespace hr {
namespace {

hr_status window_setup(int64_t n_E, double E0, double dE, double x_c, WindowGrid &G) {
    HR_REQUIRE(n_E >= 1 && n_E <= kWinMaxBins, "windowed reduction: n_E %lld outside [1, %d]", (long long)n_E,
               kWinMaxBins);
    HR_REQUIRE(dE > 0.0 && isfinite(E0), "windowed reduction: needs a uniform ascending grid");
    HR_REQUIRE(x_c > 0.0, "windowed reduction: x_c must be positive");
    G.n = n_E;
    G.E0 = E0;
    G.dE = dE;
    G.x_c = x_c;
    G.inv_dE = 1.0 / dE;
    return HR_OK;
}

// Launch window_sum + window_tail over `blocks` partials per direction; the
// workspace holds [partials | spec | dep] and dep was zeroed before the deposit.
hr_status window_finish(double *partial, int64_t blocks, int n_dir, const WindowGrid &G, double *spec, double *dep,
                        int64_t q_lo, int64_t q_hi, double *out, hipStream_t s) {
    const int64_t n = G.n;
    const int64_t tot = (int64_t)n_dir * 4 * n;
    hipLaunchKernelGGL(window_sum_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, partial, blocks, n,
                       n_dir, spec, dep);
    HR_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(window_tail_kernel, dim3((unsigned)((n + kConvTile - 1) / kConvTile), (unsigned)n_dir),
                       dim3(kConvTile), 0, s, spec, dep, n, G.dE, q_lo, q_hi, out);
    HR_CHECK_HIP(hipGetLastError());
    return HR_OK;
}

}  // namespace
}  // namespace hr

extern "C" hr_status hr_window_reduce_workspace_bytes(int64_t n_lines, int64_t n_E, size_t *bytes) {
    using namespace hr;
    HR_REQUIRE(bytes != nullptr && n_lines >= 0 && n_E >= 0, "hr_window_reduce_workspace_bytes: bad arguments");
    *bytes = 0;
    if (n_lines == 0 || n_E == 0) return HR_OK;
    int cu = 0;
    hr_status st = device_cu(cu);
    if (st != HR_OK) return st;
    const int64_t blocks = window_reduce_blocks(cu, n_lines);
    *bytes = (size_t)(blocks * 4 * n_E + n_E + 9 * n_E) * sizeof(double);
    return HR_OK;
}

extern "C" hr_status hr_window_reduce(const double *E_r, const double *a, const float *w, int64_t n_lines,
                                      int64_t n_E, double E0, double dE, double x_c, double *out, hr_workspace ws,
                                      void *stream) {
    HR_TRACE("hr_window_reduce");
    using namespace hr;
    HR_REQUIRE(n_lines >= 0, "hr_window_reduce: negative n_lines");
    if (n_lines == 0 || n_E == 0) return HR_OK;
    HR_REQUIRE(E_r && a && w && out, "hr_window_reduce: null pointer");
    WindowGrid G;
    hr_status st = window_setup(n_E, E0, dE, x_c, G);
    if (st != HR_OK) return st;
    int cu = 0;
    st = device_cu(cu);
    if (st != HR_OK) return st;
    const int64_t blocks = window_reduce_blocks(cu, n_lines);
    const int64_t n = n_E;
    const size_t need = (size_t)(blocks * 4 * n + n + 9 * n) * sizeof(double);
    HR_REQUIRE_WS(ws, need, "hr_window_reduce");
    double *partial = (double *)ws.ptr, *spec = partial + blocks * 4 * n, *dep = spec + n;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((9 * n + 255) / 256)), dim3(256), 0, s, dep, 9 * n);
    HR_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(window_given_kernel, dim3((unsigned)blocks), dim3(kWinThreads), 0, s, E_r, a, w, n_lines, G,
                       partial, dep);
    HR_CHECK_HIP(hipGetLastError());
    return window_finish(partial, blocks, 1, G, spec, dep, 0, 3 * n, out, s);
}

extern "C" hr_status hr_window_spectra_workspace_bytes(const hr_window_args *args, size_t *bytes) {
    using namespace hr;
    HR_REQUIRE(args != nullptr && args->lines != nullptr && bytes != nullptr,
               "hr_window_spectra_workspace_bytes: null argument");
    const hr_line_args &p = *args->lines;
    HR_REQUIRE(p.n_seg >= 0 && p.n_dir >= 1 && args->n_E >= 0, "hr_window_spectra_workspace_bytes: bad sizes");
    *bytes = 0;
    if (p.n_seg == 0 || args->n_E == 0) return HR_OK;
    int cu = 0;
    hr_status st = device_cu(cu);
    if (st != HR_OK) return st;
    const int64_t n = args->n_E;
    const int64_t chunks = window_chunks(cu, p.n_seg, p.n_dir);
    *bytes = (size_t)((int64_t)p.n_dir * (chunks * 4 * n + n + 9 * n)) * sizeof(double);
    return HR_OK;
}

extern "C" hr_status hr_window_spectra(const hr_window_args *args, void *stream) {
    HR_TRACE("hr_window_spectra");
    using namespace hr;
    HR_REQUIRE(args != nullptr && args->lines != nullptr, "hr_window_spectra: null args");
    const hr_line_args &p = *args->lines;
    HR_REQUIRE(p.n_seg >= 0 && p.n_dir >= 1 && p.n_g >= 1, "hr_window_spectra: bad sizes");
    if (p.n_seg == 0 || args->n_E == 0) return HR_OK;
    HR_REQUIRE(p.r_mid && p.v_hat && p.L && p.E && p.n_hat && p.dir_weight && p.g && p.wm && p.row && p.e_s &&
                   p.e_p && p.E_tab && p.delta_tab && p.chi_re && p.chi_im && p.u_re && p.u_im && p.log_mu &&
                   args->out,
               "hr_window_spectra: null pointer");
    HR_REQUIRE(p.n_tab >= 2 && p.n_mu >= 1, "hr_window_spectra: tables too small");
    HR_REQUIRE(p.n_dir <= 65535, "hr_window_spectra: at most 65535 directions");
    WindowGrid G;
    hr_status st = window_setup(args->n_E, args->E0, args->dE, args->x_c, G);
    if (st != HR_OK) return st;
    int cu = 0;
    st = device_cu(cu);
    if (st != HR_OK) return st;
    const int64_t n = G.n;
    const int64_t chunks = window_chunks(cu, p.n_seg, p.n_dir);
    const size_t need = (size_t)((int64_t)p.n_dir * (chunks * 4 * n + n + 9 * n)) * sizeof(double);
    HR_REQUIRE_WS(args->ws, need, "hr_window_spectra");
    double *partial = (double *)args->ws.ptr;
    double *spec = partial + (int64_t)p.n_dir * chunks * 4 * n;
    double *dep = spec + (int64_t)p.n_dir * n;
    hipStream_t s = (hipStream_t)stream;
    const int64_t nd9 = (int64_t)p.n_dir * 9 * n;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((nd9 + 255) / 256)), dim3(256), 0, s, dep, nd9);
    HR_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(window_lines_kernel, dim3((unsigned)chunks, (unsigned)p.n_dir), dim3(kWinThreads), 0, s, p,
                       G, partial, dep);
    HR_CHECK_HIP(hipGetLastError());
    // node slots reachable from the keep window
    int64_t q_lo = (int64_t)floor((p.lo_keep - G.E0) / G.dE) - 1 + n;
    int64_t q_hi = (int64_t)ceil((p.hi_keep - G.E0) / G.dE) + 2 + n;
    q_lo = q_lo < 0 ? 0 : (q_lo > 3 * n ? 3 * n : q_lo);
    q_hi = q_hi < q_lo ? q_lo : (q_hi > 3 * n ? 3 * n : q_hi);
    return window_finish(partial, chunks, p.n_dir, G, spec, dep, q_lo, q_hi, args->out, s);
}
