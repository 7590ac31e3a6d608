// Detector model: photons -> expectation E -> EMCCD signal + readout noise ->
// ADC counts.
//
// Reference: src/scopyon/_epifm.py:1430-1470 (__detector_output),
//            _epifm.py:355-416 (EMCCD), _epifm.py:1472-1484 (ADC).
//
// Two signal paths:
//  * parity  : the reference's discrete pmf on S in [s_min, s_max) drawn by
//              inverse CDF with a given uniform per pixel (the uniform numpy's
//              RandomState.choice would consume).  One wave per pixel sums
//              the pmf by runs of emgain terms with a Gauss rule per run, then
//              descends to the term where the cumulative mass passes
//              u * total.  Readout noise comes in pre-drawn.
//  * philox  : statistically equivalent sampler driven by Philox4x32-10:
//              n ~ Poisson(E), S = round(Gamma(n, emgain)) (S >= 1 when n >= 1),
//              noise ~ N(0, readout_noise^2).  O(1) per pixel.
#include "common.hpp"
#include "emccd_block.hpp"
#include "scopyon_hip_types.h"

#include <hipcub/hipcub.hpp>

namespace {

__device__ inline double adc_counts(double x, const smx_detector_params_t& P, double gain,
                                    double offset) {
    // _epifm.py:1475-1484, same order, no rounding
    if (x > P.fullwell) x = P.fullwell;
    x = x / gain;
    x = x + offset;
    if (x > P.adc_max) x = P.adc_max;
    if (x < 0.0) x = 0.0;
    return x;
}

__device__ inline double expectation(double photons, const smx_detector_params_t& P) {
    if (P.background_switch) photons = photons + P.background;
    return P.qe * photons;
}

// Compound Poisson-Gamma pmf term (_epifm.py:364-388) at X = a S, S > 0,
// times exp(-E): exp(-X + Y) / Y i1e(Y) with Y = 2 sqrt(E X), and
// -X + Y - E = -(sqrt(X) - sqrt(E))^2.  The draw only needs ratios of terms,
// and the exponent of this form is small where the mass is, so it rounds to
// ~25 ulp instead of the ~E ulp of -X + Y.  S = 0 has a term of its own
// (emccd_zero_term).
//
// i1e as smx::i1e (power series below SMX_I1E_YB, Chebyshev series in 1 / Y
// above) with fused multiply-adds, its exp(-Y) and division joined with the
// term's own.  A call, not inlined: five copies of its ~250 instructions cost
// the kernel 130 registers and its instruction cache (0.98 ms per 512 x 512
// frame with 10,000 emitters inlined, 0.72 ms called).
__device__ __attribute__((noinline)) double emccd_term(double X, double E, double rootE) {
    const double rootX = sqrt(X), d = rootX - rootE;
    const double Y = 2.0 * (rootE * rootX);
    if (Y <= SMX_I1E_YB) {
        const double q = Y * Y * 0.25;
        double acc = smx_i1e_series[SMX_I1E_NSERIES - 1];
#pragma unroll
        for (int k = SMX_I1E_NSERIES - 2; k >= 0; --k) acc = fma(acc, q, smx_i1e_series[k]);
        return 0.5 * acc * exp(-fma(d, d, Y));
    }
    const double t = (2.0 * SMX_I1E_YB) / Y - 1.0, t2 = 2.0 * t;
    double b1 = 0.0, b2 = 0.0;
#pragma unroll
    for (int k = SMX_I1E_NCHEB - 1; k >= 1; --k) {
        const double b0 = fma(t2, b1, smx_i1e_cheb[k] - b2);
        b2 = b1;
        b1 = b0;
    }
    return exp(-d * d) * fma(t, b1, smx_i1e_cheb[0] - b2) / (Y * sqrt(Y));
}
__device__ inline double emccd_zero_term(double E, double a) { return exp(-E) / (2.0 * a * E); }

// The reference's own terms overflow (numpy.random.choice raises ValueError)
// when exp(-X + Y) does at some S; -X + Y peaks at X = E, so at one of the two
// integers around E / a.
__device__ inline bool emccd_overflows(double E, double a) {
    const double S = floor(E / a);
    bool over = false;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double X = a * (S + k), Y = 2.0 * sqrt(E * X);
        over |= !(exp(-X + Y) < INFINITY);
    }
    return over;
}

__device__ inline void emccd_support(double E, int g, long long& s_min, long long& s_max) {
    double sigma = sqrt(E) * 5.0 + 10.0;
    long long lo = (long long)g * (long long)(E - sigma);   // int() truncates toward 0
    s_min = lo > 0 ? lo : 0;
    s_max = (long long)g * (long long)(E + sigma);
}

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__global__ void prepare_kernel(int n, const double* __restrict__ photons, smx_detector_params_t P,
                               double* __restrict__ E_out, int* __restrict__ flag) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double E = expectation(photons[i], P);
    E_out[i] = E;
    if (flag) flag[i] = E > 0.0 ? 1 : 0;
}

// The parity draw needs the total of the pmf over its support and the first S
// whose cumulative mass passes u T.  The support [s_min, s_max) is a whole
// number of runs of g = emgain consecutive S (both ends are multiples of g),
// and the term is smooth in X = S / g (exp(-X) I1(Y) / Y is entire in X), so
// the sum over one run is a Gauss rule for the counting measure on g points:
// QN nodes, exact for polynomials in S of degree 2 QN - 1.  With X moving by 1
// over a run the rule's error is below 1e-15 of the total for every E that
// does not overflow (checked against the direct sums; rounding of the terms
// dominates).  A run of g = 300 terms costs 8 evaluations, 8 runs per wave
// pass.  The draw then descends: the run from the run sums, 64-term pieces of
// it with the same kind of rule (g > 128), the term by direct evaluation.
// This kernel is float64 VALU bound (exp, i1e, two square roots and a
// division per evaluation); summing every term directly took 12.8 ms per
// 512 x 512 frame with 10,000 emitters at g = 300, this takes 0.72 ms.
// g <= QN: the runs are 64 consecutive terms, evaluated directly.
constexpr int QN = 8;
constexpr int RUNS_MAX = 320;   // runs of a support: at most 288 before E overflows

struct RunRule {
    int len;           // terms of a run
    int direct;        // 1: runs of 64 consecutive terms, no rule
    double x[QN];      // nodes in [0, len - 1]
    double w[QN];
    double x64[QN];    // the rule for 64 terms
    double w64[QN];
};

// Gauss rule for the counting measure on 0 .. N - 1 (N > QN): the zeros of the
// monic discrete Chebyshev (Gram) polynomials about the centre,
// p_{k+1} = t p_k - beta_k p_{k-1}, beta_k = k^2 (N^2 - k^2) / (4 (4 k^2 - 1)),
// found degree by degree between the zeros of the degree below (they
// interlace), and the weights N / sum_k p_k(x)^2 / (beta_1 .. beta_k).
void gram_rule(int N, double* x, double* w) {
    long double beta[QN], zero[QN + 2], below[QN + 2];
    const long double n2 = (long double)N * N;
    for (int k = 1; k < QN; ++k)
        beta[k] = (long double)k * k * (n2 - (long double)k * k) / (4.0L * (4.0L * k * k - 1.0L));
    auto eval = [&](int deg, long double t, long double& slope) {
        long double p0 = 1.0L, p1 = t, d0 = 0.0L, d1 = 1.0L;
        for (int k = 1; k < deg; ++k) {
            const long double p = t * p1 - beta[k] * p0, d = p1 + t * d1 - beta[k] * d0;
            p0 = p1; p1 = p;
            d0 = d1; d1 = d;
        }
        slope = d1;
        return p1;
    };
    below[0] = -0.5L * N;
    below[1] = 0.0L;
    below[2] = 0.5L * N;
    for (int deg = 2; deg <= QN; ++deg) {
        for (int i = 0; i < deg; ++i) {
            long double lo = below[i], hi = below[i + 1], slope;
            // the sign at the right end of the i-th interval is (-1)^(deg - 1 - i)
            const bool up = ((deg - 1 - i) & 1) == 0;
            long double t = 0.5L * (lo + hi);
            for (int it = 0; it < 60; ++it) {
                const long double p = eval(deg, t, slope);
                ((p > 0.0L) == up ? hi : lo) = t;
                long double next = t - p / slope;
                if (!(next > lo && next < hi)) next = 0.5L * (lo + hi);
                if (next == t) break;
                t = next;
            }
            zero[i + 1] = t;
        }
        for (int i = 1; i <= deg; ++i) below[i] = zero[i];
        below[deg + 1] = 0.5L * N;
    }
    for (int j = 0; j < QN; ++j) {
        const long double t = zero[j + 1];
        long double p0 = 0.0L, p1 = 1.0L, h = 1.0L, sum = 1.0L;
        for (int k = 1; k < QN; ++k) {
            const long double p = t * p1 - (k > 1 ? beta[k - 1] : 0.0L) * p0;
            p0 = p1; p1 = p;
            h *= beta[k];
            sum += p * p / h;
        }
        x[j] = (double)(t + 0.5L * (N - 1));
        w[j] = (double)((long double)N / sum);
    }
}

RunRule make_run_rule(int g) {
    RunRule R = {};
    R.direct = g <= QN ? 1 : 0;
    R.len = R.direct ? 64 : g;
    if (!R.direct) {
        gram_rule(g, R.x, R.w);
        gram_rule(64, R.x64, R.w64);
    }
    return R;
}

__device__ inline void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Pmf {
    double E, rootE, a;
    long long s_min, len;   // support [s_min, s_min + len)
};

__device__ inline Pmf make_pmf(double E, int g) {
    Pmf p;
    long long s_max;
    emccd_support(E, g, p.s_min, s_max);
    p.E = E;
    p.rootE = sqrt(E);
    p.a = 1.0 / (double)g;
    p.len = s_max - p.s_min;
    return p;
}

// pmf at support index k (integer)
__device__ inline double pmf_at(const Pmf& p, long long k) {
    const long long S = p.s_min + k;
    return S == 0 ? emccd_zero_term(p.E, p.a) : emccd_term(p.a * (double)S, p.E, p.rootE);
}

// Eight 8-node rules at once, one per group of eight lanes: the sum over the
// `span` terms from support index `first` (per group), 0 where !on.  Every
// lane of a group gets the group's sum.
__device__ inline double group_rule(const Pmf& p, long long first, bool on, double xn, double wn) {
    double v = 0.0;
    if (on) {
        const double S = (double)(p.s_min + first) + xn;
        v = wn * emccd_term(p.a * S, p.E, p.rootE);
        // S = 0 does not follow the formula, whose limit there is 1/2
        if (p.s_min + first == 0 && (threadIdx.x & 7) == 0)
            v += emccd_zero_term(p.E, p.a) - 0.5 * exp(-p.E);
    }
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    return v;
}

// Run sums into ch[0 .. runs - 1]; returns the total, added in run order.
__device__ inline double run_sums(const Pmf& p, const RunRule& R, int runs, int lane, double* ch) {
    double T = 0.0;
    if (R.direct) {
        for (int c = 0; c < runs; ++c) {
            const long long k = 64LL * c + lane;
            const double v = wave_sum(k < p.len ? pmf_at(p, k) : 0.0);
            if (lane == 0) ch[c] = v;
            T += v;
        }
    } else {
        const double xn = R.x[lane & 7], wn = R.w[lane & 7];
        for (int c0 = 0; c0 < runs; c0 += 8) {
            const int c = c0 + (lane >> 3);
            const double v = group_rule(p, (long long)R.len * c, c < runs, xn, wn);
            if ((lane & 7) == 0 && c < runs) ch[c] = v;
            T += v;   // the group's own runs; joined below
        }
        T += __shfl_xor(T, 8, 64);
        T += __shfl_xor(T, 16, 64);
        T += __shfl_xor(T, 32, 64);
    }
    wave_sync_lds();
    return T;
}

// The first support index whose cumulative mass exceeds thr (the last index
// when rounding leaves none).
__device__ inline long long emccd_find(const Pmf& p, const RunRule& R, int runs, const double* ch,
                                       double thr, int lane) {
    double carry = 0.0;   // mass before support index pos
    int run = runs;
    for (int b = 0; b < runs; b += 64) {
        const int c = b + lane;
        double v = c < runs ? ch[c] : 0.0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_up(v, off, 64);
            if (lane >= off) v += o;
        }
        const double cum = carry + v;
        const double up = __shfl_up(cum, 1, 64);
        const double before = lane == 0 ? carry : up;
        const unsigned long long hit = __ballot(c < runs && cum > thr);
        if (hit) {
            const int l = __ffsll((long long)hit) - 1;
            run = b + l;
            carry = __shfl(before, l, 64);
            break;
        }
        carry = __shfl(cum, 63, 64);
    }
    if (run >= runs) return p.len - 1;
    long long pos = (long long)R.len * run;
    if (R.len > 128) {
        // the run's whole 64-term pieces, eight at a time
        const double xn = R.x64[lane & 7], wn = R.w64[lane & 7];
        const int pieces = R.len >> 6;
        bool found = false;
        for (int b = 0; b < pieces && !found; b += 8) {
            const int s = lane >> 3;
            double v = group_rule(p, pos + 64LL * s, b + s < pieces, xn, wn);
#pragma unroll
            for (int off = 8; off < 64; off <<= 1) {
                const double o = __shfl_up(v, off, 64);
                if (lane >= off) v += o;
            }
            const double cum = carry + v;
            const double up = __shfl_up(cum, 8, 64);
            const double before = lane < 8 ? carry : up;
            const unsigned long long hit = __ballot(b + s < pieces && cum > thr);
            if (hit) {
                const int l = __ffsll((long long)hit) - 1;
                carry = __shfl(before, l, 64);
                pos += 64LL * (l >> 3);
                found = true;
            } else {
                carry = __shfl(cum, 63, 64);
                pos += 64LL * min(8, pieces - b);
            }
        }
    }
    // term by term (into the next run if these terms have not yet passed thr
    // at this one's end)
    for (; pos < p.len; pos += 64) {
        const long long k = pos + lane;
        double v = k < p.len ? pmf_at(p, k) : 0.0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_up(v, off, 64);
            if (lane >= off) v += o;
        }
        const double cum = carry + v;
        const unsigned long long hit = __ballot(k < p.len && cum > thr);
        if (hit) {
            const long long at = pos + (long long)(__ffsll((long long)hit) - 1);
            return at < p.len - 1 ? at : p.len - 1;
        }
        carry = __shfl(cum, 63, 64);
    }
    return p.len - 1;
}

__device__ inline int run_count(const Pmf& p, const RunRule& R) {
    return (int)((p.len + R.len - 1) / R.len);
}

// The pmf of one expectation value shared by many pixels: T_out[0] = total
// (0 when the reference's pmf overflows), T_out[1 ..] = its run sums.
__global__ void emccd_common_total_kernel(double E, int g, RunRule R, double* __restrict__ T_out) {
    const int lane = threadIdx.x & 63;
    double T = 0.0;
    if (E > 0.0 && E <= 1.0e4) {
        const Pmf p = make_pmf(E, g);
        const int runs = run_count(p, R);
        if (runs <= RUNS_MAX && !emccd_overflows(E, p.a))
            T = run_sums(p, R, runs, lane, T_out + 1);
    }
    if (lane == 0) *T_out = T;
}

__global__ void __launch_bounds__(256) emccd_parity_kernel(
        int n, const double* __restrict__ E_arr, const double* __restrict__ noise,
        const double* __restrict__ uniforms, const int* __restrict__ uidx,
        const double* __restrict__ gain_map, const double* __restrict__ offset_map,
        smx_detector_params_t P, RunRule R, double E_common, const double* __restrict__ T_common,
        double* __restrict__ adc_out, double* __restrict__ signal_out, int* __restrict__ status) {
    __shared__ double s_ch[4][RUNS_MAX];   // run sums, one pixel per wave
    const int lane = threadIdx.x & 63;
    const int pix = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (pix >= n) return;
    const double E = E_arr[pix];
    double S = 0.0;
    if (!(E <= 1.0e4)) {
        // NaN (int(nan) raises in the reference) or far beyond E ~ 709.8, where
        // exp(-X + Y) overflows and numpy.random.choice raises ValueError
        if (lane == 0) atomicOr(status, 4);
    } else if (E > 0.0) {
        const Pmf p = make_pmf(E, P.emgain);
        const int runs = run_count(p, R);
        const bool common = T_common && E == E_common;
        double* const ch = s_ch[threadIdx.x >> 6];
        double T = 0.0;
        if (common) T = *T_common;
        else if (runs <= RUNS_MAX && !emccd_overflows(E, p.a)) T = run_sums(p, R, runs, lane, ch);
        if (!(T > 0.0) || !(T * exp(E - 1.0) < 0x1.78b56362cef37p+1022)) {
            // the reference's pmf or its sum T exp(E) overflows here (the
            // bound is DBL_MAX / e; numpy.random.choice raises ValueError)
            if (lane == 0) atomicOr(status, 4);
        } else {
            const double thr = uniforms[uidx[pix]] * T;
            S = (double)(p.s_min + emccd_find(p, R, runs, common ? T_common + 1 : ch, thr, lane));
        }
    }
    if (lane == 0) {
        double x = S + (noise ? noise[pix] : 0.0);
        double gain = gain_map ? gain_map[pix] : P.gain;
        double offset = offset_map ? offset_map[pix] : P.offset;
        adc_out[pix] = adc_counts(x, P, gain, offset);
        if (signal_out) signal_out[pix] = S;
    }
}

// ---------------------------------------------------------------------------
// Philox samplers: emccd_block.hpp (shared with the fused splat + detector
// tile pass).  Float32 arithmetic: these paths are statistical, not
// bit-parity paths.
// ---------------------------------------------------------------------------
using namespace smx::emccd;

// EMCCD + ADC on Philox streams: a block of 256 threads owns 1024 consecutive
// pixels (4 per thread, coalesced) and runs emccd_block's work queues over
// them.
constexpr int EQ_THREADS = 256, EQ_PPT = 4, EQ_PIX = EQ_THREADS * EQ_PPT;

template <typename OutT>
__global__ void __launch_bounds__(EQ_THREADS) emccd_queue_kernel(
        int n, const double* __restrict__ photons, const double* __restrict__ gain_map,
        const double* __restrict__ offset_map, smx_detector_params_t P, uint64_t seed,
        uint32_t frame, uint32_t pix_base, const uint32_t* __restrict__ frame_dev,
        double* __restrict__ E_out, OutT* __restrict__ adc_out) {
    __shared__ __align__(16) char s_lds[lds_bytes(EQ_PIX)];
    const BlockLds L = carve(s_lds, EQ_PIX);
    const int t = threadIdx.x;
    const long long base = (long long)blockIdx.x * EQ_PIX;
    if (frame_dev) frame += *frame_dev;
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    float E[EQ_PPT];
    bool in[EQ_PPT];
#pragma unroll
    for (int j = 0; j < EQ_PPT; ++j) {
        const long long i = base + t + j * EQ_THREADS;
        in[j] = i < n;
        E[j] = 0.0f;
        if (in[j]) {
            E[j] = expectation_f32(photons[i], P);
            if (E_out) E_out[i] = (double)E[j];
        }
    }
    float S[EQ_PPT], noise[EQ_PPT];
    emccd_block<EQ_THREADS, EQ_PPT>(
            L, E, in, [&](int loc) { return pix_base + (uint32_t)(base + loc); }, frame, k0, k1,
            P, S, noise);
    // readout noise and ADC (_epifm.py:1475-1484)
#pragma unroll
    for (int j = 0; j < EQ_PPT; ++j) {
        const long long i = base + t + j * EQ_THREADS;
        if (!in[j]) continue;
        const float gain = (float)(gain_map ? gain_map[i] : P.gain);
        const float offset = (float)(offset_map ? offset_map[i] : P.offset);
        adc_out[i] = (OutT)adc_f32(S[j], noise[j], P, gain, offset);
    }
}

// searchsorted(cdf, u, side='right') clamped to the last index: the draw of
// RandomState.choice(values, p=p) given its uniform u (cdf as numpy builds it).
__device__ inline int table_index(const double* __restrict__ cdf, int m, double u) {
    int lo = 0, hi = m;   // first index with cdf[idx] > u
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (cdf[mid] <= u) lo = mid + 1;
        else hi = mid;
    }
    return lo < m ? lo : m - 1;
}

// CCD / CMOS with caller-drawn numbers (_epifm.py:1443-1469).
__global__ void adc_parity_kernel(int n, const double* __restrict__ signal,
                                  const double* __restrict__ noise_in,
                                  const double* __restrict__ tvals,
                                  const double* __restrict__ tcdf, int tn,
                                  const double* __restrict__ gain_map,
                                  const double* __restrict__ offset_map, smx_detector_params_t P,
                                  double* __restrict__ adc_out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double noise = 0.0;
    if (noise_in) noise = tn > 0 ? tvals[table_index(tcdf, tn, noise_in[i])] : noise_in[i];
    const double gain = gain_map ? gain_map[i] : P.gain;
    const double offset = offset_map ? offset_map[i] : P.offset;
    adc_out[i] = adc_counts(signal[i] + noise, P, gain, offset);
}

// CCD (Gaussian readout noise) or CMOS (readout noise from a value table)
// with Philox randomness: Poisson(E) photo-electrons + noise, float32 ADC.
template <typename OutT>
__global__ void photon_philox_kernel(int n, const double* __restrict__ photons,
                                     const double* __restrict__ gain_map,
                                     const double* __restrict__ offset_map,
                                     smx_detector_params_t P, const double* __restrict__ tvals,
                                     const double* __restrict__ tcdf, int tn, uint64_t seed,
                                     uint32_t frame, uint32_t pix_base,
                                     const uint32_t* __restrict__ frame_dev,
                                     double* __restrict__ E_out, OutT* __restrict__ adc_out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (frame_dev) frame += *frame_dev;
    float ph = (float)photons[i];
    if (P.background_switch) ph += (float)P.background;
    const float E = (float)P.qe * ph;
    PixelRng R{pix_base + (uint32_t)i, frame, (uint32_t)seed, (uint32_t)(seed >> 32)};
    const smx::u32x4 r0 = R.block(0);
    float noise = 0.0f;
    if (tn > 0) noise = (float)tvals[table_index(tcdf, tn, smx::u01_53(r0.x, r0.y))];
    else if (P.readout_noise > 0.0) noise = (float)P.readout_noise * normal_f(r0.x, r0.y);
    int k = 0;
    if (E > 0.0f) k = E < 12.0f ? poisson_inversion(E, u01f(r0.z)) : poisson_ptrs(R, E);
    const float gain = (float)(gain_map ? gain_map[i] : P.gain);
    const float offset = (float)(offset_map ? offset_map[i] : P.offset);
    float x = (float)k + noise;
    x = fminf(x, (float)P.fullwell);
    x = x * __builtin_amdgcn_rcpf(gain) + offset;
    x = fminf(fmaxf(x, 0.0f), (float)P.adc_max);
    if (E_out) E_out[i] = (double)E;
    adc_out[i] = (OutT)x;
}

}  // namespace

extern "C" {

int smx_detector_expectation(int n, const double* photons, const smx_detector_params_t* params,
                             double* E_out, int* flag_out, hipStream_t stream) {
    if (n < 0 || !params || (n > 0 && (!photons || !E_out))) {
        smx::set_error("smx_detector_expectation: invalid arguments (n=%d)", n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    hipLaunchKernelGGL(prepare_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, photons,
                       *params, E_out, flag_out);
    SMX_CHECK_LAUNCH("prepare_kernel");
    return SMX_OK;
}

size_t smx_scan_workspace_bytes(int n) {
    size_t bytes = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (int*)nullptr, (int*)nullptr, n);
    return bytes;
}

int smx_exclusive_scan_i32(int n, const int* in, int* out, void* workspace, size_t bytes,
                           hipStream_t stream) {
    if (n < 0 || (n > 0 && (!in || !out || !workspace))) {
        smx::set_error("smx_exclusive_scan_i32: invalid arguments (n=%d)", n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    size_t need = smx_scan_workspace_bytes(n);
    if (bytes < need) {
        smx::set_error("smx_exclusive_scan_i32: workspace too small (%zu < %zu)", bytes, need);
        return SMX_EVALUE;
    }
    if (smx::check_hip(hipcub::DeviceScan::ExclusiveSum(workspace, need, in, out, n, stream),
                       "hipcub ExclusiveSum"))
        return SMX_ERUNTIME;
    return SMX_OK;
}

size_t smx_emccd_common_elems(void) { return 1 + RUNS_MAX; }

int smx_emccd_common_total(double E, int emgain, double* T_out, hipStream_t stream) {
    if (emgain <= 0 || !T_out) {
        smx::set_error("smx_emccd_common_total: invalid arguments (emgain=%d)", emgain);
        return SMX_EVALUE;
    }
    hipLaunchKernelGGL(emccd_common_total_kernel, dim3(1), dim3(64), 0, stream, E, emgain,
                       make_run_rule(emgain), T_out);
    SMX_CHECK_LAUNCH("emccd_common_total_kernel");
    return SMX_OK;
}

int smx_emccd_parity(int n, const double* E, const double* noise, const double* uniforms,
                     const int* uidx, const double* gain_map, const double* offset_map,
                     const smx_detector_params_t* params, double E_common,
                     const double* T_common, double* adc_out, double* signal_out,
                     int* status_dev, hipStream_t stream) {
    if (n < 0 || !params || params->emgain <= 0 ||
        (n > 0 && (!E || !uniforms || !uidx || !adc_out || !status_dev))) {
        smx::set_error("smx_emccd_parity: invalid arguments (n=%d)", n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    hipLaunchKernelGGL(emccd_parity_kernel, dim3((n + 3) / 4), dim3(256), 0, stream, n, E, noise,
                       uniforms, uidx, gain_map, offset_map, *params, make_run_rule(params->emgain),
                       E_common, T_common, adc_out, signal_out, status_dev);
    SMX_CHECK_LAUNCH("emccd_parity_kernel");
    return SMX_OK;
}

int smx_emccd_philox(int n, const double* photons, const double* gain_map,
                     const double* offset_map, const smx_detector_params_t* params,
                     uint64_t seed, uint32_t frame, uint32_t pix_base,
                     const uint32_t* frame_dev, double* E_out, void* adc_out,
                     int adc_is_float32, hipStream_t stream) {
    if (n < 0 || !params || params->emgain <= 0 || (n > 0 && (!photons || !adc_out))) {
        smx::set_error("smx_emccd_philox: invalid arguments (n=%d)", n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    const dim3 grid((unsigned)((n + EQ_PIX - 1) / EQ_PIX));
    if (adc_is_float32)
        hipLaunchKernelGGL(emccd_queue_kernel<float>, grid, dim3(EQ_THREADS), 0, stream, n,
                           photons, gain_map, offset_map, *params, seed, frame, pix_base,
                           frame_dev, E_out, (float*)adc_out);
    else
        hipLaunchKernelGGL(emccd_queue_kernel<double>, grid, dim3(EQ_THREADS), 0, stream, n,
                           photons, gain_map, offset_map, *params, seed, frame, pix_base,
                           frame_dev, E_out, (double*)adc_out);
    SMX_CHECK_LAUNCH("emccd_queue_kernel");
    return SMX_OK;
}

int smx_adc_parity(int n, const double* signal, const double* noise_in, const double* table_values,
                   const double* table_cdf, int table_n, const double* gain_map,
                   const double* offset_map, const smx_detector_params_t* params, double* adc_out,
                   hipStream_t stream) {
    if (n < 0 || !params || table_n < 0 || (table_n > 0 && (!table_values || !table_cdf)) ||
        (n > 0 && (!signal || !adc_out))) {
        smx::set_error("smx_adc_parity: invalid arguments (n=%d, table_n=%d)", n, table_n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    hipLaunchKernelGGL(adc_parity_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, signal,
                       noise_in, table_values, table_cdf, table_n, gain_map, offset_map, *params,
                       adc_out);
    SMX_CHECK_LAUNCH("adc_parity_kernel");
    return SMX_OK;
}

int smx_photon_detector_philox(int n, const double* photons, const double* gain_map,
                               const double* offset_map, const smx_detector_params_t* params,
                               const double* table_values, const double* table_cdf, int table_n,
                               uint64_t seed, uint32_t frame, uint32_t pix_base,
                               const uint32_t* frame_dev, double* E_out, void* adc_out,
                               int adc_is_float32, hipStream_t stream) {
    if (n < 0 || !params || table_n < 0 || (table_n > 0 && (!table_values || !table_cdf)) ||
        (n > 0 && (!photons || !adc_out))) {
        smx::set_error("smx_photon_detector_philox: invalid arguments (n=%d)", n);
        return SMX_EVALUE;
    }
    if (n == 0) return SMX_OK;
    if (adc_is_float32)
        hipLaunchKernelGGL(photon_philox_kernel<float>, dim3((n + 255) / 256), dim3(256), 0,
                           stream, n, photons, gain_map, offset_map, *params, table_values,
                           table_cdf, table_n, seed, frame, pix_base, frame_dev, E_out,
                           (float*)adc_out);
    else
        hipLaunchKernelGGL(photon_philox_kernel<double>, dim3((n + 255) / 256), dim3(256), 0,
                           stream, n, photons, gain_map, offset_map, *params, table_values,
                           table_cdf, table_n, seed, frame, pix_base, frame_dev, E_out,
                           (double*)adc_out);
    SMX_CHECK_LAUNCH("photon_philox_kernel");
    return SMX_OK;
}

}  // extern "C"
