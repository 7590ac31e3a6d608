// PSF tables: radial profiles (Born-Wolf / Gaussian, float64) and the
// summed-area table (SAT) of the (2n-1)^2 cartesian table for each profile.
//
// Reference: src/scopyon/_epifm.py:90-134 (radial profile, cartesian table),
//            _epifm.py:180-213 (Born-Wolf 100-point Riemann sum).
// The cartesian table is never stored: each SAT row pass evaluates its cells
// from the radial profile on the fly (same interpolation as interp1d).
#include "common.hpp"

#include <algorithm>
#include <utility>
#include <vector>

namespace {

constexpr int kRho = 100;   // _epifm.py:191

// J0(x * alpha * rho_n) for every (rho, radial sample) pair; independent of z.
__global__ void bw_j0_kernel(int nr, double res, double alpha, double* __restrict__ j0tab) {
    int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nr * kRho) return;
    int ri = idx % nr, n = idx / nr;
    double r = (double)ri * res;                   // numpy.arange(0, cut, res)[ri]
    double rho = (double)(n + 1) * (1.0 / kRho);   // numpy.arange(1, 101) * drho
    j0tab[idx] = j0((r * alpha) * rho);
}

// psf[z][r] = |sum_n J0[n][r] * exp(-2i z gamma rho^2) rho drho|^2 * alpha^2/pi.
// A block shares its depth's 100 phase factors (one sincos each, in LDS
// instead of one per radial sample) and its loads of J0 are coalesced:
// one depth of 1,000 samples 35 us with the factors evaluated per sample,
// 6 us so.
constexpr int kProfThreads = 64;
__global__ void __launch_bounds__(kProfThreads) bw_profile_kernel(
        int nr, int nz, const double* __restrict__ depths, double gamma, double scale,
        const double* __restrict__ j0tab, double* __restrict__ out) {
    __shared__ double2 s_y[kRho];
    const int ri = blockIdx.x * kProfThreads + threadIdx.x;
    const int zi = blockIdx.y;
    const double z = depths[zi];
    const double drho = 1.0 / kRho;
    for (int n = threadIdx.x; n < kRho; n += kProfThreads) {
        double rho = (double)(n + 1) * drho;
        // -2 * 1j * z * gamma * rho * rho: imaginary part (((-2z) gamma) rho) rho
        double theta = (((-2.0 * z) * gamma) * rho) * rho;
        double s, c;
        sincos(theta, &s, &c);
        s_y[n] = make_double2((c * rho) * drho, (s * rho) * drho);
    }
    __syncthreads();
    if (ri >= nr) return;
    double re = 0.0, im = 0.0;
#pragma unroll 20
    for (int n = 0; n < kRho; ++n) {
        const double j = j0tab[(size_t)n * nr + ri];
        const double2 y = s_y[n];
        re += y.x * j;
        im += y.y * j;
    }
    double mag = hypot(re, im);
    out[(size_t)zi * nr + ri] = (mag * mag) * scale;
}

__global__ void gaussian_profile_kernel(int nr, double res, double width, double denom,
                                        double* __restrict__ out) {
    int ri = blockIdx.x * blockDim.x + threadIdx.x;
    if (ri >= nr) return;
    double r = (double)ri * res;
    double q = r / width;
    out[ri] = exp(-0.5 * (q * q)) / denom;
}

// Linear interpolation of the radial profile at R (scipy interp1d 'linear':
// lo = clip(searchsorted_left(x, R), 1, n-1) - 1).
__device__ inline double interp_radial(const double* __restrict__ prof, int nr, double res,
                                       double R) {
    int m = (int)(R / res);
    if (m > nr) m = nr;
    if (m < 0) m = 0;
    // m := number of grid points x_k = k*res with x_k < R
    while (m < nr && (double)m * res < R) ++m;
    while (m > 0 && (double)(m - 1) * res >= R) --m;
    int k = m < 1 ? 1 : (m > nr - 1 ? nr - 1 : m);
    double xlo = (double)(k - 1) * res, xhi = (double)k * res;
    double ylo = prof[k - 1], yhi = prof[k];
    double slope = (yhi - ylo) / (xhi - xlo);
    return slope * (R - xlo) + ylo;
}

// Summed-area tables in three launches.  The table of one depth is 2000^2
// corners (32 MB), so the floor is writing it once (~7 us); the work is one
// evaluation of every cell per pass, two passes:
//   1. sat_segment_kernel: column sums of each segment of `seg` table rows;
//   2. sat_segment_scan_kernel: exclusive running sums over the segments;
//   3. sat_rows_kernel: a block walks its segment's rows with the running
//      column sums in registers (kCols columns a thread), scans each row
//      across the block and writes it, in the layout's column order, from LDS.
// Every segment of every table is a block, so one table already spreads over
// the chip (a serial column walk ran 32 waves for 274 us per table), and no
// pass re-reads row sums from memory.  A block takes ZB depths: a cell's
// radius, interval and offset do not depend on the depth, only the profile
// value and slope do (LDS).
// One 2000^2 table 312 us with one wave per row and a serial walk down the
// columns, 66 us so; 117 tables 14.5 ms before, 1.4 ms so.
constexpr int kCols = 4;              // columns per thread
constexpr int kSatMax = 1024 * kCols; // widest table of this form
static_assert(kSatMax == smx::SAT_SORTED_MAX, "sorted tables are built by this form only");

// Interval k and offset into it of the cell at (X, Y) on the radial grid
// (scipy interp1d 'linear': the interval [x_{k-1}, x_k] with x_{k-1} < R <= x_k,
// ends clamped), R limited to the last sample.
__device__ inline int radial_interval(double X2, double Y2, double rmax, double res,
                                      double inv_res, int nr, double& off) {
    double R = sqrt(X2 + Y2);
    if (R > rmax) R = rmax;
    int m = (int)(R * inv_res);       // within one of the number of x_k < R
    if ((double)m * res < R) ++m;
    if ((double)m * res < R) ++m;
    if (m > 0 && (double)(m - 1) * res >= R) --m;
    if (m > 0 && (double)(m - 1) * res >= R) --m;
    const int k = m < 1 ? 1 : (m > nr - 1 ? nr - 1 : m);
    off = R - (double)(k - 1) * res;
    return k;
}

// LDS copy of ZB profiles: value at x_{k-1} and slope of interval k, at k.
template <int ZB>
__device__ inline void load_profiles(double2* lds, const double* __restrict__ prof, int nr,
                                     double res, int z0, int nz) {
    for (int i = threadIdx.x; i < ZB * nr; i += blockDim.x) {
        const int z = i / nr, k = i - z * nr;
        if (k == 0 || z0 + z >= nz) continue;
        const double* p = prof + (size_t)(z0 + z) * nr;
        const double lo = p[k - 1];
        lds[i] = make_double2(lo, (p[k] - lo) / ((double)k * res - (double)(k - 1) * res));
    }
}

// Grid: (segments, depth groups, column panels).
constexpr int kSegThreads = 512;
template <int ZB>
__global__ void __launch_bounds__(kSegThreads) sat_segment_kernel(
        int nr, int nz, double res, const double* __restrict__ prof, int ntab, int seg, int nseg,
        double* __restrict__ sums) {
    extern __shared__ __align__(16) double2 s_prof[];
    const int z0 = blockIdx.y * ZB;
    load_profiles<ZB>(s_prof, prof, nr, res, z0, nz);
    __syncthreads();
    const double rmax = (double)(nr - 1) * res, inv_res = 1.0 / res;
    const int r0 = blockIdx.x * seg, r1 = min(r0 + seg, ntab);
    for (int col = blockIdx.z * kSegThreads + threadIdx.x; col < ntab;
         col += gridDim.z * kSegThreads) {
        const double X = (double)(col - (nr - 1)) * res, X2 = X * X;
        double acc[ZB];
#pragma unroll
        for (int z = 0; z < ZB; ++z) acc[z] = 0.0;
#pragma unroll 2
        for (int row = r0; row < r1; ++row) {
            const double Y = (double)(row - (nr - 1)) * res;
            double off;
            const int k = radial_interval(X2, Y * Y, rmax, res, inv_res, nr, off);
#pragma unroll
            for (int z = 0; z < ZB; ++z) {
                const double2 p = s_prof[z * nr + k];
                acc[z] += p.y * off + p.x;
            }
        }
#pragma unroll
        for (int z = 0; z < ZB; ++z)
            if (z0 + z < nz) sums[((size_t)(z0 + z) * nseg + blockIdx.x) * ntab + col] = acc[z];
    }
}

// Exclusive running sums over the segments, in place; one column per thread,
// loads eight segments ahead.
__global__ void __launch_bounds__(64) sat_segment_scan_kernel(int ntab, int nseg,
                                                              double* __restrict__ sums) {
    const int col = blockIdx.x * 64 + threadIdx.x;
    if (col >= ntab) return;
    double* s = sums + (size_t)blockIdx.y * nseg * ntab + col;
    double acc = 0.0;
    int i = 0;
    for (; i + 16 <= nseg; i += 16) {
        double v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = s[(size_t)(i + j) * ntab];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            s[(size_t)(i + j) * ntab] = acc;
            acc += v[j];
        }
    }
    for (; i < nseg; ++i) {
        const double v = s[(size_t)i * ntab];
        s[(size_t)i * ntab] = acc;
        acc += v;
    }
}

// Grid: (segments, depth groups); threads: ntab / kCols rounded up to waves.
// STAGED: a row goes out through LDS in layout order (coalesced); else straight
// from the registers (layouts padded beyond what LDS holds).
template <int ZB, bool STAGED>
__global__ void __launch_bounds__(1024) sat_rows_kernel(int nr, int nz, double res,
                                                        const double* __restrict__ prof, int ntab,
                                                        int seg, int nseg,
                                                        const double* __restrict__ sums,
                                                        smx::SatLayout L,
                                                        const int* __restrict__ places,
                                                        size_t sat_stride,
                                                        double* __restrict__ sat) {
    // sorted layout (smx::SAT_SORTED_MAX): the axis order comes from `places`
    auto place_of = [&](int a) { return places ? places[a] : L.place(a); };
    extern __shared__ __align__(16) double2 s_prof[];
    double* const s_wave = (double*)(s_prof + ZB * nr);  // wave totals
    double* const s_row = s_wave + 16;                   // one row in layout order
    const int z0 = blockIdx.y * ZB, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int waves = blockDim.x >> 6;
    load_profiles<ZB>(s_prof, prof, nr, res, z0, nz);
    // column 0 of every row and the layout's unused places hold 0
    if (STAGED)
        for (int i = t; i < L.width; i += blockDim.x) s_row[i] = 0.0;
    const double rmax = (double)(nr - 1) * res, inv_res = 1.0 / res;
    double X2[kCols], C[ZB][kCols];
    int place[kCols];
#pragma unroll
    for (int j = 0; j < kCols; ++j) {
        const int col = t * kCols + j;
        const double X = (double)(col - (nr - 1)) * res;
        X2[j] = X * X;
        place[j] = place_of(min(col + 1, ntab));
#pragma unroll
        for (int z = 0; z < ZB; ++z)
            C[z][j] = col < ntab && z0 + z < nz
                              ? sums[((size_t)(z0 + z) * nseg + blockIdx.x) * ntab + col]
                              : 0.0;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        for (int z = 0; z < ZB && z0 + z < nz; ++z) {
            double* T = sat + (size_t)(z0 + z) * sat_stride;
            double* row0 = T + (size_t)place_of(0) * L.width;
            for (int i = t; i < L.width; i += blockDim.x) row0[i] = 0.0;
            if (places) {   // the zeros, and row 0 of the last column
                for (int i = t; i < L.width; i += blockDim.x) T[(size_t)L.width * L.width + i] = 0.0;
                if (t == 0) T[(size_t)L.width * (L.width + 1) + place_of(0)] = 0.0;
            }
        }
    }
    const int r0 = blockIdx.x * seg, r1 = min(r0 + seg, ntab);
    for (int row = r0; row < r1; ++row) {
        const double Y = (double)(row - (nr - 1)) * res, Y2 = Y * Y;
        const int prow = place_of(row + 1);
#pragma unroll
        for (int j = 0; j < kCols; ++j) {
            double off;
            const int k = radial_interval(X2[j], Y2, rmax, res, inv_res, nr, off);
            if (t * kCols + j < ntab)
#pragma unroll
                for (int z = 0; z < ZB; ++z) {
                    const double2 p = s_prof[z * nr + k];
                    C[z][j] += p.y * off + p.x;
                }
        }
#pragma unroll
        for (int z = 0; z < ZB; ++z) {
            if (z0 + z >= nz) break;
            double run[kCols];
            double tot = 0.0;
#pragma unroll
            for (int j = 0; j < kCols; ++j) {
                tot += C[z][j];
                run[j] = tot;
            }
            double v = tot;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const double a = __shfl_up(v, o, 64);
                if (lane >= o) v += a;
            }
            if (lane == 63) s_wave[wave] = v;
            __syncthreads();   // also: the last row is read out of s_row
            double base = v - tot;
            // sums of the waves before this one, in wave order
            double before = 0.0;
            for (int w = 0; w < waves; ++w)
                if (w < wave) before += s_wave[w];
            base += before;
            double* out = sat + (size_t)(z0 + z) * sat_stride + (size_t)prow * L.width;
            if (places && t == (ntab - 1) / kCols) {   // the row's last corner
                const int j = (ntab - 1) % kCols;
                double c = 0.0;
#pragma unroll
                for (int y = 0; y < kCols; ++y) c = y == j ? base + run[y] : c;
                sat[(size_t)(z0 + z) * sat_stride + (size_t)L.width * (L.width + 1) + prow] = c;
            }
            double* to = STAGED ? s_row : out;
#pragma unroll
            for (int j = 0; j < kCols; ++j)
                if (t * kCols + j < ntab) to[place[j]] = base + run[j];
            if (!STAGED && t == 0) out[place_of(0)] = 0.0;
            __syncthreads();
            if (STAGED)
                for (int i = t; i < L.width; i += blockDim.x)
                    __builtin_nontemporal_store(s_row[i], out + i);
        }
    }
}

// Tables wider than kSatMax cells (radial cutoffs above 2 um): row scans to
// memory, then a running sum down each column.
// One wave per table row: inclusive scan of the row's cells (evaluated from
// the radial profile) -> rowsum[row][col+1]; rowsum[row][0] = 0.
__global__ void __launch_bounds__(256) sat_row_kernel(int nr, double res, const double* __restrict__ prof,
                                                      int ntab, double* __restrict__ rowsum) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row = blockIdx.x * 4 + wave;
    const int zi = blockIdx.y;
    if (row >= ntab) return;
    const int side = ntab + 1;
    const double* p = prof + (size_t)zi * nr;
    double* out = rowsum + ((size_t)zi * ntab + row) * side;
    const double rmax = (double)(nr - 1) * res;
    const double Y = (double)(row - (nr - 1)) * res;
    double carry = 0.0;
    if (lane == 0) out[0] = 0.0;
    for (int c0 = 0; c0 < ntab; c0 += 64) {
        int col = c0 + lane;
        double v = 0.0;
        if (col < ntab) {
            double X = (double)(col - (nr - 1)) * res;
            double R = sqrt(X * X + Y * Y);
            if (R > rmax) R = rmax;
            v = interp_radial(p, nr, res, R);
        }
        // wave-wide inclusive scan
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            double o = __shfl_up(v, off, 64);
            if (lane >= off) v += o;
        }
        double s = carry + v;
        if (col < ntab) out[col + 1] = s;
        carry = __shfl(s, 63, 64);
    }
}

// 64 columns per wave: running sum down the rows -> SAT in the chosen layout.
__global__ void __launch_bounds__(64) sat_col_kernel(int ntab, const double* __restrict__ rowsum,
                                                     smx::SatLayout L, size_t sat_stride,
                                                     double* __restrict__ sat) {
    const int side = ntab + 1;
    const int col = blockIdx.x * 64 + threadIdx.x;
    const int zi = blockIdx.y;
    if (col >= side) return;
    const double* rs = rowsum + (size_t)zi * ntab * side;
    double* out = sat + (size_t)zi * sat_stride;
    double acc = 0.0;
    out[L.index(0, col)] = 0.0;
    int row = 0;
    for (; row + 4 <= ntab; row += 4) {
        double a0 = rs[(size_t)(row + 0) * side + col];
        double a1 = rs[(size_t)(row + 1) * side + col];
        double a2 = rs[(size_t)(row + 2) * side + col];
        double a3 = rs[(size_t)(row + 3) * side + col];
        acc += a0; out[L.index(row + 1, col)] = acc;
        acc += a1; out[L.index(row + 2, col)] = acc;
        acc += a2; out[L.index(row + 3, col)] = acc;
        acc += a3; out[L.index(row + 4, col)] = acc;
    }
    for (; row < ntab; ++row) {
        acc += rs[(size_t)row * side + col];
        out[L.index(row + 1, col)] = acc;
    }
}

// Rows per segment.  One height for any number of tables: it sets the order in
// which a column is added up, and a table's bits must not depend on what else is
// built with it.  Whole build in us with 8 / 16 / 32 rows: 64 tables 830 / 750 /
// 735, 53 tables 720 / 670 / 715; one table 52 / 66, of it the row kernel's 250 /
// 125 / 63 blocks 25 / 44 / 82.
constexpr int kSegRows = 16;

template <int ZB, bool STAGED>
int sat_build(const double* radial, int nz, int nr, double res, int ntab, smx::SatLayout L,
              const int* places, size_t stride, double* sums, double* sat, hipStream_t stream) {
    const int seg = kSegRows, nseg = (ntab + seg - 1) / seg, nzb = (nz + ZB - 1) / ZB;
    const size_t lds = sizeof(double2) * ZB * (size_t)nr;
    // every block computes the slopes of its profiles, so a block takes whole
    // rows (64 tables in segments of 32 rows: 168 us, 270 us in panels) unless that
    // leaves CUs idle
    const int panels = nseg * nzb >= 512 ? 1 : (ntab + kSegThreads - 1) / kSegThreads;
    if (ZB > 1 && 2 * lds <= (64u << 10))
        hipLaunchKernelGGL(sat_segment_kernel<2 * ZB>, dim3(nseg, (nzb + 1) / 2, panels),
                           dim3(kSegThreads), 2 * lds, stream, nr, nz, res, radial, ntab, seg, nseg, sums);
    else
        hipLaunchKernelGGL(sat_segment_kernel<ZB>, dim3(nseg, nzb, panels), dim3(kSegThreads),
                           lds, stream, nr, nz, res, radial, ntab, seg, nseg, sums);
    SMX_CHECK_LAUNCH("sat_segment_kernel");
    hipLaunchKernelGGL(sat_segment_scan_kernel, dim3((ntab + 63) / 64, nz), dim3(64), 0, stream,
                       ntab, nseg, sums);
    SMX_CHECK_LAUNCH("sat_segment_scan_kernel");
    const int threads = ((ntab + kCols - 1) / kCols + 63) / 64 * 64;
    hipLaunchKernelGGL((sat_rows_kernel<ZB, STAGED>), dim3(nseg, nzb), dim3(threads),
                       lds + sizeof(double) * (size_t)(16 + (STAGED ? L.width : 0)), stream, nr,
                       nz, res, radial, ntab, seg, nseg, sums, L, places, stride, sat);
    SMX_CHECK_LAUNCH("sat_rows_kernel");
    return SMX_OK;
}

int sat_build_any(const double* radial, int nz, int nr, double res, int ntab, smx::SatLayout L,
                  const int* places, size_t stride, double* sums, double* sat, hipStream_t stream) {
    // two depths' profiles a block and the staged row while 64 KB of LDS
    // hold them (they do up to 1 um radial cutoff and beyond)
    const size_t profile = sizeof(double2) * (size_t)nr;
    const size_t row = sizeof(double) * (size_t)(16 + L.width), most = 64 << 10;
    if (nz > 1 && 2 * profile + row <= most)
        return sat_build<2, true>(radial, nz, nr, res, ntab, L, places, stride, sums, sat, stream);
    if (profile + row <= most)
        return sat_build<1, true>(radial, nz, nr, res, ntab, L, places, stride, sums, sat, stream);
    return sat_build<1, false>(radial, nz, nr, res, ntab, L, places, stride, sums, sat, stream);
}

}  // namespace

extern "C" {

int smx_psf_radial_born_wolf(const double* depths, int nz, int nr, double res, double alpha,
                             double gamma, double scale, double* j0_work, double* out,
                             hipStream_t stream) {
    if (nz < 0 || nr < 2 || !depths || !j0_work || !out) {
        smx::set_error("smx_psf_radial_born_wolf: invalid arguments (nz=%d, nr=%d)", nz, nr);
        return SMX_EVALUE;
    }
    if (nz == 0) return SMX_OK;
    int total = nr * kRho;
    hipLaunchKernelGGL(bw_j0_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, nr, res,
                       alpha, j0_work);
    SMX_CHECK_LAUNCH("bw_j0_kernel");
    hipLaunchKernelGGL(bw_profile_kernel, dim3((nr + kProfThreads - 1) / kProfThreads, nz),
                       dim3(kProfThreads), 0, stream, nr, nz, depths, gamma, scale, j0_work, out);
    SMX_CHECK_LAUNCH("bw_profile_kernel");
    return SMX_OK;
}

int smx_psf_radial_gaussian(int nr, double res, double width, double* out, hipStream_t stream) {
    if (nr < 2 || !(width > 0.0) || !out) {
        smx::set_error("smx_psf_radial_gaussian: invalid arguments (nr=%d, width=%g)", nr, width);
        return SMX_EVALUE;
    }
    double denom = 2.0 * 3.141592653589793 * width * width;
    hipLaunchKernelGGL(gaussian_profile_kernel, dim3((nr + 255) / 256), dim3(256), 0, stream, nr,
                       res, width, denom, out);
    SMX_CHECK_LAUNCH("gaussian_profile_kernel");
    return SMX_OK;
}

size_t smx_psf_sat_elems(int nr, int period) {
    if (nr < 2) return 0;
    return smx::make_sat_layout(2 * nr, period).elems();
}

size_t smx_psf_sat_workspace_bytes(int nr, int nz) {
    if (nr < 2 || nz < 0) return 0;
    size_t ntab = 2 * (size_t)nr - 1;
    if (ntab <= (size_t)kSatMax)   // segment sums
        return (ntab + kSegRows - 1) / kSegRows * ntab * (size_t)nz * sizeof(double);
    return ntab * (ntab + 1) * (size_t)nz * sizeof(double);
}

int smx_psf_sat_build(const double* radial, int nz, int nr, double res, int period,
                      double* workspace, double* sat, hipStream_t stream) {
    if (nz < 0 || nr < 2 || period < 1 || !radial || !workspace || !sat) {
        smx::set_error("smx_psf_sat_build: invalid arguments (nz=%d, nr=%d, period=%d)", nz, nr,
                       period);
        return SMX_EVALUE;
    }
    if (nz == 0) return SMX_OK;
    int ntab = 2 * nr - 1;
    smx::SatLayout L = smx::make_sat_layout(ntab + 1, period);
    if (ntab <= kSatMax)
        return sat_build_any(radial, nz, nr, res, ntab, L, nullptr, L.elems(), workspace, sat, stream);
    hipLaunchKernelGGL(sat_row_kernel, dim3((ntab + 3) / 4, nz), dim3(256), 0, stream, nr, res,
                       radial, ntab, workspace);
    SMX_CHECK_LAUNCH("sat_row_kernel");
    hipLaunchKernelGGL(sat_col_kernel, dim3((ntab + 1 + 63) / 64, nz), dim3(64), 0, stream, ntab,
                       workspace, L, L.elems(), sat);
    SMX_CHECK_LAUNCH("sat_col_kernel");
    return SMX_OK;
}

size_t smx_psf_sat_sorted_elems(int nr) {
    if (nr < 2 || 2 * nr - 1 > smx::SAT_SORTED_MAX) return 0;
    return smx::sat_sorted_elems(2 * nr);
}

int smx_sat_sorted_places(int nr, double ratio, int* places) {
    if (nr < 2 || 2 * nr - 1 > smx::SAT_SORTED_MAX || !(ratio > 1.0) || !places) {
        smx::set_error("smx_sat_sorted_places: invalid arguments (nr=%d, ratio=%g)", nr, ratio);
        return SMX_EVALUE;
    }
    // phase of every corner; within a phase the order of the pixels
    std::vector<std::pair<double, int>> order(2 * (size_t)nr);
    for (int b = 0; b < 2 * nr; ++b) order[b] = {(double)b - ratio * floor((double)b / ratio), b};
    std::stable_sort(order.begin(), order.end(),
                     [](const auto& x, const auto& y) { return x.first < y.first; });
    for (size_t k = 0; k < order.size(); ++k) places[order[k].second] = (int)k;
    return SMX_OK;
}

int smx_psf_sat_build_sorted(const double* radial, int nz, int nr, double res, const int* places,
                             double* workspace, double* sat, hipStream_t stream) {
    if (nz < 0 || nr < 2 || 2 * nr - 1 > smx::SAT_SORTED_MAX || !radial || !places || !workspace ||
        !sat) {
        smx::set_error("smx_psf_sat_build_sorted: invalid arguments (nz=%d, nr=%d)", nz, nr);
        return SMX_EVALUE;
    }
    if (nz == 0) return SMX_OK;
    return sat_build_any(radial, nz, nr, res, 2 * nr - 1, smx::make_sat_layout(2 * nr, 1), places,
                         smx::sat_sorted_elems(2 * nr), workspace, sat, stream);
}

}  // extern "C"
