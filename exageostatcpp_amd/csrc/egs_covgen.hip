// Covariance generation on gfx950: the device side of
// Kernel<T>::GenerateCovarianceMatrix (Kernel.hpp:93-97) for every lower tile of
// Sigma at once (the reference submits one dcmg task per tile,
// dcmg-codelet.cpp:47-74, and evaluates GSL's K_nu per element on CPU threads).
// Arithmetic is FP64 throughout; the store converts to the tile's storage
// precision.  Orders without a closed form go through the tables of
// matern_table_eval.
#include <algorithm>

#include "egs_common.hpp"
#include "egs_kernels.hpp"
#include "egs_matern.hpp"

namespace egs {

// ------------------------------------------------------------------------
// Matern tables (see matern_table_eval): one wave per row, each lane
// evaluating K_nu at one Chebyshev node; grid (row groups, slots).  The sums
// over the nodes are compensated and a_0 is kept to twice the precision: a
// row's own error is common to all entries it serves, so that the jumps
// between rows, unlike rounding noise, add up in z'Sigma^-1 z (at 40,000
// locations and nu = 1, 16 nodes and one double for a_0 put 1.3e-11 into the
// log-likelihood).  Bound: latency, 28 us whatever the size (K_nu, then
// the sums over its nodes).
// ------------------------------------------------------------------------
constexpr int kNodes = 64;
constexpr int kDegree = kTabDegree;
constexpr int kRowsPerGroup = kThreads / kNodes;

// Powers of t in T_k(t): kCheb[k][m].
__constant__ const double kCheb[kDegree + 1][kDegree + 1] = {
    {1}, {0, 1}, {-1, 0, 2}, {0, -3, 0, 4}, {1, 0, -8, 0, 8}, {0, 5, 0, -20, 0, 16}, {-1, 0, 18, 0, -48, 0, 32},
    {0, -7, 0, 56, 0, -112, 0, 64}, {1, 0, -32, 0, 160, 0, -256, 0, 128}, {0, 9, 0, -120, 0, 432, 0, -576, 0, 256},
    {-1, 0, 50, 0, -400, 0, 1120, 0, -1280, 0, 512}};

// d where row r begins: 8 log2(d) + 2 d + 80 = r.  Newton in log(d) (convex,
// increasing; FP32 is enough, the rows' fits overlap).
__device__ __forceinline__ float table_edge(float r) {
    float x = fminf((r - 80.0f) * 0.0866434f, 5.0f);   // log(d) without the 2 d term: from above
    for (int it = 0; it < 12; ++it) {
        const float d = expf(x);
        x -= (11.5415603f * x + 2.0f * d + 80.0f - r) / (11.5415603f + 2.0f * d);
    }
    return expf(x);
}

// sum += a * b with the rounding errors in err (two-product, two-sum)
__device__ __forceinline__ void add_product(double &sum, double &err, double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b;
    const double pe = fma(a, b, -p);
    const double t = sum + p;
    const double z = t - sum;
    err += ((sum - (t - z)) + (p - z)) + pe;
    sum = t;
}

__device__ __forceinline__ void matern_table(double *tabs, const MaternParams &prm) {
    __shared__ double s_cos[4 * kNodes];   // cos(pi m / (2 kNodes))
    __shared__ double s_f[kRowsPerGroup][kNodes];
    __shared__ double s_c[kRowsPerGroup][kDegree + 1], s_e[kRowsPerGroup][kDegree + 1];
    const int slot = blockIdx.y;
    if (slot >= prm.ntab) return;
    const int pair = prm.tab_pair[slot];
    const int g = threadIdx.x / kNodes, j = threadIdx.x % kNodes;
    const int row = blockIdx.x * kRowsPerGroup + g;
    s_cos[threadIdx.x] = cospi((double) threadIdx.x / (2.0 * kNodes));
    const double d0 = table_edge((float) row), d1 = table_edge((float) row + 1.0f);
    const double pad = 2e-3 * (d1 * d1 - d0 * d0);
    const double lo = d0 * d0 - pad, hi = d1 * d1 + pad;
    const double mid = (float) (0.5 * (lo + hi)), half = 0.5 * (hi - lo);
    __syncthreads();
    const double d = sqrt(fma(half, s_cos[2 * j + 1], mid));
    s_f[g][j] = prm.con[pair] * pow(d, prm.nu[pair]) * bessel_knu(prm.nu[pair], d);
    __syncthreads();
    if (j <= kDegree) {
        double c = 0.0, e = 0.0;
        for (int q = 0; q < kNodes; ++q) add_product(c, e, s_f[g][q], s_cos[(j * (2 * q + 1)) % (4 * kNodes)]);
        s_c[g][j] = c * (j == 0 ? 1.0 / kNodes : 2.0 / kNodes);   // powers of two: exact
        s_e[g][j] = e * (j == 0 ? 1.0 / kNodes : 2.0 / kNodes);
    }
    __syncthreads();
    if (row >= kTabRows) return;
    double *tab = tabs + (int64_t) slot * kTabDoubles;
    double *out = tab + row * kTabWidth;
    if (j <= kDegree) {
        double a = 0.0, e = 0.0;
        for (int k = kDegree; k >= j; --k) {
            add_product(a, e, s_c[g][k], kCheb[k][j]);
            e += s_e[g][k] * kCheb[k][j];
        }
        if (j == 0) {
            out[0] = a + e;
            out[1] = (a - (a + e)) + e;
        } else {
            a += e;
            for (int m = 0; m < j; ++m) a /= half;
            out[1 + j] = a;
        }
    } else if (j == kDegree + 1) {
        reinterpret_cast<float *>(tab + kTabRows * kTabWidth)[row] = (float) mid;
    }
}

__global__ void __launch_bounds__(kThreads) matern_table_kernel(double *tabs, MaternParams prm,
                                                                const MaternParams *prm_dev) {
    const MaternParams p = prm_dev ? *prm_dev : prm;
    matern_table(tabs, p);
}

__global__ void __launch_bounds__(kThreads) matern_table_batch_kernel(const CovJob *jobs) {
    const CovJob &J = jobs[blockIdx.z];   // in memory: its parameters are indexed
    matern_table(J.tabs, J.prm);
}

constexpr int kTableGroups = (kTabRows + kRowsPerGroup - 1) / kRowsPerGroup;

void launch_matern_tables(double *tabs, const MaternParams &prm, const MaternParams *prm_dev, hipStream_t s) {
    const int slots = prm_dev ? (prm.kernel == 1 ? kTabSlots : 1) : prm.ntab;
    if (slots == 0) return;
    hipLaunchKernelGGL(matern_table_kernel, dim3(kTableGroups, slots), dim3(kThreads), 0, s, tabs, prm, prm_dev);
}

// One workgroup per 64-row strip and `cols` columns of a tile: the strip's row
// locations and the tables sit in LDS, the columns' locations pass through it
// 256 at a time; each wave writes 64 consecutive rows (512 bytes in FP64) of
// one column at a time.
//
// Bound: FP64 VALU and, for orders without a closed form, the table's LDS
// reads (96 bytes per entry, 64 neighbouring rows share few table rows).
// Measured with K_nu per entry -> with the table: 10,007 locations, nu 0.83,
// ts 384: 6.14 -> 0.13 ms (plus 0.02 ms for the table); 45,001, nu 0.55, ts
// 960 with the FP64 copy: 69 -> 2.6 ms.  24 regions of 500-3,000 in turn:
// 1.08 ms -> 16 us each (one strip of 64 x ts per workgroup left most of the
// GPU idle there; see the split in launch_covgen_tiles).
template <int kTabs, bool kSphere>
__device__ __forceinline__ void covgen_strip(const CovJob &a, const MaternParams &prm, int cols, int part) {
    constexpr int kStageCols = 256;
    __shared__ double s_cx[kStageCols], s_cy[kStageCols], s_cz[kStageCols];
    __shared__ __align__(16) double s_tab[kTabs > 0 ? kTabs * kTabDoubles : 1];
    const int ts = a.map.ts;
    const int2 ij = a.pairs[blockIdx.y];
    const int sbr = blockIdx.x;
    const int64_t r0 = (int64_t) ij.x * ts + sbr * kBlk;
    const int c_beg = part * cols, c_end = min(ts, c_beg + cols);
    const int t = threadIdx.x;
    const bool three_d = a.loc.z != nullptr;
    if (kTabs > 0 && prm.ntab > 0)
        for (int e = t; e < kTabs * kTabDoubles; e += kThreads) s_tab[e] = a.tabs[e];

    const int r = t % kBlk;
    const int64_t gr = r0 + r;
    const bool row_pad = gr >= a.n;
    StagedLoc row{0.0, 0.0, 0.0};
    if (!row_pad) row = stage_location<kSphere>(a.loc.x[gr], a.loc.y[gr], three_d ? a.loc.z[gr] : 0.0);
    const uint8_t store = a.map.store[ij.x * a.map.nt + ij.y];
    char *tile = a.map.base + a.map.off[ij.x * a.map.nt + ij.y];
    const int64_t sig_base = ((int64_t) ij.x * (ij.x + 1) / 2 + ij.y) * ts * ts;
    for (int cb = c_beg; cb < c_end; cb += kStageCols) {
        const int64_t gc0 = (int64_t) ij.y * ts + cb;
        const int ncol = min(kStageCols, c_end - cb);
        __syncthreads();   // the tables are staged; the columns before are done
        if (t < ncol && gc0 + t < a.n) {
            const StagedLoc col = stage_location<kSphere>(a.loc.x[gc0 + t], a.loc.y[gc0 + t],
                                                 three_d ? a.loc.z[gc0 + t] : 0.0);
            s_cx[t] = col.x;
            s_cy[t] = col.y;
            s_cz[t] = col.z;
        }
        __syncthreads();
#pragma unroll 1
        for (int cc = t / kBlk; cc < ncol; cc += kThreads / kBlk) {
            const int64_t gc = gc0 + cc;
            double v;
            if (row_pad || gc >= a.n) {
                v = (gr == gc) ? 1.0 : 0.0;
            } else {
                const StagedLoc col{s_cx[cc], s_cy[cc], s_cz[cc]};
                v = staged_covariance<(kTabs > 0), kSphere>(prm, 0, staged_separation<kSphere>(row, col, three_d), s_tab);
            }
            const int64_t idx = (int64_t) (sbr * kBlk + r) + (int64_t) (cb + cc) * ts;
            if (store == kStoreF64) reinterpret_cast<double *>(tile)[idx] = v;
            else reinterpret_cast<float *>(tile)[idx] = (float) v;
            if (a.sig64) a.sig64[sig_base + idx] = v;
        }
    }
}

// The bivariate kernel: a thread takes a pair of locations, whose distance
// serves the 2 x 2 covariances of their variables (the two cross terms are
// equal); 32 row locations, 16 column locations at a time.  9,001 locations on
// the sphere, orders 0.5 and 1: 14.3 ms with a distance and K_nu per entry,
// 0.67 ms so.
constexpr int kBivThreads = 512;

template <int kTabs, bool kSphere>
__device__ __forceinline__ void covgen_strip_biv(const CovJob &a, const MaternParams &prm, int cols, int part) {
    constexpr int kRowLocs = kBlk / 2, kColStep = kBivThreads / kRowLocs;
    __shared__ __align__(16) double s_tab[kTabs > 0 ? kTabs * kTabDoubles : 1];
    const int ts = a.map.ts;
    const int2 ij = a.pairs[blockIdx.y];
    const int sbr = blockIdx.x;
    const int64_t r0 = (int64_t) ij.x * ts + sbr * kBlk, c0 = (int64_t) ij.y * ts;
    const int c_beg = part * cols, c_end = min(ts, c_beg + cols);
    const int t = threadIdx.x;
    if (kTabs > 0 && prm.ntab > 0) {
        for (int e = t; e < kTabs * kTabDoubles; e += kBivThreads) s_tab[e] = a.tabs[e];
        __syncthreads();
    }
    const int r = t % kRowLocs;
    const int64_t gr = r0 + 2 * r;       // n is even: a location's two rows are both real or both padding
    const bool row_pad = gr >= a.n;
    StagedLoc row{0.0, 0.0, 0.0};
    if (!row_pad) row = stage_location<kSphere>(a.loc.x[gr >> 1], a.loc.y[gr >> 1], 0.0);
    const uint8_t store = a.map.store[ij.x * a.map.nt + ij.y];
    char *tile = a.map.base + a.map.off[ij.x * a.map.nt + ij.y];
    const int64_t sig_base = ((int64_t) ij.x * (ij.x + 1) / 2 + ij.y) * ts * ts;
#pragma unroll 1
    for (int cc = c_beg + 2 * (t / kRowLocs); cc < c_end; cc += 2 * kColStep) {
        const int64_t gc = c0 + cc;
        double v00, v01, v11;
        if (row_pad || gc >= a.n) {
            v00 = v11 = (gr == gc) ? 1.0 : 0.0;
            v01 = 0.0;
        } else {
            const StagedLoc col = stage_location<kSphere>(a.loc.x[gc >> 1], a.loc.y[gc >> 1], 0.0);
            const double q = staged_separation<kSphere>(row, col, false);
            v00 = staged_covariance<(kTabs > 0), kSphere>(prm, 0, q, s_tab);
            v01 = staged_covariance<(kTabs > 0), kSphere>(prm, 1, q, s_tab);
            v11 = staged_covariance<(kTabs > 0), kSphere>(prm, 3, q, s_tab);
        }
        const int64_t idx = (int64_t) (sbr * kBlk + 2 * r) + (int64_t) cc * ts;   // even: ts and cc are
        const f64x2 left{v00, v01}, right{v01, v11};
        if (store == kStoreF64) {
            *reinterpret_cast<f64x2 *>(reinterpret_cast<double *>(tile) + idx) = left;
            *reinterpret_cast<f64x2 *>(reinterpret_cast<double *>(tile) + idx + ts) = right;
        } else {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<f32x2 *>(reinterpret_cast<float *>(tile) + idx) = f32x2{(float) v00, (float) v01};
            *reinterpret_cast<f32x2 *>(reinterpret_cast<float *>(tile) + idx + ts) = f32x2{(float) v01, (float) v11};
        }
        if (a.sig64) {
            *reinterpret_cast<f64x2 *>(a.sig64 + sig_base + idx) = left;
            *reinterpret_cast<f64x2 *>(a.sig64 + sig_base + idx + ts) = right;
        }
    }
}

// One problem's tiles, or those of a batch (blockIdx.z: its jobs, `parts` column
// parts each; workgroups past a job's tiles exit at once).  The parameters come
// from device memory when prm_dev is given (a captured graph replays with new
// theta).
template <int kTabs, bool kSphere>
__global__ void __launch_bounds__(kThreads, 4) covgen_tiles_kernel(CovJob a, int cols) {
    const MaternParams prm = a.prm_dev ? *a.prm_dev : a.prm;
    covgen_strip<kTabs, kSphere>(a, prm, cols, blockIdx.z);
}

template <int kTabs, bool kSphere>
__global__ void __launch_bounds__(kThreads, 4) covgen_tiles_batch_kernel(const CovJob *jobs, int cols, int parts) {
    const CovJob J = scalar_load(jobs + blockIdx.z / parts);
    if ((int) blockIdx.y < J.npairs) covgen_strip<kTabs, kSphere>(J, J.prm, cols, blockIdx.z % parts);
}

template <int kTabs, bool kSphere>
__global__ void __launch_bounds__(kBivThreads, kTabs < 3 ? 4 : 2) covgen_tiles_biv_kernel(CovJob a, int cols) {
    const MaternParams prm = a.prm_dev ? *a.prm_dev : a.prm;
    covgen_strip_biv<kTabs, kSphere>(a, prm, cols, blockIdx.z);
}

template <int kTabs, bool kSphere>
__global__ void __launch_bounds__(kBivThreads, kTabs < 3 ? 4 : 2)
    covgen_tiles_biv_batch_kernel(const CovJob *jobs, int cols, int parts) {
    const CovJob J = scalar_load(jobs + blockIdx.z / parts);
    if ((int) blockIdx.y < J.npairs) covgen_strip_biv<kTabs, kSphere>(J, J.prm, cols, blockIdx.z % parts);
}

// A rows x cols column-major block (ld = rows) of Sigma(l1, l2) starting at
// matrix row row_off and column col_off: the plugin interface
// Kernel<T>::GenerateCovarianceMatrix evaluated on the device.
struct CovRectArgs {
    double *out;
    int rows, cols;
    int64_t row_off, col_off;
    MaternParams prm;
    Locs l1, l2;
    int three_d;
};

__global__ void __launch_bounds__(kThreads) covgen_rect_kernel(CovRectArgs a) {
    const int64_t idx = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    const int64_t total = (int64_t) a.rows * a.cols;
    if (idx >= total) return;
    const int i = (int) (idx % a.rows);
    const int j = (int) (idx / a.rows);
    a.out[idx] = covariance_entry(a.prm, a.l1, a.l2, a.row_off + i, a.col_off + j, a.three_d != 0);
}

// A strip's columns are split over workgroups until `tiles` tiles fill the GPU
// (kFill: eight per CU); whole strips stage the tables once each.  Returns the
// 64-column blocks per workgroup.
static int covgen_blocks(int nsb, int64_t tiles) {
    constexpr int kFill = 2048;
    const int want = (int) std::min<int64_t>(nsb, (kFill + nsb * tiles - 1) / (nsb * tiles));
    return (nsb + want - 1) / want;
}

void launch_covgen_tiles(const CovJob &job, hipStream_t s) {
    if (job.npairs <= 0) return;
    const int nsb = job.map.ts / kBlk, per = covgen_blocks(nsb, job.npairs);
    const dim3 grid(nsb, job.npairs, (nsb + per - 1) / per);
    // a captured launch serves every theta: as many tables as the kernel may need
    const MaternParams &prm = job.prm;
    const int tables = job.prm_dev ? (prm.kernel == 1 ? kTabSlots : 1) : prm.ntab;
    using Kernel = void (*)(CovJob, int);
    static const Kernel univariate[2][2] = {{covgen_tiles_kernel<0, false>, covgen_tiles_kernel<1, false>},
                                            {covgen_tiles_kernel<0, true>, covgen_tiles_kernel<1, true>}};
    static const Kernel bivariate[2][kTabSlots + 1] = {
        {covgen_tiles_biv_kernel<0, false>, covgen_tiles_biv_kernel<1, false>, covgen_tiles_biv_kernel<2, false>,
         covgen_tiles_biv_kernel<3, false>},
        {covgen_tiles_biv_kernel<0, true>, covgen_tiles_biv_kernel<1, true>, covgen_tiles_biv_kernel<2, true>,
         covgen_tiles_biv_kernel<3, true>}};
    const bool sphere = prm.metric == 1;
    if (prm.kernel == 1)
        hipLaunchKernelGGL(bivariate[sphere][tables], grid, dim3(kBivThreads), 0, s, job, per * kBlk);
    else
        hipLaunchKernelGGL(univariate[sphere][tables], grid, dim3(kThreads), 0, s, job, per * kBlk);
}

bool covgen_same_launch(const MaternParams &a, const MaternParams &b) {
    return a.kernel == b.kernel && a.ntab == b.ntab && (a.metric == 1) == (b.metric == 1);
}

void launch_covgen_batch(const CovJob *jobs, const CovJob *h_jobs, int count, hipStream_t s) {
    if (count <= 0) return;
    const MaternParams &prm = h_jobs[0].prm;
    if (prm.ntab > 0)
        hipLaunchKernelGGL(matern_table_batch_kernel, dim3(kTableGroups, prm.ntab, count), dim3(kThreads), 0, s, jobs);
    int64_t tiles = 0;
    int most = 0;
    for (int b = 0; b < count; ++b) {
        tiles += h_jobs[b].npairs;
        most = std::max(most, h_jobs[b].npairs);
    }
    const int nsb = h_jobs[0].map.ts / kBlk, per = covgen_blocks(nsb, tiles), parts = (nsb + per - 1) / per;
    const dim3 grid(nsb, most, count * parts);
    using Kernel = void (*)(const CovJob *, int, int);
    static const Kernel univariate[2][2] = {
        {covgen_tiles_batch_kernel<0, false>, covgen_tiles_batch_kernel<1, false>},
        {covgen_tiles_batch_kernel<0, true>, covgen_tiles_batch_kernel<1, true>}};
    static const Kernel bivariate[2][kTabSlots + 1] = {
        {covgen_tiles_biv_batch_kernel<0, false>, covgen_tiles_biv_batch_kernel<1, false>,
         covgen_tiles_biv_batch_kernel<2, false>, covgen_tiles_biv_batch_kernel<3, false>},
        {covgen_tiles_biv_batch_kernel<0, true>, covgen_tiles_biv_batch_kernel<1, true>,
         covgen_tiles_biv_batch_kernel<2, true>, covgen_tiles_biv_batch_kernel<3, true>}};
    const bool sphere = prm.metric == 1;
    if (prm.kernel == 1)
        hipLaunchKernelGGL(bivariate[sphere][prm.ntab], grid, dim3(kBivThreads), 0, s, jobs, per * kBlk, parts);
    else
        hipLaunchKernelGGL(univariate[sphere][prm.ntab], grid, dim3(kThreads), 0, s, jobs, per * kBlk, parts);
}

void launch_covgen_rect(double *out, int rows, int cols, int64_t row_off, int64_t col_off, const MaternParams &prm,
                        const double *x1, const double *y1, const double *z1, const double *x2, const double *y2,
                        const double *z2, hipStream_t s) {
    CovRectArgs a;
    a.out = out;
    a.rows = rows;
    a.cols = cols;
    a.row_off = row_off;
    a.col_off = col_off;
    a.prm = prm;
    a.l1 = Locs{x1, y1, z1};
    a.l2 = Locs{x2, y2, z2};
    a.three_d = (z1 != nullptr && z2 != nullptr);
    const int64_t total = (int64_t) rows * cols;
    if (total <= 0) return;
    const unsigned blocks = (unsigned) ((total + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(covgen_rect_kernel, dim3(blocks), dim3(kThreads), 0, s, a);
}

}  // namespace egs
