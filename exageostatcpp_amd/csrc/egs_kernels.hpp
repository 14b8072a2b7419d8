// Host-side launchers of the gfx950 kernels.  All launches are asynchronous on
// the given stream; shapes are validated by the caller (egs_capi.cpp) before
// any launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "egs_common.hpp"
#include "egs_matern.hpp"

namespace egs {

// One problem's share of a batched step (FP64 plan): step k of the tiled
// Cholesky on the tiles of `map`, with that problem's update order (pairs),
// diagonal-block inverses of tile k, the tile column's ticket and flags
// (launch_tile_column), not-SPD flag (n: its real dimension); with step 0, the
// forward solve's vector, words (launch_init) and partials.
struct BatchJob {
    TileMap map;
    int k;
    const int2 *pairs;
    double *winv_k;
    int *sync;
    int *info;
    int64_t n;
    double *z;
    double *pending;
    double *partials;
};

// ---- covariance generation (egs_covgen.hip)
// Tables of the orders prm marks (MaternParams::tab) into tabs, kTabSlots of
// kTabDoubles; prm_dev as in launch_covgen_tiles.
void launch_matern_tables(double *tabs, const MaternParams &prm, const MaternParams *prm_dev, hipStream_t s);
// The lower tiles (i, j) of pairs; rows and columns >= n are identity padding.
// loc.z may be null (2D).  tabs: the tables of prm (launch_matern_tables, earlier
// on the same stream).  sig64 (may be null): also writes every generated tile in
// FP64 to sig64 + (i*(i+1)/2 + j) * ts * ts, column-major.  prm_dev, when given,
// holds the parameters in device memory (read instead of prm, so that a captured
// launch can be replayed for another theta).
struct CovJob {
    TileMap map;
    const int2 *pairs;
    int npairs;
    MaternParams prm;
    Locs loc;
    int64_t n;
    double *tabs;
    double *sig64;
    const MaternParams *prm_dev;
};
void launch_covgen_tiles(const CovJob &job, hipStream_t s);
// The tables and tiles of `count` jobs of one tile size, in device memory (and
// h_jobs, the same on the host), that a launch can serve together: one table and
// one covariance launch.  24 regions of 500-3,000, 18 with tables: 0.91 -> 0.19 ms.
bool covgen_same_launch(const MaternParams &a, const MaternParams &b);
void launch_covgen_batch(const CovJob *jobs, const CovJob *h_jobs, int count, hipStream_t s);
void launch_covgen_rect(double *out, int rows, int cols, int64_t row_off, int64_t col_off, const MaternParams &prm,
                        const double *x1, const double *y1, const double *z1, const double *x2, const double *y2,
                        const double *z2, hipStream_t s);

// ---- tiled Cholesky (egs_chol.hip)
// Triangular solve X L_kk^T = B for row blocks [g0, g0 + count) of tile column k
// (global 64-row block g lives in tile g / nsb at row (g % nsb) * 64).
void launch_trsm_rows(const TileMap &map, int k, int64_t g0, int count, const double *winv_k, hipStream_t s,
                      bool x_f32 = false, bool f32mfma = false);
// Both panel solves of a mixed plan in one launch on FP64 MFMA: count64 FP64
// row blocks from g0 on, then count32 FP32 ones.
void launch_trsm_rows_mixed(const TileMap &map, int k, int64_t g0, int count64, int count32, const double *winv_k,
                            hipStream_t s);
// Trailing update C_ij -= L_ik L_jk^T for npairs lower tiles with i >= j > k;
// p64 (may be null): read panel k from its contiguous FP64 copy (tile i at
// p64 + (i-k-1) ts^2) instead of from the tiles.  critical: the next panel waits
// for these tiles.
// panels = 2 (FP64 plans): with the panels k and k + 1.
void launch_update(const TileMap &map, const double *p64, const int2 *pairs, int npairs, int k, bool critical,
                   hipStream_t s, int panels = 1);
// Its 96 x 192-block form (egs_update.hip), for ts % 192 == 0.
bool update192_supported(int ts);
void launch_update192(const TileMap &map, const double *p64, const int2 *pairs, int npairs, int k, int panels,
                      hipStream_t s);

// ---- triangular solves and reductions (egs_solve.hip)
// What a factorization (sync, null for none) and a solve (pending, null for none)
// start from: sync_ints zeros in sync, winv_words empty words (kPending) of the
// inverses; no failed minor and no lost wait in info (null: as they are); z = src
// (n values) padded with zeros to npad, or as it is when src is null, and pending
// (npad + 1 doubles) emptied.
struct InitJob {
    int *sync;
    int64_t sync_ints;
    double *winv;
    int64_t winv_words;
    int *info;
    double *z;
    const double *src;
    int64_t n, npad;
    double *pending;
};
void launch_init(const InitJob &job, hipStream_t s);
// Several jobs (device memory), `most` the largest extent of any (init_extent).
int64_t init_extent(const InitJob &job);
void launch_init_batch(const InitJob *jobs, int count, int64_t most, hipStream_t s);
// z = L^{-1} z and z = L^{-T} z with the factor's tiles (mixed: some may be FP32)
// and its diagonal-block inverses.  partials (may be null): of 64-row block b,
// partials[2b] = sum log L_ii (L_ii > 0), partials[2b+1] = y_b . y_b.
// info: as for launch_tile_column.
void launch_forward(const TileMap &map, bool mixed, const double *winv, double *z, double *pending, double *partials,
                    int *info, hipStream_t s);
void launch_backward(const TileMap &map, bool mixed, const double *winv, double *z, double *pending, int *info,
                     hipStream_t s);
// out = L e (lower-triangular product over the tiles).
void launch_trmv(const TileMap &map, const double *e, double *out, hipStream_t s);
// out[r] = sum_c Sigma(l1_r, l2_c) x[c] for r < rows, c < cols (kriging mean);
// out[-1] = *word.
void launch_cov_gemv(double *out, int64_t rows, int64_t cols, const MaternParams &prm, const double *x1,
                     const double *y1, const double *z1, const double *x2, const double *y2, const double *z2,
                     const double *xv, const double *tabs, const double *word, hipStream_t s);
// partial[cb * npad + r] = sum over column chunk cb of Sigma(r, c) v[c] (FP64,
// regenerated from the locations); matvec_chunks(n) chunks.
void launch_cov_matvec(double *partial, const double *v, int64_t n, int64_t npad, const MaternParams &prm,
                       const double *x, const double *y, const double *z, hipStream_t s);
int matvec_chunks(int64_t n);
// Cholesky of diagonal tile k in place, in 64 x 64 blocks, with the inverses of
// its diagonal blocks in winv_k, and the panel solve of the first `blocks` 64-row
// blocks below it, FP64 ones (tile_column_solves_rows: whether that many should
// be; the others take launch_trsm_rows afterwards).  sync: the column's ticket and flags,
// tile_column_sync_ints(ts) ints, zero before the launch, winv_k empty
// (launch_init).  info[0]: the first minor without a positive pivot, if it is 0;
// info[1] becomes 1 if a wait between workgroups ends in vain (Patience).  Tiles
// above 1,152 take several launches, none of which has such waits, and no rows below.
int tile_column_sync_ints(int ts);
bool tile_column_solves_rows(int ts, int blocks);
void launch_tile_column(const TileMap &map, int k, double *winv_k, int *sync, int *info, int64_t n, int blocks,
                        hipStream_t s);
// Batched steps over problems of tile size ts (jobs in device memory, those
// with most tiles first): factor tile column k of each of njobs, then apply
// panel k to tile columns k+1 .. of the first nrest, the ones that have them
// (rest = the largest nt - k - 1; jobs with fewer tiles exit early).
void launch_step_batch(const BatchJob *jobs, int njobs, int ts, int rest, int nrest, hipStream_t s);
// The forward solves of the jobs of step 0, with their partials (max_nt: the
// first job's tiles).
void launch_forward_batch(const BatchJob *jobs, int njobs, int ts, int max_nt, hipStream_t s);
// The log-det partials alone, of an FP64 or mixed factor (partials[2b+1] = 0).
void launch_diag_logdet(const TileMap &map, double *partials, hipStream_t s);
// Sigma v from the FP64 lower tiles written by launch_covgen_tiles: one
// workgroup per tile (i, j) writes T_ij v_j to prow[t * ts ..] and, off the
// diagonal, T_ij' v_i to pcol[t * ts ..] (t = i*(i+1)/2 + j).
void launch_sigma_tile_matvec(const double *sig64, const int2 *pairs, int npairs, int ts, const double *v,
                              double *prow, double *pcol, hipStream_t s);
// out[g] = base[g] + scale * (Sigma v)[g] for g < n (0 for padding rows), summing
// the tile partials of row block g / ts in a fixed order.
void launch_sigma_reduce(double *out, const double *base, double scale, const double *prow, const double *pcol,
                         int nt, int ts, int64_t n, int64_t npad, hipStream_t s);
// out = base + scale * (sum of the chunk partials), padding rows set to zero.
void launch_matvec_reduce(double *out, const double *base, double scale, const double *partial, int nchunks,
                          int64_t n, int64_t npad, hipStream_t s);
// partial[b] (b < dot_blocks()) = fixed-order partial sums of x . y.
int dot_blocks();
void launch_dot(const double *x, const double *y, int64_t n, double *partial, hipStream_t s);
// y = a x + b y
void launch_axpby(double *y, const double *x, double a, double b, int64_t n, hipStream_t s);
// Mixed-precision factorization pieces (egs_mixed.hip).
// inv_scale[slot * ts + r] = 2^(e+1) for the largest |x| = f 2^e of row r of panel
// slot; bmax[slot * (ts/192) + b] the largest of 192-row block b; pmax[k] raised
// to the largest of the panel (bits of a float, must start at zero).
void launch_panel_rowscale(const TileMap &map, int k, float *inv_scale, float *bmax, unsigned *pmax,
                           hipStream_t s);
void launch_zero_u32(unsigned *p, int n, hipStream_t s);
// Panel k to FP64 and FP32 column-major copies and 16-bit hi/lo row-major parts:
// FP16 of the row-scaled values when inv_scale is given, BF16 of the values otherwise.
// With inv_scale, p8 (optional) receives the OCP e4m3 byte of each row-scaled
// value, row-major like the 16-bit parts.
void launch_panel_convert(const TileMap &map, int k, double *p64, float *p32, uint16_t *p16h, uint16_t *p16l,
                          uint8_t *p8, const float *inv_scale, hipStream_t s);
void launch_update192_f32(const TileMap &map, const float *p32, const int2 *pairs, int npairs, int k, hipStream_t s);
// Operands of the 16-bit update: split FP16 (hi*hi + hi*lo + lo*hi of the
// row-scaled parts), one FP16 product of the row-scaled hi parts, the choice
// between the two per 192 x 192 block (one product when bmax(A rows) *
// bmax(B rows) <= tau * pmax[k]^2), or one BF16 product of unscaled values.
// FP16 forms undo the row scales with inv_scale.
// The C64 forms update an FP64 tile: the split product, one product, or the
// choice per block.
enum Operands {
    kSplitF16 = 0, kSingleF16 = 1, kAdaptiveF16 = 2, kSingleBF16 = 3, kSplitF16C64 = 4, kSingleF16C64 = 5,
    kAdaptiveF16C64 = 6
};
// C -= A B^T from the 16-bit parts of panel k.  The single and per-block forms
// add the number of 192 x 192 blocks they update with the split product to
// counts[0], with one product to counts[1] and with one FP8 product to
// counts[2].  kAdaptiveF16 with tau8 > 0 takes one e4m3 product from p8 (the
// panel's FP8 copy) for blocks with bmax(A) bmax(B) <= tau8 pmax[k]^2.
void launch_update192_16(const TileMap &map, const uint16_t *p16h, const uint16_t *p16l, const float *inv_scale,
                         const float *bmax, const unsigned *pmax, float tau, const uint8_t *p8, float tau8,
                         const int2 *pairs, int npairs, int k, Operands op, unsigned long long *counts,
                         hipStream_t s);
// e = LAPACK dlarnv(3, iseed) N(0,1) values (48-bit LCG stream, Box-Muller).
void launch_dlarnv_normal(double *e, int64_t n, uint64_t seed48, hipStream_t s);
// dst = src (n doubles), padding [n, npad) with zeros.
void launch_copy_pad(double *dst, const double *src, int64_t n, int64_t npad, hipStream_t s);

}  // namespace egs
