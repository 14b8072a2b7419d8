// Tiled Cholesky factorization on gfx950 (the reference calls
// CHAMELEON_dpotrf_Tile(Lower) at ChameleonDense.cpp:29: POTRF of the diagonal
// tile, TRSM of the panel below it, SYRK/GEMM of the trailing tiles).
//
// Step k of the factorization:
//   * the diagonal tile is factored in 64 x 64 blocks, which also leaves the
//     64 x 64 inverses of its diagonal blocks, and a short panel below it is
//     solved by the same launch (tile_column_kernel; tiles above kOneLaunchTile:
//     block_column_kernel);
//   * a longer panel is solved by one workgroup per 64-row block, marching over
//     the 64-column blocks of L_kk and applying the 64 x 64 inverses
//     (trsm_rows_kernel);
//   * the trailing tiles are updated with FP64 MFMA: update192 (egs_update.hip)
//     when ts is a multiple of 192 and the tiles are many, else update_kernel
//     here, one workgroup per 64 x 64 output block (or half of one) with K = ts.
// The panel solves and update_kernel contract through wg_gemm_nt: four waves each
// own a 32 x 32 quadrant of the 64 x 64 output (16 columns of 32 rows); K is staged
// through LDS in chunks of 32 columns, double buffered, with the loads of the next
// two chunks in flight during a chunk's MFMAs.  The tasks of a diagonal tile
// multiply whole 64 x 64 blocks in LDS.
#include <algorithm>

#include "egs_common.hpp"
#include "egs_kernels.hpp"

namespace egs {

constexpr int kKc = 32;          // K chunk staged in LDS
constexpr int kLdsPad = 65;      // LDS row stride for 64-wide panels

// Staging buffers of the contractions, in the compute type.
template <typename CT>
struct Smem {
    CT a[2][kKc][kLdsPad];
    CT b[2][kKc][kLdsPad];
};
using GemmSmem = Smem<double>;

// The 16 x 16 x 4 MFMA of a compute type: element v of lane l's result holds
// column col(l / 16, v) of the second operand's 16 and row l % 16 of the first.
template <typename CT>
struct Mfma;
template <>
struct Mfma<double> {
    typedef f64x4 vec;
    static __device__ __forceinline__ vec mul(double b, double a, vec c) { return mfma_f64(b, a, c); }
    static __device__ __forceinline__ int col(int lk, int v) { return lk + 4 * v; }
};
template <>
struct Mfma<float> {
    typedef f32x4 vec;
    static __device__ __forceinline__ vec mul(float b, float a, vec c) { return mfma_f32(b, a, c); }
    static __device__ __forceinline__ int col(int lk, int v) { return 4 * lk + v; }
};

// A kRows x 64 block over the workgroup's four waves: with 64 rows wave w holds
// the 32 x 32 quadrant (w & 1, w >> 1), with 32 rows columns 16 w .. +15;
// v[ni][mi] are its 16 x 16 tiles.
template <typename CT, int kRows>
struct Acc {
    static constexpr int kNi = kRows / 32;
    typename Mfma<CT>::vec v[kNi][2];
    static __device__ __forceinline__ int row0() { return kRows == 64 ? ((threadIdx.x >> 6) & 1) * 32 : 0; }
    static __device__ __forceinline__ int col0() {
        return kRows == 64 ? (threadIdx.x >> 7) * 32 : (threadIdx.x >> 6) * 16;
    }
};
using Acc64 = Acc<double, 64>;

template <typename CT, int kRows>
__device__ __forceinline__ void acc_zero(Acc<CT, kRows> &acc) {
#pragma unroll
    for (int i = 0; i < Acc<CT, kRows>::kNi; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc.v[i][j] = typename Mfma<CT>::vec{0, 0, 0, 0};
}

// Visit every (row, col, value) of the accumulator.
template <typename CT, int kRows, typename F>
__device__ __forceinline__ void acc_foreach(const Acc<CT, kRows> &acc, F f) {
    using A = Acc<CT, kRows>;
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int ni = 0; ni < A::kNi; ++ni)
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                f(A::row0() + mi * 16 + lr, A::col0() + ni * 16 + Mfma<CT>::col(lk, v), acc.v[ni][mi][v]);
}

// acc += the product of K columns of a (rows) and b (columns), element (row,
// k) at k * kLdsPad + row.
template <typename CT, int kRows, int K>
__device__ __forceinline__ void lds_product(Acc<CT, kRows> &acc, const CT *a, const CT *b) {
    using A = Acc<CT, kRows>;
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll 4
    for (int kk = 0; kk < K; kk += 4) {
        CT x[2], y[A::kNi];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) x[mi] = a[(kk + lk) * kLdsPad + A::row0() + mi * 16 + lr];
#pragma unroll
        for (int ni = 0; ni < A::kNi; ++ni) y[ni] = b[(kk + lk) * kLdsPad + A::col0() + ni * 16 + lr];
#pragma unroll
        for (int ni = 0; ni < A::kNi; ++ni)
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) acc.v[ni][mi] = Mfma<CT>::mul(y[ni], x[mi], acc.v[ni][mi]);
    }
}

template <bool kShared> __device__ __forceinline__ double load_as(const double *p) {
    if constexpr (kShared) return load_shared(p);
    else return *p;
}

// acc += A (kRows x K, column-major, lda) * B (64 x K, column-major, ldb)^T; K a
// multiple of 64.  K chunks of 32 columns go through LDS, double buffered; two
// chunks' loads are in flight in registers while one is multiplied (these
// kernels run on few workgroups, so each has to hide its own memory latency).
// Against one chunk in flight, and with C, B_j and W_j loaded ahead of the
// products (below): the panel solve of 60 row blocks of 960 columns 268 -> 246
// us, one evaluation of 1,600 locations 0.85 -> 0.79 ms, of 20,000 55.4 ->
// 53.8 ms.
template <typename CT, int kRows, bool kShared = false, typename TA>
__device__ void wg_gemm_nt(Acc<CT, kRows> &acc, const TA *__restrict__ A, int64_t lda, const double *__restrict__ B,
                           int64_t ldb, int K, Smem<CT> &sm) {
    constexpr int kA = kRows * kKc / kThreads, kB = kBlk * kKc / kThreads;   // elements per thread and chunk
    const int t = threadIdx.x;
    const int arow = t % kRows, acol = t / kRows;
    const int brow = t % kBlk, bcol = t / kBlk;
    const TA *Ap = A + arow + (int64_t) acol * lda;
    const double *Bp = B + brow + (int64_t) bcol * ldb;
    TA ra[2][kA];
    double rb[2][kB];
    auto issue = [&](int set, int c) {
        const int64_t k0 = (int64_t) c * kKc;
#pragma unroll
        for (int q = 0; q < kA; ++q) ra[set][q] = Ap[(k0 + q * (kThreads / kRows)) * lda];
#pragma unroll
        for (int q = 0; q < kB; ++q) rb[set][q] = load_as<kShared>(Bp + (k0 + q * (kThreads / kBlk)) * ldb);
    };
    auto stage = [&](int set) {
#pragma unroll
        for (int q = 0; q < kA; ++q) sm.a[set][acol + q * (kThreads / kRows)][arow] = (CT) ra[set][q];
#pragma unroll
        for (int q = 0; q < kB; ++q) sm.b[set][bcol + q * (kThreads / kBlk)][brow] = (CT) rb[set][q];
    };
    const int nch = K / kKc;   // even
    issue(0, 0);
    issue(1, 1);
    stage(0);
    __syncthreads();
    for (int c0 = 0; c0 < nch; c0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = c0 + u;
            if (c + 2 < nch) issue(u, c + 2);
            lds_product<CT, kRows, kKc>(acc, &sm.a[u][0][0], &sm.b[u][0][0]);
            if (c + 1 < nch) stage(u ^ 1);
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------------
// Panel solve X L_kk^T = B of kRows rows: marching over the 64-column blocks of
// L_kk, X_j = (B_j - X_0..j-1 L_j,0..j-1^T) W_j^T with the 64 x 64 inverses W.
// CT is the compute type (FP32 for FP32 rows of univariate mixed plans: 1.8x
// the rate; the bivariate field's error grew 3-14x with it).  B_j and W_j are
// loaded ahead of the product they wait for.  `wait` blocks until row block j
// of L_kk's earlier columns (row) and W_j (inverse) are there; kAhead: they are
// from the start.  T goes through the product's LDS (sm), so that a workgroup
// fits beside the trailing update's.
// ------------------------------------------------------------------------
struct NoWait {
    static constexpr bool kAhead = true;
    __device__ __forceinline__ void row(int) const {}
    __device__ __forceinline__ void inverse(int) const {}
};

template <typename CT, int kRows, typename TX, typename Wait>
__device__ __forceinline__ void solve_rows(const double *T, int ts, int nsb, TX *X, const double *winv_k, Smem<CT> &sm,
                                           const Wait &wait) {
    using A = Acc<CT, kRows>;
    const int row = threadIdx.x & 63, w = threadIdx.x >> 6;
    CT *sT = &sm.a[0][0][0], *sW = &sm.b[0][0][0];
    for (int jb = 0; jb < nsb; ++jb) {
        TX *Xj = X + (int64_t) jb * kBlk * ts;
        const double *W = winv_k + (int64_t) jb * kBlk * kBlk;
        double wv[16];
        TX xv[A::kNi * 8];
        int e = 0;
        A acc;
        acc_zero(acc);
        acc_foreach(acc, [&](int r, int c, CT) { xv[e++] = Xj[r + (int64_t) c * ts]; });
        if (Wait::kAhead)
#pragma unroll
            for (int q = 0; q < 16; ++q) wv[q] = W[row + (w + 4 * q) * kBlk];
        if (jb > 0) {
            wait.row(jb);
            wg_gemm_nt<CT, kRows, !Wait::kAhead>(acc, X, ts, T + jb * kBlk, ts, jb * kBlk, sm);
        }
        e = 0;
        acc_foreach(acc, [&](int r, int c, CT v) { sT[c * kLdsPad + r] = (CT) xv[e++] - v; });
        if (!Wait::kAhead) {
            wait.inverse(jb);
#pragma unroll
            for (int q = 0; q < 16; ++q) wv[q] = load_shared(W + row + (w + 4 * q) * kBlk);
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) sW[(w + 4 * q) * kLdsPad + row] = (CT) wv[q];
        __syncthreads();
        acc_zero(acc);
        lds_product<CT, kRows, kBlk>(acc, sT, sW);
        acc_foreach(acc, [&](int r, int c, CT v) { Xj[r + (int64_t) c * ts] = (TX) v; });
        __syncthreads();
    }
}

// Row block g of kRows rows of the tile column's panel.
template <typename CT, int kRows, typename TX>
__device__ __forceinline__ void solve_row_block(const TileMap &map, int k, int64_t g, const double *winv_k,
                                                Smem<CT> &sm) {
    const int per = map.ts / kRows;
    TX *X = reinterpret_cast<TX *>(map.base + map.off[(g / per) * map.nt + k]) + (g % per) * kRows;
    solve_rows<CT, kRows>(tile_f64(map, k, k), map.ts, map.ts / kBlk, X, winv_k, sm, NoWait());
}

// Row blocks of kRows rows from g0 on, one workgroup each.  A row block's solve
// is a chain of ts / 64 dependent steps bound by its CU's MFMA rate; in 32-row
// blocks a short panel spreads over twice the CUs, each with half the MFMA work
// (and the same loads of L_kk).
template <typename CT, int kRows, typename TX>
__global__ void __launch_bounds__(kThreads) trsm_rows_kernel(TileMap map, int k, int64_t g0, const double *winv_k) {
    __shared__ Smem<CT> sm;
    solve_row_block<CT, kRows, TX>(map, k, g0 + blockIdx.x, winv_k, sm);
}

// FP64 rows [g0, g0 + count64) and FP32 rows after them in one launch, both
// on FP64 MFMA, so that the two panel solves of a mixed plan run side by side
// rather than one after the other (each is a chain of ts / 64 dependent steps
// per workgroup).  Plans whose FP32 rows are solved on FP32 MFMA keep two
// launches: that kernel's lighter workgroups (33 KB of LDS) would otherwise
// carry the FP64 body's LDS and registers.
template <int kRows>
__global__ void __launch_bounds__(kThreads) trsm_rows_mixed_kernel(TileMap map, int k, int64_t g0, int count64,
                                                                   const double *winv_k) {
    __shared__ GemmSmem sm;
    if ((int) blockIdx.x < count64)
        solve_row_block<double, kRows, double>(map, k, g0 + blockIdx.x, winv_k, sm);
    else
        solve_row_block<double, kRows, float>(map, k, g0 + blockIdx.x, winv_k, sm);
}

// ------------------------------------------------------------------------
// Trailing update, FP64.
// ------------------------------------------------------------------------
// p64 (may be null): read panel k from its contiguous FP64 copy (tile i at
// p64 + (i - k - 1) ts^2) instead of from the tiles.
// panels = 2 (without p64): with the panels k and k + 1.
template <int kRows>
__device__ __forceinline__ void update_body(const TileMap &map, const double *p64, const int2 *pairs, int k, int bx,
                                            int by, int panels) {
    __shared__ GemmSmem sm;
    const int ts = map.ts;
    const int per = ts / kRows;
    const int2 ij = pairs[by];
    const int r0 = (bx % per) * kRows, sbm = r0 / kBlk;
    const int sbn = bx / per;
    if (ij.x == ij.y && sbm < sbn) return;
    if (sbm >= map.blocks(ij.x) || sbn >= map.blocks(ij.y)) return;
    double *C = tile_f64(map, ij.x, ij.y) + r0 + (int64_t) sbn * kBlk * ts;
    const int64_t tt = (int64_t) ts * ts;
    const double *A = (p64 ? p64 + (ij.x - k - 1) * tt : tile_f64(map, ij.x, k)) + r0;
    const double *B = (p64 ? p64 + (ij.y - k - 1) * tt : tile_f64(map, ij.y, k)) + sbn * kBlk;
    // C's values are loaded ahead of the product, whose loads follow in flight
    using Block = Acc<double, kRows>;
    Block acc;
    acc_zero(acc);
    double cv[Block::kNi * 8];
    int q = 0;
    acc_foreach(acc, [&](int r, int c, double) { cv[q++] = C[r + (int64_t) c * ts]; });
    wg_gemm_nt(acc, A, ts, B, ts, ts, sm);
    if (panels == 2)
        wg_gemm_nt(acc, tile_f64(map, ij.x, k + 1) + r0, ts, tile_f64(map, ij.y, k + 1) + sbn * kBlk, ts, ts, sm);
    q = 0;
    acc_foreach(acc, [&](int r, int c, double v) { C[r + (int64_t) c * ts] = cv[q++] - v; });
}

template <int kRows>
__global__ void __launch_bounds__(kThreads) update_kernel(TileMap map, const double *p64, const int2 *pairs, int k,
                                                          int panels) {
    update_body<kRows>(map, p64, pairs, k, blockIdx.x, blockIdx.y, panels);
}

// A panel of fewer 64-row blocks than this is solved in 32-row blocks (with
// more, every CU already holds a row block, and 64-row blocks load L_kk half
// as often per flop).
constexpr int kHalfRowsBelow = 256;

void launch_trsm_rows(const TileMap &map, int k, int64_t g0, int count, const double *winv_k, hipStream_t s, bool x_f32,
                      bool f32mfma) {
    if (count <= 0) return;
    using Kernel = void (*)(TileMap, int, int64_t, const double *);
    static const Kernel kernels[3][2] = {
        {trsm_rows_kernel<double, 64, double>, trsm_rows_kernel<double, 32, double>},
        {trsm_rows_kernel<double, 64, float>, trsm_rows_kernel<double, 32, float>},
        {trsm_rows_kernel<float, 64, float>, trsm_rows_kernel<float, 32, float>}};
    const int half = count < kHalfRowsBelow;
    hipLaunchKernelGGL(kernels[x_f32 ? (f32mfma ? 2 : 1) : 0][half], dim3((unsigned) (count << half)), dim3(kThreads),
                       0, s, map, k, g0 << half, winv_k);
}

void launch_trsm_rows_mixed(const TileMap &map, int k, int64_t g0, int count64, int count32, const double *winv_k,
                            hipStream_t s) {
    if (count64 + count32 <= 0) return;
    const int half = count64 + count32 < kHalfRowsBelow;
    hipLaunchKernelGGL(half ? trsm_rows_mixed_kernel<32> : trsm_rows_mixed_kernel<64>,
                       dim3((unsigned) ((count64 + count32) << half)), dim3(kThreads), 0, s, map, k, g0 << half,
                       count64 << half, winv_k);
}

// Up to this many 64 x 64 blocks (three per CU) are updated one workgroup each:
// they run at once, and end sooner than the 96 x 192 blocks of update192, of
// which a few tiles have too few (measured: 8 tiles of 384 44 against 68 us,
// 20 75 / 79, 40 119 / 122, 160 407 / 334; 2 tiles of 960 94 / 154, 4 184 /
// 166; 64 tiles of 192 39 / 46).  On the critical path, where the update shares
// the GPU with the one before, the shorter workgroups pay up to twice as many
// (6,001 locations, tiles of 960: 5.2 against 5.4 ms).
// Up to half a block per CU are updated in halves of 32 rows, on twice the CUs
// with half of a chunk's products each (what bounds such a launch is one
// workgroup's way through ts / 32 chunks): 400 locations, tiles of 320, 192.0 ->
// 186.0 us, 1,600 552 -> 524 us; up to two per CU measured alike there and at
// 10,007 (8.75 ms), and a mixed evaluation of 45,001, whose halves wait for room
// beside the 16-bit updates, 0.6% slower.
constexpr int kSmallBlocks = 768, kSmallBlocksCritical = 1800, kHalfBlocks = 128;

void launch_update(const TileMap &map, const double *p64, const int2 *pairs, int npairs, int k, bool critical,
                   hipStream_t s, int panels) {
    if (npairs <= 0) return;
    const int nsb = map.ts / kBlk;
    if (update192_supported(map.ts) &&
        (int64_t) npairs * nsb * nsb > (critical ? kSmallBlocksCritical : kSmallBlocks)) {
        launch_update192(map, p64, pairs, npairs, k, panels, s);
        return;
    }
    const bool half = (int64_t) npairs * nsb * nsb <= kHalfBlocks;
    hipLaunchKernelGGL(half ? update_kernel<32> : update_kernel<64>, dim3((nsb << half) * nsb, npairs), dim3(kThreads), 0,
                       s, map, p64, pairs, k, panels);
}

// ------------------------------------------------------------------------
// Cholesky and inverse of one 64 x 64 block, held in LDS (row stride kPv
// doubles).  On entry the lower part of sD is the block A (its upper part is
// never used) and sE is anything; on return the lower part of sD holds L and the
// upper part of sE L^{-T}.  The identity is stacked under A and takes the same
// column operations: A L^{-T} = L turns I into L^{-T}.
//
// Four panels of 16 columns.  Waves 0 and 1 factor a panel in registers, one
// row per lane: wave 0 the rows of A from the panel's diagonal down and, in the
// lanes above, the identity's rows that are no longer zero; wave 1 the
// identity's 16 rows of the panel.  Both keep the 16 diagonal rows in every
// 16-lane row as well, so that a column step y_c -= y_j a_cj is one
// v_fmac_f64_dpp per register, the a_cj broadcast inside the 16 lanes (lane
// reads into scalar registers cost three times the issue slots).  The columns
// are scaled by 1 / sqrt(pivot) before they are subtracted (unscaled, with
// 1 / pivot and the scale at the end, the inverse is off by 1.4 times as much).
// The next pivot a_j+1,j+1 - a_j+1,j^2 and its reciprocal
// root (hardware estimate and one third-order step) are formed ahead of the
// update, so that no step waits for it.  The other columns are updated with FP64
// MFMA: after panel p the 16 columns of panel p + 1 (one 16 x 16 tile per wave),
// the rest by waves 2 and 3 while waves 0 and 1 factor panel p + 1.
//
// Bound: the issue of wave 0 (64 column steps of about 160 cycles); 7.8 us per
// block from LDS to LDS.  The form before (the block over four waves, one LDS
// exchange and one barrier per column) took 26 us.
// ------------------------------------------------------------------------
constexpr int kHalf = 32;         // rows of a panel block solved beside the diagonal tile
constexpr int kPan = 16;
constexpr int kPv = kLdsPad;

// yc -= z_j[lane C of the 16-lane row] * y_j, zc likewise
template <int C>
__device__ __forceinline__ void fmac2_bcast(double &yc, double &zc, double zj, double yj) {
    asm("v_fmac_f64_dpp %0, %2, -%3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, -%2 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
        : "+v"(yc), "+v"(zc)
        : "v"(zj), "v"(yj), "n"(C));
}

// a and b of lane N of the 16-lane row (after two wait states, which a DPP
// read of a register that a vector instruction has just written needs)
template <int N>
__device__ __forceinline__ void bcast2(double a, double b, double &oa, double &ob) {
    asm("s_nop 1\n\t"
        "v_mov_b64_dpp %0, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b64_dpp %1, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
        : "=&v"(oa), "=&v"(ob)
        : "v"(a), "v"(b), "n"(N));
}

// Columns J + 2 .. 15 of column step J: the G-th of four parts of them, column
// J + 2 (the next step's pivot column) first.
template <int J, int G, int C = J + 2>
__device__ __forceinline__ void panel_group(double (&y)[kPan], double (&z)[kPan]) {
    if constexpr (C < kPan) {
        constexpr int rest = kPan - 3 - J;
        constexpr int g = C == J + 2 ? 0 : (C - J - 3) * 4 / rest;
        if constexpr (g == G) fmac2_bcast<C>(y[C], z[C], z[J], y[J]);
        panel_group<J, G, C + 1>(y, z);
    }
}

// Column steps J .. 15 of a panel: piv is pivot J (kept in s_piv, the same from
// every lane), rs its reciprocal root.  The scheduling fences keep the dependent
// steps of the next one apart, with the update's FMAs between them.
template <int J>
__device__ __forceinline__ void panel_steps(double (&y)[kPan], double (&z)[kPan], double piv, double rs, double *s_piv) {
    s_piv[J] = piv;
    y[J] *= rs;
    if constexpr (J + 1 < kPan) {
        z[J] *= rs;
        double zb, zd;
        bcast2<J + 1>(z[J], z[J + 1], zb, zd);
        const double next = fma(-zb, zb, zd);   // rounded as the update below rounds it
        const double q = __builtin_amdgcn_rsq(next);
        fmac2_bcast<J + 1>(y[J + 1], z[J + 1], z[J], y[J]);
        __builtin_amdgcn_sched_barrier(0);
        panel_group<J, 0>(y, z);
        __builtin_amdgcn_sched_barrier(0);
        const double t = next * q;
        __builtin_amdgcn_sched_barrier(0);
        panel_group<J, 1>(y, z);
        __builtin_amdgcn_sched_barrier(0);
        const double e = fma(-t, q, 1.0);
        __builtin_amdgcn_sched_barrier(0);
        panel_group<J, 2>(y, z);
        __builtin_amdgcn_sched_barrier(0);
        const double m = q * e, h = fma(0.375, e, 0.5);
        __builtin_amdgcn_sched_barrier(0);
        panel_group<J, 3>(y, z);
        __builtin_amdgcn_sched_barrier(0);
        panel_steps<J + 1>(y, z, next, fma(m, h, q), s_piv);
    }
}

// Tile (rb, cb) of 16 x 16 minus panel p's product, summed in halves: rows of A
// (rb > p) or of the identity (rb <= p; still zero at rb == p).
__device__ __forceinline__ void panel_tile(double *sD, double *sE, int p, int rb, int cb) {
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    double *S = rb <= p ? sE : sD;
    double old[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) old[v] = rb == p ? 0.0 : S[(kPan * rb + lk + 4 * v) * kPv + kPan * cb + lr];
    f64x4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int kk = 0; kk < kPan; kk += 4) {
        const int c = kPan * p + kk + lk;
        acc[kk / 8] = mfma_f64(S[(kPan * rb + lr) * kPv + c], sD[(kPan * cb + lr) * kPv + c], acc[kk / 8]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) S[(kPan * rb + lk + 4 * v) * kPv + kPan * cb + lr] = old[v] - (acc[0][v] + acc[1][v]);
}

// s_piv: 64 + 16 doubles.  Thread 0 gets the first column without a
// positive pivot (-1: none).  Wave 3 calls beside(p) at the start of panel p:
// rows 0 .. 16 p - 1 of the inverse are there by then.
template <typename Beside>
__device__ __forceinline__ int potrf64_lds(double *sD, double *sE, double *s_piv, const Beside &beside) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave index, held in a scalar register
    const int lr = lane & 15;
    constexpr int kPanels = kBlk / kPan;
#pragma unroll 1
    for (int p = 0; p < kPanels; ++p) {
        const int c0 = kPan * p;
        if (w < 2) {
            double *row = w == 1 ? sE + (c0 + lr) * kPv + c0 : (lane >= c0 ? sD : sE) + lane * kPv + c0;
            const double *dia = sD + (c0 + lr) * kPv + c0;
            double y[kPan], z[kPan];
#pragma unroll
            for (int q = 0; q < kPan; ++q) z[q] = dia[q];
#pragma unroll
            for (int q = 0; q < kPan; ++q) y[q] = w == 0 ? row[q] : (lr == q ? 1.0 : 0.0);
            __syncthreads();   // both waves have read the diagonal rows
            double piv, unused;
            bcast2<0>(z[0], z[0], piv, unused);
            const double q = __builtin_amdgcn_rsq(piv);
            const double e = fma(-(piv * q), q, 1.0);
            panel_steps<0>(y, z, piv, fma(q * e, fma(0.375, e, 0.5), q), w == 0 ? s_piv + c0 : s_piv + kBlk);
            if (w == 0 || lane < kPan) {
#pragma unroll
                for (int q = 0; q < kPan; ++q) row[q] = y[q];
            }
        } else {
            __syncthreads();
            if (w == 3) beside(p);
            // the columns beyond panel p, minus panel p - 1
            int idx = 0;
            if (p > 0)
                for (int cb = p + 1; cb < kPanels; ++cb)
                    for (int rb = 0; rb < kPanels; ++rb)
                        if ((rb < p || rb >= cb) && (idx++ & 1) == (w & 1)) panel_tile(sD, sE, p - 1, rb, cb);
        }
        __syncthreads();
        if (p + 1 < kPanels) {
            panel_tile(sD, sE, p, w, p + 1);
            __syncthreads();
        }
    }
    int bad = -1;
    if (w == 0) {
        const unsigned long long m = __ballot(!(s_piv[lane] > 0.0));
        if (m) bad = __ffsll((long long) m) - 1;
    }
    __syncthreads();
    return bad;
}

// ------------------------------------------------------------------------
// Tile column k in one launch: the Cholesky of its diagonal tile in 64 x 64
// blocks, the inverses of the diagonal blocks (winv_k), and the panel solve of
// `halves` blocks of 32 rows below it.
//
// Workgroups take a ticket each and run the task of that number; a task waits
// only for blocks of lower tickets, so the workgroups that run can always
// finish, however few of them the GPU holds.  Tasks, with L_rc the solved block
// (r, c) of the diagonal tile:
//   per block column c:  the diagonal task c (blocks (c, c - 1) and (c, c)),
//                        then the tasks (r, c), r >= c + 2 (one block each);
//   after them           the 32-row blocks below the tile, all block columns.
// A task adds up its blocks' products with the earlier block columns as those
// are published (flags in `sync`, one per block, zero at the launch).  The inverse
// comes in four panels of 16 rows while its block is still being factored (its
// words are their own flags, empty at the launch), and X = T W^T and D -= X X^T
// follow panel by panel, so that a diagonal task has only a quarter of both left
// when the last rows arrive.  What is handed over is stored and loaded past the
// L2s, without fences: a release or acquire fence of agent scope writes back or
// invalidates the L2 of its XCD, with everything the trailing update has there.
// Bound: the chain of diagonal tasks, 14.4 us per 64 columns alone (7.8 us of it
// the factorization, the rest the way of the last rows through memory, a quarter
// of two products and the exchange through LDS); with the whole inverse published
// at the end, between fences, 19 us.  Tile of 960 alone 284 -> 218 us, with 60
// row blocks below 372 -> 310 us, of 384 109 -> 86 us; 400 locations 225 -> 194
// us, 1,600 674 -> 568 us.  One launch per block column (each waiting anew for
// room beside the trailing update), a copy, and the panel solve after the whole
// tile took 36 us per 64 columns alone, 90 to 140 us beside the trailing update.
// ------------------------------------------------------------------------
namespace {

struct PanelSmem {
    double a[kBlk * kPv];   // operand columns: element (row, col) at col * kPv + row
    double b[kBlk * kPv];
    double piv[kBlk + kPan];
};
static_assert(sizeof(GemmSmem) <= sizeof(PanelSmem), "the row blocks stage through the same LDS");

// A flag says that the stores of a wave (store_shared) are complete.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void set_flag(int *flag) {
    __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits, wave by wave, until the flag is set.
__device__ __forceinline__ void wait_flag(const int *flag, int *lost) {
    Patience patience{lost};
    while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0 &&
           !patience.over())
        __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
}

// A published 64 x 64 block of a column-major matrix into LDS, in flight as 16
// loads per thread.
__device__ __forceinline__ void load_block(double (&v)[16], const double *src, int64_t ld) {
    const int row = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = load_shared(src + row + (int64_t) (w + 4 * q) * ld);
}
__device__ __forceinline__ void put_block(double *s, const double (&v)[16]) {
    const int row = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < 16; ++q) s[(w + 4 * q) * kPv + row] = v[q];
}

// acc -= A B^T for 64 x 64 operands in LDS, 32 columns at a time (see solve_block).
__device__ __forceinline__ void subtract_block(Acc64 &acc, const double *a, const double *b) {
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int half = 0; half < kBlk; half += kBlk / 2) {
        Acc64 p;
        acc_zero(p);
#pragma unroll 4
        for (int kk = half; kk < half + kBlk / 2; kk += 4) {
            const double *x = a + (kk + lk) * kPv + Acc64::row0() + lr, *y = b + (kk + lk) * kPv + Acc64::col0() + lr;
            const double a0 = x[0], a1 = x[16], b0 = y[0], b1 = y[16];
            p.v[0][0] = mfma_f64(b0, a0, p.v[0][0]);
            p.v[0][1] = mfma_f64(b0, a1, p.v[0][1]);
            p.v[1][0] = mfma_f64(b1, a0, p.v[1][0]);
            p.v[1][1] = mfma_f64(b1, a1, p.v[1][1]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc.v[i][j] -= p.v[i][j];
    }
}

// The accumulators hold the block C (column-major, ld).
__device__ __forceinline__ void acc_load(Acc64 &acc, const double *C, int64_t ld) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = (w & 1) * 32 + (lane & 15), c = (w >> 1) * 32 + (lane >> 4);
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc.v[ni][mi][v] = C[r + mi * 16 + (int64_t) (c + ni * 16 + 4 * v) * ld];
}

// The lower 16 x 16 tiles of a diagonal block, ten, dealt to the waves: tile w +
// 4 q of the rows' order (waves 2 and 3 carry the last one along as their third,
// of no effect: a branch around it cost as much).
struct DiagAcc {
    f64x4 v[3];
    static __device__ __forceinline__ int tile(int w, int q) { return 4 * min(w + 4 * q, 9); }
    static __device__ __forceinline__ int row(int w, int q) { return (int) (0x3333222110ull >> tile(w, q) & 15) * 16; }
    static __device__ __forceinline__ int col(int w, int q) { return (int) (0x3210210100ull >> tile(w, q) & 15) * 16; }

    // every element's value becomes f(row, col, value)
    template <typename F> __device__ __forceinline__ void foreach(int w, F f) {
        const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[q][e] = f(row(w, q) + lr, col(w, q) + lk + 4 * e, v[q][e]);
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int q = 0; q < 3; ++q) v[q] = f64x4{0.0, 0.0, 0.0, 0.0};
    }
    __device__ __forceinline__ void subtract(const DiagAcc &p) {
#pragma unroll
        for (int q = 0; q < 3; ++q) v[q] -= p.v[q];
    }
    // plus X X^T for K columns of X in LDS
    template <int K> __device__ __forceinline__ void add(int w, const double *x) {
        const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll 4
        for (int kk = 0; kk < K; kk += 4) {
            const double *xk = x + (kk + lk) * kPv + lr;
#pragma unroll
            for (int q = 0; q < 3; ++q) v[q] = mfma_f64(xk[col(w, q)], xk[row(w, q)], v[q]);
        }
    }
};

// Block (r, c) of the tile T (ld ts), r > c, solved in place: X = T W^T in panels
// of 16 columns, as the inverse's rows come.  Without kDia it is published; with
// it, dia -= L_rb L_rb^T for every b <= c, and the last panel stays in LDS
// (last_panel) for the caller to store and publish.  Products of 32 (for dia 64)
// columns are summed first and subtracted then.  Subtracted one MFMA after another,
// each rounds at the size of the block, and the error of the factor grows with the
// tile: nine fields of 1,600 in tiles of 64 to 960, against 80-bit factors of the
// same matrices, geometric mean of the rms errors of the log-determinant 6.1e-13 ->
// 3.7e-13 and of z' Sigma^-1 z (relative) 8.4e-16 -> 4.7e-16; it costs an evaluation
// of 1,600 1.5% (523 -> 531 us; 400 locations 183 -> 184).  Summed over all block columns
// first, the sums round at that size.
// kApplied: block columns before c - 1 are already subtracted from the block, and
// all before c from dia.
__device__ __forceinline__ double *last_panel(PanelSmem &sm) { return sm.b + 16 * kPv; }

// Columns 16 P .. 16 P + 15 of X, their product with themselves added to dia; W, t,
// out: this lane's element of each.
template <bool kDia, int P>
__device__ __forceinline__ void solve_panel(const double *W, const double *t, double *out, int ts, int w, PanelSmem &sm,
                                            DiagAcc &dia, int *lost) {
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    constexpr int kSteps = 4 * (P + 1);
    double wv[kSteps];
    Patience patience{lost};
    bool waiting;
    do {
#pragma unroll
        for (int q = 0; q < kSteps; ++q) wv[q] = load_shared(W + kPan * P + 4 * q * kBlk);
        waiting = false;
#pragma unroll
        for (int q = 0; q < kSteps; ++q) waiting |= is_pending(wv[q]);
        if (!kDia && __ballot(waiting) != 0) __builtin_amdgcn_s_sleep(4);   // off the chain: ask less often
    } while (__ballot(waiting) != 0 && !patience.over());
    f64x4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kSteps; ++q) x = mfma_f64(wv[q], t[4 * q * kPv], x);
    if (kDia) {
        double *s = sm.b + (P & 1) * kPan * kPv;
#pragma unroll
        for (int e = 0; e < 4; ++e) s[(lk + 4 * e) * kPv + 16 * w + lr] = x[e];
        __syncthreads();
        dia.add<kPan>(w, s);
    }
    if (!kDia || P < 3) {
#pragma unroll
        for (int e = 0; e < 4; ++e) store_shared(out + (int64_t) (kPan * P + 4 * e) * ts, x[e]);
    }
}

template <bool kDia, bool kApplied>
__device__ __forceinline__ void solve_block(double *T, int ts, int nsb, int r, int c, const double *winv_k, int *flags,
                                            PanelSmem &sm, DiagAcc &dia, int *lost) {
    double *X = T + r * kBlk + (int64_t) c * kBlk * ts;
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    DiagAcc part;
    {
        double va[16], vb[16];
        Acc64 acc;
        acc_load(acc, X, ts);
        for (int b = kApplied ? max(c - 1, 0) : 0; b < c; ++b) {
            wait_flag(flags + r * nsb + b, lost);
            load_block(va, T + r * kBlk + (int64_t) b * kBlk * ts, ts);
            wait_flag(flags + c * nsb + b, lost);
            load_block(vb, T + c * kBlk + (int64_t) b * kBlk * ts, ts);
            put_block(sm.a, va);
            put_block(sm.b, vb);
            __syncthreads();
            subtract_block(acc, sm.a, sm.b);
            if (kDia && !kApplied) {
                part.zero();
                part.add<kBlk>(w, sm.a);
                dia.subtract(part);
            }
            __syncthreads();
        }
        acc_foreach(acc, [&](int i, int j, double v) { sm.a[j * kPv + i] = v; });
        __syncthreads();
    }
    const double *W = winv_k + (int64_t) c * kBlk * kBlk + lr + lk * kBlk;
    const double *t = sm.a + lk * kPv + 16 * w + lr;
    double *out = X + 16 * w + lr + (int64_t) lk * ts;
    part.zero();
    solve_panel<kDia, 0>(W, t, out, ts, w, sm, part, lost);
    solve_panel<kDia, 1>(W, t, out, ts, w, sm, part, lost);
    solve_panel<kDia, 2>(W, t, out, ts, w, sm, part, lost);
    solve_panel<kDia, 3>(W, t, out, ts, w, sm, part, lost);
    if (kDia) dia.subtract(part);
    if (!kDia) {
        wait_stores();
        __syncthreads();
        if (threadIdx.x == 0) set_flag(flags + r * nsb + c);
    }
}

// Rows 16 p .. 16 p + 15 of the inverse, columns lk + 4 q for q in [q0, q1), from
// L^{-T} in LDS.
__device__ __forceinline__ void store_inverse_rows(double *W, const PanelSmem &sm, int p, int q0, int q1) {
    const int i = kPan * p + (threadIdx.x & 15), lk = (threadIdx.x & 63) >> 4;
#pragma unroll 4
    for (int q = q0; q < q1; ++q) {
        const int j = lk + 4 * q;
        store_word(W + i + j * kBlk, i >= j ? sm.b[j * kPv + i] : 0.0);
    }
}

// What wave 3 hands out while a diagonal block is factored: the last panel of the
// block left of it, then the inverse's rows, a panel behind.  It waits for none
// of its stores where the factorization would wait for it.
struct HandOut {
    double *W, *X;   // X null for the first block
    int ts;
    PanelSmem &sm;
    int *x_flag;
    __device__ __forceinline__ void operator()(int p) const {
        const int lane = threadIdx.x & 63;
        if (p == 0 && X) {
            const double *s = last_panel(sm) + lane;
#pragma unroll
            for (int q = 0; q < 16; ++q) store_shared(X + lane + (int64_t) (48 + q) * ts, s[q * kPv]);
        }
        if (p == 1 && X) {
            wait_stores();
            if (lane == 0) set_flag(x_flag);
        }
        if (p > 0) store_inverse_rows(W, sm, p - 1, 0, 16);
    }
};

// Diagonal task r: block (r, r - 1), then block (r, r) factored and inverted.
template <bool kApplied>
__device__ __forceinline__ void diagonal_task(double *T, int ts, int nsb, int r, double *winv_k, int *flags, int *info,
                                              int64_t col0, int64_t n, PanelSmem &sm) {
    double *D = T + r * kBlk + (int64_t) r * kBlk * ts;
    double *W = winv_k + (int64_t) r * kBlk * kBlk;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    DiagAcc dia;
    dia.foreach(w, [&](int i, int j, double) { return D[i + (int64_t) j * ts]; });
    if (r > 0) {
        solve_block<true, kApplied>(T, ts, nsb, r, r - 1, winv_k, flags, sm, dia, info + 1);
        wait_stores();   // the panels before the last: long done
    }
    dia.foreach(w, [&](int i, int j, double v) { return sm.a[i * kPv + j] = v; });
    __syncthreads();
    const HandOut beside{W, r > 0 ? D - (int64_t) kBlk * ts : nullptr, ts, sm, flags + r * nsb + r - 1};
    const int bad = potrf64_lds(sm.a, sm.b, sm.piv, beside);
    store_inverse_rows(W, sm, kBlk / kPan - 1, 4 * w, 4 * w + 4);
    wait_stores();
    __syncthreads();
    if (threadIdx.x == 0) {
        set_flag(flags + r * nsb + r);
        if (bad >= 0 && col0 + r * kBlk + bad < n) atomicCAS(info, 0, (int) (col0 + r * kBlk + bad + 1));
    }
    const int i = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int j = w + 4 * q;
        D[i + (int64_t) j * ts] = i >= j ? sm.a[i * kPv + j] : 0.0;
    }
}

// What a row block below the tile waits for (the diagonal task of block column
// j has itself waited for the row's earlier blocks).
struct BlockWait {
    static constexpr bool kAhead = false;
    const int *flags;
    int nsb;
    int *lost;
    __device__ __forceinline__ void row(int j) const { wait_flag(flags + j * nsb + j - 1, lost); }
    __device__ __forceinline__ void inverse(int j) const { wait_flag(flags + j * nsb + j, lost); }
};

// Tasks of a diagonal tile of so many 64 x 64 blocks.
__host__ __device__ inline int tile_tasks(int blocks) { return blocks + (blocks - 1) * (blocks - 2) / 2; }

}  // namespace

// Task idx of block column c of diagonal tile k: 0 the diagonal task, then the
// blocks (c + 1 + idx, c).
template <bool kApplied>
__device__ __forceinline__ void block_column_task(const TileMap &map, int k, double *winv_k, int *sync, int *info,
                                                  int64_t n, int c, int idx, PanelSmem &sm) {
    const int nsb = map.ts / kBlk;
    double *T = tile_f64(map, k, k);
    if (idx == 0) {
        diagonal_task<kApplied>(T, map.ts, nsb, c, winv_k, sync + 1, info, (int64_t) k * map.ts, n, sm);
    } else {
        DiagAcc none;
        solve_block<false, kApplied>(T, map.ts, nsb, c + 1 + idx, c, winv_k, sync + 1, sm, none, info + 1);
    }
}

// One task of tile column k; sync: the column's ticket (unused here) and flags.
__device__ __forceinline__ void tile_column_task(const TileMap &map, int k, double *winv_k, int *sync, int *info,
                                                 int64_t n, int halves, int task, PanelSmem &sm) {
    const int ts = map.ts;
    const int nsb = ts / kBlk;
    const int live = map.blocks(k);
    if (task >= tile_tasks(live)) {
        const int h = task - tile_tasks(live);
        if (h >= halves) return;
        const int per = ts / kHalf;
        double *X = tile_f64(map, k + 1 + h / per, k) + (h % per) * kHalf;
        solve_rows<double, kHalf>(tile_f64(map, k, k), ts, nsb, X, winv_k, *reinterpret_cast<GemmSmem *>(&sm),
                                  BlockWait{sync + 1, nsb, info + 1});
        return;
    }
    // block column c holds the diagonal task and live - 2 - c others
    int c = 0, idx = task;
    while (idx > max(0, live - 2 - c)) {
        idx -= 1 + max(0, live - 2 - c);
        ++c;
    }
    block_column_task<false>(map, k, winv_k, sync, info, n, c, idx, sm);
}

__device__ __forceinline__ int take_ticket(int *counter) {
    __shared__ int s_ticket;
    if (threadIdx.x == 0) s_ticket = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return s_ticket;
}

__global__ void __launch_bounds__(kThreads) tile_column_kernel(TileMap map, int k, double *winv_k, int *sync, int *info,
                                                               int64_t n, int halves) {
    __shared__ PanelSmem sm;
    tile_column_task(map, k, winv_k, sync, info, n, halves, take_ticket(sync), sm);
}

// A larger diagonal tile (kOneLaunchTile), in three launches per block column
// whose workgroups wait for earlier launches only (the flags and words they look
// for are there): the diagonal task, the blocks below it, and their products off
// the blocks (r, s), r >= s >= c + 2.  (Column c + 1's blocks are left to their
// tasks: block (c + 1, c) comes with the next diagonal task.)
enum BlockColumnPart { kDiagonalPart, kBelowPart, kUpdatePart };

__device__ __forceinline__ void block_column_part(const TileMap &map, int k, double *winv_k, int *sync, int *info,
                                                  int64_t n, int c, BlockColumnPart part, int at, PanelSmem &sm) {
    const int live = map.blocks(k), ts = map.ts;
    if (part == kDiagonalPart) {
        if (c < live) block_column_task<true>(map, k, winv_k, sync, info, n, c, 0, sm);
        return;
    }
    if (part == kBelowPart) {
        if (c + 2 + at < live) block_column_task<true>(map, k, winv_k, sync, info, n, c, 1 + at, sm);
        return;
    }
    int i = 0;   // row of `at` in the lower triangle
    while (at > i) at -= ++i;
    const int r = c + 2 + i, q = c + 2 + at;
    if (r >= live) return;
    double *T = tile_f64(map, k, k);
    double *C = T + r * kBlk + (int64_t) q * kBlk * ts;
    double va[16], vb[16];
    Acc64 acc;
    acc_load(acc, C, ts);
    load_block(va, T + r * kBlk + (int64_t) c * kBlk * ts, ts);
    load_block(vb, T + q * kBlk + (int64_t) c * kBlk * ts, ts);
    put_block(sm.a, va);
    put_block(sm.b, vb);
    __syncthreads();
    subtract_block(acc, sm.a, sm.b);
    acc_foreach(acc, [&](int row, int col, double v) { C[row + (int64_t) col * ts] = v; });
}

template <BlockColumnPart kPart>
__global__ void __launch_bounds__(kThreads) block_column_kernel(TileMap map, int k, double *winv_k, int *sync, int *info,
                                                                int64_t n, int c) {
    __shared__ PanelSmem sm;
    block_column_part(map, k, winv_k, sync, info, n, c, kPart, blockIdx.x, sm);
}

// ------------------------------------------------------------------------
// Batched forms: one launch applies the same step to several problems of the
// same tile size, problem b described by jobs[b] (blockIdx.y, or blockIdx.z
// for the update); workgroups beyond a problem's extent exit at once.
// ------------------------------------------------------------------------
// Tickets interleave the problems: task t / njobs of problem t % njobs.
__global__ void __launch_bounds__(kThreads) tile_column_batch_kernel(const BatchJob *jobs, int njobs, int with_rows) {
    __shared__ PanelSmem sm;
    const int t = take_ticket(jobs[0].sync);
    const BatchJob J = scalar_load(jobs + t % njobs);
    const int below = J.map.blocks() - (J.k + 1) * (J.map.ts / kBlk);   // none at or below the last tile
    const int halves = with_rows ? 2 * max(below, 0) : 0;
    tile_column_task(J.map, J.k, J.winv_k, J.sync, J.info, J.n, halves, t / njobs, sm);
}

template <BlockColumnPart kPart>
__global__ void __launch_bounds__(kThreads) block_column_batch_kernel(const BatchJob *jobs, int c) {
    __shared__ PanelSmem sm;
    const BatchJob J = scalar_load(jobs + blockIdx.y);
    block_column_part(J.map, J.k, J.winv_k, J.sync, J.info, J.n, c, kPart, blockIdx.x, sm);
}

template <int kRows>
__global__ void __launch_bounds__(kThreads) trsm_rows_batch_kernel(const BatchJob *jobs) {
    const BatchJob J = scalar_load(jobs + blockIdx.y);
    const int per = J.map.ts / kRows;
    if ((int) blockIdx.x * kRows >= (J.map.blocks() - (J.k + 1) * (J.map.ts / kBlk)) * kBlk) return;
    __shared__ GemmSmem sm;
    solve_row_block<double, kRows, double>(J.map, J.k, (int64_t) (J.k + 1) * per + blockIdx.x, J.winv_k, sm);
}

__global__ void __launch_bounds__(kThreads) update_batch_kernel(const BatchJob *jobs) {
    const BatchJob J = scalar_load(jobs + blockIdx.z);
    const int rest = J.map.nt - J.k - 1;   // tile columns k+1 .. nt-1: the first rest (rest + 1) / 2 pairs
    if ((int) blockIdx.y >= rest * (rest + 1) / 2) return;
    update_body<kBlk>(J.map, nullptr, J.pairs, J.k, blockIdx.x, blockIdx.y, 1);
}

// Panels of at most this many 64-row blocks are solved by the launch that
// factors the diagonal tile; a longer one by its own launch after it (its
// workgroups would hold the GPU's slots while they wait for the diagonal tile,
// and 64-row blocks load L_kk half as often per flop).
constexpr int kFusedRows = 128;

// Tiles up to this size are factored by one launch per tile column, whose
// workgroups wait for each other.  Larger ones take three launches per block
// column, without such waits: one call with tiles of 2,048 (or of 64: the record
// does not say which of two) has not returned, for a reason that is not known, and
// up to here that launch has run often.  1,500 locations in tiles of 1,216 1.5 ms,
// 4,000 in tiles of 1,984 5.4 ms, eight of 1,500 in a batch 1.5 ms; in two launches
// per block column, each block adding up its products in turn, 2.6, 12.2 and 3.3.
constexpr int kOneLaunchTile = 1152;

void launch_step_batch(const BatchJob *jobs, int njobs, int ts, int rest, int nrest, hipStream_t s) {
    if (njobs <= 0) return;
    const int nsb = ts / kBlk;
    const bool one_launch = ts <= kOneLaunchTile;
    const bool fused = one_launch && rest * nsb * nrest <= kFusedRows;
    if (one_launch) {
        const int tasks = tile_tasks(nsb) + (fused ? rest * (ts / kHalf) : 0);
        hipLaunchKernelGGL(tile_column_batch_kernel, dim3((unsigned) (tasks * njobs)), dim3(kThreads), 0, s, jobs, njobs,
                           fused ? 1 : 0);
    }
    for (int c = 0; c < nsb && !one_launch; ++c) {
        const int below = std::max(nsb - 2 - c, 0);
        const unsigned count = (unsigned) njobs;
        hipLaunchKernelGGL(block_column_batch_kernel<kDiagonalPart>, dim3(1, count), dim3(kThreads), 0, s, jobs, c);
        if (below == 0) continue;
        hipLaunchKernelGGL(block_column_batch_kernel<kBelowPart>, dim3((unsigned) below, count), dim3(kThreads), 0, s, jobs, c);
        hipLaunchKernelGGL(block_column_batch_kernel<kUpdatePart>, dim3((unsigned) (below * (below + 1) / 2), count),
                           dim3(kThreads), 0, s, jobs, c);
    }
    if (rest <= 0 || nrest <= 0) return;
    if (!fused) {
        const int half = rest * nsb * nrest < kHalfRowsBelow;
        hipLaunchKernelGGL(half ? trsm_rows_batch_kernel<32> : trsm_rows_batch_kernel<64>,
                           dim3((unsigned) ((rest * nsb) << half), nrest), dim3(kThreads), 0, s, jobs);
    }
    hipLaunchKernelGGL(update_batch_kernel, dim3((unsigned) (nsb * nsb), (unsigned) (rest * (rest + 1) / 2), nrest),
                       dim3(kThreads), 0, s, jobs);
}

int tile_column_sync_ints(int ts) { return 1 + (ts / kBlk) * (ts / kBlk); }

bool tile_column_solves_rows(int ts, int blocks) { return ts <= kOneLaunchTile && blocks <= kFusedRows; }

void launch_tile_column(const TileMap &map, int k, double *winv_k, int *sync, int *info, int64_t n, int blocks,
                        hipStream_t s) {
    const int live = map.blocks(k);
    for (int c = 0; c < live && map.ts > kOneLaunchTile; ++c) {
        const int below = std::max(live - 2 - c, 0);
        hipLaunchKernelGGL(block_column_kernel<kDiagonalPart>, dim3(1), dim3(kThreads), 0, s, map, k, winv_k, sync, info, n, c);
        if (below == 0) continue;
        hipLaunchKernelGGL(block_column_kernel<kBelowPart>, dim3((unsigned) below), dim3(kThreads), 0, s, map, k, winv_k, sync,
                           info, n, c);
        hipLaunchKernelGGL(block_column_kernel<kUpdatePart>, dim3((unsigned) (below * (below + 1) / 2)), dim3(kThreads), 0, s,
                           map, k, winv_k, sync, info, n, c);
    }
    if (map.ts > kOneLaunchTile) return;
    hipLaunchKernelGGL(tile_column_kernel, dim3((unsigned) (tile_tasks(map.blocks(k)) + 2 * blocks)), dim3(kThreads), 0,
                       s, map, k, winv_k, sync, info, n, 2 * blocks);
}

}  // namespace egs
