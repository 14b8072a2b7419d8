// Triangular solves, log-determinant / quadratic-form partials, kriging product
// and the synthetic-data helpers on gfx950.
//
// The forward solve replaces CHAMELEON_dtrsm_Tile(Left, Lower, NoTrans) on Z
// (ChameleonImplementation.cpp:216-217, 337-347) and fuses the reductions the
// reference runs per tile as dmdet (dmdet-codelet.cpp:70-80) and ddotp
// (ddotp-codelet.cpp:62-72) tasks: the workgroup that solves a block b of 64 rows
// also writes sum(log L_ii) over L_ii > 0 and y_b . y_b of that block.  The host
// sums the blocks' partials in order, so results do not depend on scheduling.  All
// reductions inside a workgroup use a fixed order.
#include <algorithm>

#include "egs_common.hpp"
#include "egs_kernels.hpp"
#include "egs_matern.hpp"

namespace egs {

constexpr int kMaxTs = 2048;

// Fixed-order sum of one value per thread over the workgroup.
__device__ double wg_sum(double v, double *red) {
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if (t < s) red[t] += red[t + s];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

// ------------------------------------------------------------------------
// Triangular solves with the tiled factor, one launch each.  A workgroup owns
// one 64-row block of the solution; it walks the blocks of L of its row (of its
// column, backward) in the order in which their solution blocks appear, and the
// last one, the inverse of the diagonal block (winv) and the publication of the
// result are the chain from block to block.  Workgroups take tickets, and a
// ticket waits only for lower ones, so those that run can always go on.
//
// Bounded by that chain for a few hundred blocks (one hop through memory, two
// 64 x 64 products spread over four waves and two exchanges through LDS) and by
// reading L once above.  The loads of two blocks of L are in flight per
// wave and do not wait for the solution; the solution itself is its own flag (a
// word that holds ~0 has not been published), which saves a hop one flag load
// and one fence.  20,000 locations, tiles of 960 (1.6 GB of L):
// 0.57 ms forward and 0.58 backward; with one workgroup solving the diagonal
// tile and a launch per panel, 2.8 and 7.8 ms.
// ------------------------------------------------------------------------
// v, loaded from p earlier, once every lane's word is published.  far: other blocks
// come before this one is waited for; it asks less often, so that the words of
// the chain's next block are not queued behind everybody's requests.
__device__ __forceinline__ double await(const double *p, double v, bool far, int *lost) {
    auto pending = [&] { return __ballot(is_pending(v)) != 0; };
    if (pending()) {   // apart from the loop, whose wait for its own load would also be one for all in flight
        Patience patience{lost};
        do {
            if (far) __builtin_amdgcn_s_sleep(16);
            v = load_shared(p);
        } while (pending() && !patience.over());
    }
    return v;
}

// sum_q m[q] * x[lane q of the 16-lane row], in two interleaved sums (the two wait
// states are what a DPP read of a just written register needs).
__device__ __forceinline__ double row_product(const double (&m)[16], double x) {
    double a = 0.0, b = 0.0;
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %2, %3 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %4 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %5 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %6 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %7 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %8 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %9 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %10 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %11 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %12 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %13 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %14 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %15 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %16 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %2, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %18 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "+&v"(a), "+&v"(b)
        : "v"(x), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]), "v"(m[7]), "v"(m[8]),
          "v"(m[9]), "v"(m[10]), "v"(m[11]), "v"(m[12]), "v"(m[13]), "v"(m[14]), "v"(m[15]));
    return a + b;
}

// A sum of many terms, in groups of 16: the terms of a group round at its size, only
// the groups at that of the whole.  With every product added to the running sum, the
// residual of a forward solve grew with the square root of the rows: 5,700 locations
// 1.04e-15 rms, 11,500 1.38e-15; so 1.8e-16 and 2.0e-16, for 0 to 1% of the solve.
struct GroupedSum {
    double sum, part = 0.0;
    __device__ __forceinline__ void add(double v, int m) {   // the m-th
        const bool last = (m & 15) == 15;
        part += v;
        sum += last ? part : 0.0;
        part = last ? 0.0 : part;
    }
    __device__ __forceinline__ double total() const { return sum + part; }
};

// A lane's 16 elements of a block of L in flight, with the word of the solution
// they multiply: a row's, ts apart, or (kAcross) a column's, one after the other.
// kMixed: of an FP32 tile the aligned 8 bytes around an element are loaded, so
// that one sequence of loads, with none waiting, serves both kinds of tiles.
template <bool kMixed, bool kAcross = false> struct Cols {
    double v[16], y;
    bool f32;

    __device__ __forceinline__ void load(const TileMap &map, int i, int j, int row, int col) {
        const int e = i * map.nt + j;
        if constexpr (kMixed)
            f32 = (scalar_load(reinterpret_cast<const unsigned *>(map.store) + e / 4) >> 8 * (e % 4) & 255u) == kStoreF32;
        const int size = kMixed && f32 ? 4 : 8;
        const char *A = map.base + scalar_load(map.off + e);
        const int64_t at = row + (int64_t) col * map.ts;
#pragma unroll
        for (int q = 0; q < 16; ++q)
            v[q] = *reinterpret_cast<const double *>(A + ((at + (kAcross ? q : q * (int64_t) map.ts)) * size & ~int64_t(7)));
        asm volatile("" ::: "memory");   // the loads stay here, and are made again for the same block
    }
    // the elements in FP64 (row: the row of the first of them; ts is even)
    __device__ __forceinline__ void widen(int row) {
        if (kMixed && f32) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const unsigned long long bits = __builtin_bit_cast(unsigned long long, v[q]);
                const bool high = (kAcross ? row + q : row) & 1;
                v[q] = (double) __builtin_bit_cast(float, (unsigned) (high ? bits >> 32 : bits));
            }
        }
    }
};

// use(c, 0 .. count - 1) in order, each after a fetch(c), two of which are in
// flight.  The loop has one path, on which the compiler can count them: there
// is no branch around a fetch (up to two past the last are made and dropped),
// and the odd step comes first.
template <typename C, typename Fetch, typename Use>
__device__ __forceinline__ void two_in_flight(int count, Fetch fetch, Use use) {
    int m = 0;
    if (count & 1) {
        C a;
        fetch(a);
        use(a, m++);
    }
    if (m >= count) return;
    C a, b;
    fetch(a);
    fetch(b);
#pragma unroll 1
    do {
        use(a, m);
        fetch(a);
        use(b, m + 1);
        fetch(b);
        m += 2;
    } while (m < count);
}

struct SolveSmem {
    double part[2][4][kBlk];
    double base[kBlk];
    int ticket;
};

__device__ __forceinline__ int solve_ticket(double *pending, int64_t npad, SolveSmem &sm) {
    if (threadIdx.x == 0)   // the word starts as all ones
        sm.ticket = 1 + __hip_atomic_fetch_add(reinterpret_cast<int *>(pending + npad), 1, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sm.ticket);
}

// The end of a block: x (wave w's share of the right-hand side), then the product
// with the diagonal block's inverse (m: this wave's 16 columns of it, or of its
// transpose).  The solution is valid in wave 0.
__device__ __forceinline__ double finish_block(double x, const double (&m)[16], int w, int lane, SolveSmem &sm) {
    sm.part[0][w][lane] = x;
    __syncthreads();
    const int c = 16 * w + (lane & 15);
    const double t = ((sm.part[0][0][c] + sm.part[0][1][c]) + sm.part[0][2][c]) + sm.part[0][3][c];
    sm.part[1][w][lane] = row_product(m, t);
    __syncthreads();
    return ((sm.part[1][0][lane] + sm.part[1][1][lane]) + sm.part[1][2][lane]) + sm.part[1][3][lane];
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Block b of L y = z, y in z's place and in pending; partials (may be null):
// [2b] = sum log L_ii over L_ii > 0, [2b+1] = y_b . y_b.
template <bool kMixed>
__device__ __forceinline__ void forward_block(const TileMap &map, const double *winv, double *z, double *pending,
                                              double *partials, int b, SolveSmem &sm, int *lost) {
    const int ts = map.ts, nsb = ts / kBlk;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const int ti = b / nsb, rb = b % nsb;
    const double *yw = pending + 16 * w + (lane & 15);
    double m[16];
    const double *W = winv + (int64_t) b * kBlk * kBlk + lane + 16 * w * kBlk;
#pragma unroll
    for (int q = 0; q < 16; ++q) m[q] = W[q * kBlk];
    double d = 1.0;
    if (partials && w == 3) d = tile_f64(map, ti, ti)[(int64_t) (rb * kBlk + lane) * (ts + 1)];
    GroupedSum acc{w == 0 ? z[(int64_t) b * kBlk + lane] : 0.0};
    int next = 0, tj = 0, cb = 0;   // the next fetch's block, its tile column and block column there
    auto fetch = [&](Cols<kMixed> &c) {
        c.load(map, ti, tj, rb * kBlk + lane, cb * kBlk + 16 * w);
        c.y = load_shared(yw + (int64_t) next * kBlk);
        if (next < b - 1) {   // the last block is fetched again (two_in_flight)
            ++next;
            if (++cb == nsb) cb = 0, ++tj;
        }
    };
    auto use = [&](Cols<kMixed> &c, int j) {
        const double y = await(yw + (int64_t) j * kBlk, c.y, b - j > 2, lost);
        c.widen(lane);
        acc.add(row_product(c.v, -y), j);
    };
    two_in_flight<Cols<kMixed>>(b, fetch, use);
    const double y = finish_block(acc.total(), m, w, lane, sm);
    if (w == 0) {
        store_word(pending + (int64_t) b * kBlk + lane, y);
        z[(int64_t) b * kBlk + lane] = y;
        if (partials) {
            const double q = wave_sum(y * y);
            if (lane == 0) partials[2 * b + 1] = q;
        }
    } else if (partials && w == 3) {
        const double ld = wave_sum(d > 0.0 ? log(d) : 0.0);
        if (lane == 0) partials[2 * b] = ld;
    }
}

template <bool kMixed>
__global__ void __launch_bounds__(kThreads) forward_kernel(TileMap map, const double *winv, double *z, double *pending,
                                                           double *partials, int *info) {
    __shared__ SolveSmem sm;
    const int b = solve_ticket(pending, (int64_t) map.nt * map.ts, sm);
    forward_block<kMixed>(map, winv, z, pending, partials, b, sm, info + 1);
}

// The jobs' blocks in turn, so that a ticket's chain is in lower tickets.
__global__ void __launch_bounds__(kThreads) forward_batch_kernel(const BatchJob *jobs, int njobs) {
    __shared__ SolveSmem sm;
    const int t = solve_ticket(jobs[0].pending, (int64_t) jobs[0].map.nt * jobs[0].map.ts, sm);
    const BatchJob J = scalar_load(jobs + t % njobs);
    const int b = t / njobs;
    if (b >= J.map.blocks()) return;
    forward_block<false>(J.map, J.winv_k, J.z, J.pending, J.partials, b, sm, J.info + 1);
}

// Block b of L^T y = z, y in z's place and in pending.  Down the block's column
// lanes hold rows (coalesced), so the 16 column sums of a wave stay spread over
// its lanes and are added up before the last two blocks, which are read
// transposed: nothing but a block's product waits for the block solved just
// before (with the sums added up between the last two, 0.9 us more per block).
template <bool kMixed>
__device__ __forceinline__ void backward_block(const TileMap &map, const double *winv, double *z, double *pending, int b,
                                               SolveSmem &sm, int *lost) {
    const int ts = map.ts, nsb = ts / kBlk, nb = map.blocks();
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const int tj = b / nsb, cb = b % nsb;
    // the last two blocks are read transposed
    const int last = b + 2;
    Cols<kMixed, true> T[2];
    const double *y_last[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = min(last - u, nb - 1);
        T[u].load(map, i / nsb, tj, (i % nsb) * kBlk + 16 * w, cb * kBlk + lane);
        y_last[u] = pending + (int64_t) i * kBlk + 16 * w + (lane & 15);
    }
    double m[16];
    const double *W = winv + (int64_t) b * kBlk * kBlk + lane * kBlk + 16 * w;
#pragma unroll
    for (int q = 0; q < 16; ++q) m[q] = W[q];
    const double zb = w == 0 ? z[(int64_t) b * kBlk + lane] : 0.0;
    double acc[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.0;
    int next = nb - 1, ti = map.nt - 1, rb = map.last_blocks - 1;   // the next fetch's block and its place
    auto fetch = [&](Cols<kMixed> &c) {
        c.load(map, ti, tj, rb * kBlk + lane, cb * kBlk + 16 * w);
        c.y = load_shared(pending + (int64_t) next * kBlk + lane);
        if (next > last + 1) {
            --next;
            if (--rb < 0) rb = nsb - 1, --ti;
        }
    };
    auto use = [&](Cols<kMixed> &c, int m) {
        const double y = -await(pending + (int64_t) (nb - 1 - m) * kBlk + lane, c.y, nb - 1 - m - b > 3, lost);
        c.widen(lane);
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[q] = fma(c.v[q], y, acc[q]);
    };
    two_in_flight<Cols<kMixed>>(max(nb - 1 - last, 0), fetch, use);   // none for the last three blocks
    if (last < nb) T[0].y = load_shared(y_last[0]);
    if (last - 1 < nb) T[1].y = load_shared(y_last[1]);
    // the sums over the 64 lanes: each step halves the columns a lane keeps
#pragma unroll
    for (int half = 8, bit = 32; half > 0; half >>= 1, bit >>= 1) {
        const bool up = lane & bit;
#pragma unroll
        for (int q = 0; q < half; ++q) {
            const double keep = up ? acc[q + half] : acc[q], give = up ? acc[q] : acc[q + half];
            acc[q] = keep + __shfl_xor(give, bit, 64);
        }
    }
    acc[0] += __shfl_xor(acc[0], 2, 64);
    acc[0] += __shfl_xor(acc[0], 1, 64);
    if ((lane & 3) == 0) sm.base[16 * w + (lane >> 2)] = acc[0];
    __syncthreads();
    double x = w == 0 ? zb + sm.base[lane] : 0.0;
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (last - u < nb) {
            T[u].widen(0);
            x += row_product(T[u].v, -await(y_last[u], T[u].y, false, lost));
        }
    const double y = finish_block(x, m, w, lane, sm);
    if (w == 0) {
        store_word(pending + (int64_t) b * kBlk + lane, y);
        z[(int64_t) b * kBlk + lane] = y;
    }
}

template <bool kMixed>
__global__ void __launch_bounds__(kThreads) backward_kernel(TileMap map, const double *winv, double *z, double *pending,
                                                            int *info) {
    __shared__ SolveSmem sm;
    const int t = solve_ticket(pending, (int64_t) map.nt * map.ts, sm);
    backward_block<kMixed>(map, winv, z, pending, map.blocks() - 1 - t, sm, info + 1);
}

// out = L e: one workgroup of 16 waves per 64 rows, the longest rows first; the
// waves deal out the 16-column strips, two in flight each.  Bounded by the
// bytes of L a CU can have in flight: 6,001 locations 53 us, with four waves
// and one load at a time 515 us.
constexpr int kTrmvThreads = 1024;

__global__ void __launch_bounds__(kTrmvThreads) trmv_kernel(TileMap map, const double *e, double *out) {
    constexpr int kWaves = kTrmvThreads / 64;
    __shared__ double sp[kWaves][kBlk];
    const int ts = map.ts, nsb = ts / kBlk;
    const int b = gridDim.x - 1 - blockIdx.x;
    const int i = b / nsb, rb = b % nsb;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const int strips = 4 * (b + 1), per_tile = 4 * nsb;
    int next = w;
    auto fetch = [&](Cols<false> &c) {
        const int k = next / per_tile, c0 = 16 * (next % per_tile);
        c.y = e[16 * (int64_t) next + (lane & 15)];
        c.load(map, i, k, rb * kBlk + lane, c0);
        if (next + kWaves < strips) next += kWaves;
    };
    GroupedSum acc{0.0};
    auto use = [&](Cols<false> &c, int m) {
        const int s = w + m * kWaves;
        if (s >= 4 * b) {   // the diagonal block
#pragma unroll
            for (int q = 0; q < 16; ++q) c.v[q] = 16 * (s - 4 * b) + q <= lane ? c.v[q] : 0.0;
        }
        acc.add(row_product(c.v, c.y), m);
    };
    two_in_flight<Cols<false>>((strips - w + kWaves - 1) / kWaves, fetch, use);
    sp[w][lane] = acc.total();
    __syncthreads();
    if (w == 0) {
        double a = 0.0;
        for (int q = 0; q < kWaves; ++q) a += sp[q][lane];
        out[(int64_t) b * kBlk + lane] = a;
    }
}

// Kriging mean: out[r] = sum_c Sigma(l1_r, l2_c) x[c], one workgroup per row;
// the tables of the row's orders (see matern_table_eval) are staged in LDS.
struct CovGemvArgs {
    double *out;
    int64_t rows, cols;
    MaternParams prm;
    Locs l1, l2;
    const double *x;
    const double *tabs;
    const double *word;   // copied to out[-1]
    int three_d;
};

template <int kTabs, bool kSphere>
__global__ void __launch_bounds__(kThreads, kTabs < 2 ? 4 : 4 - kTabs) cov_gemv_kernel(CovGemvArgs a) {
    __shared__ double red[kThreads];
    __shared__ __align__(16) double s_tab[kTabs > 0 ? kTabs * kTabDoubles : 1];
    for (int e = threadIdx.x; e < kTabs * kTabDoubles; e += kThreads) s_tab[e] = a.tabs[e];
    __syncthreads();
    const int64_t r = blockIdx.x;
    const bool three_d = a.three_d != 0;
    const int shift = a.prm.kernel == 1 ? 1 : 0;
    const int64_t i = r >> shift;
    const StagedLoc row = stage_location<kSphere>(a.l1.x[i], a.l1.y[i], three_d ? a.l1.z[i] : 0.0);
    double s = 0.0;
#pragma unroll 1
    for (int64_t c = threadIdx.x; c < a.cols; c += kThreads) {
        const int64_t j = c >> shift;
        const StagedLoc col = stage_location<kSphere>(a.l2.x[j], a.l2.y[j], three_d ? a.l2.z[j] : 0.0);
        const int pair = shift ? (int) ((r & 1) * 2 + (c & 1)) : 0;
        s += staged_covariance<(kTabs > 0), kSphere>(a.prm, pair, staged_separation<kSphere>(row, col, three_d), s_tab) * a.x[c];
    }
    s = wg_sum(s, red);
    if (threadIdx.x == 0) a.out[r] = s;
    if (r == 0 && threadIdx.x == 0) a.out[-1] = *a.word;
}

// dlarnv(idist = 3): value m uses the uniforms number 2m and 2m+1 of the
// stream u_j = (s0 * A^(j+1) mod 2^48) / 2^48 with A = 33952834046453.
__device__ __forceinline__ uint64_t lcg_pow(uint64_t e) {
    const uint64_t mask = (1ull << 48) - 1;
    uint64_t base = 33952834046453ull, r = 1;
    while (e) {
        if (e & 1) r = (r * base) & mask;
        base = (base * base) & mask;
        e >>= 1;
    }
    return r;
}

__global__ void __launch_bounds__(kThreads) dlarnv_normal_kernel(double *e, int64_t n, uint64_t seed48) {
    const int64_t m = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    if (m >= n) return;
    const uint64_t mask = (1ull << 48) - 1;
    const uint64_t s1 = (seed48 * lcg_pow((uint64_t) (2 * m + 1))) & mask;
    const uint64_t s2 = (s1 * 33952834046453ull) & mask;
    const double u1 = (double) s1 * 0x1p-48;
    const double u2 = (double) s2 * 0x1p-48;
    e[m] = sqrt(-2.0 * log(u1)) * cos(6.2831853071795864769252867663 * u2);
}

__global__ void __launch_bounds__(kThreads) copy_pad_kernel(double *dst, const double *src, int64_t n, int64_t npad) {
    const int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    if (i < npad) dst[i] = (i < n) ? src[i] : 0.0;
}

__device__ __forceinline__ void init_element(const InitJob &j, int64_t i) {
    if (j.info && i < 2) j.info[i] = 0;
    if (j.sync) {
        if (i < j.sync_ints) j.sync[i] = 0;
        if (i < j.winv_words) reinterpret_cast<unsigned long long *>(j.winv)[i] = kPending;
    }
    if (j.pending) {
        if (j.src && i < j.npad) j.z[i] = (i < j.n) ? j.src[i] : 0.0;
        if (i <= j.npad) reinterpret_cast<unsigned long long *>(j.pending)[i] = kPending;
    }
}

__global__ void __launch_bounds__(kThreads) init_kernel(InitJob job) {
    init_element(job, (int64_t) blockIdx.x * kThreads + threadIdx.x);
}

__global__ void __launch_bounds__(kThreads) init_batch_kernel(const InitJob *jobs) {
    init_element(jobs[blockIdx.y], (int64_t) blockIdx.x * kThreads + threadIdx.x);
}

// ------------------------------------------------------------------------
// Matrix-free Sigma v in FP64 for the refinement residual: the covariance is
// regenerated from the locations, never stored.  Workgroup (row block rb,
// column chunk cb) writes partial[cb * npad + row] = sum over the chunk's
// columns; reduce kernels add the chunks in a fixed order.
// ------------------------------------------------------------------------
constexpr int kChunk = 2048;

struct MatvecArgs {
    double *partial;
    const double *v;
    int64_t n, npad;
    MaternParams prm;
    Locs loc;
    int three_d;
};

__global__ void __launch_bounds__(kThreads) cov_matvec_kernel(MatvecArgs a) {
    __shared__ double sx[kChunk], sy[kChunk], sz[kChunk], sv[kChunk];
    __shared__ double sp[4][kBlk];
    const int t = threadIdx.x;
    const int r = t & 63, g = t >> 6;
    const int64_t row = (int64_t) blockIdx.x * kBlk + r;
    const int64_t c0 = (int64_t) blockIdx.y * kChunk;
    const int shift = a.prm.kernel == 1 ? 1 : 0;
    const bool three_d = a.three_d != 0;
    for (int e = t; e < kChunk; e += kThreads) {
        const int64_t c = c0 + e;
        const bool ok = c < a.n;
        const int64_t l = c >> shift;
        sx[e] = ok ? a.loc.x[l] : 0.0;
        sy[e] = ok ? a.loc.y[l] : 0.0;
        sz[e] = (ok && three_d) ? a.loc.z[l] : 0.0;
        sv[e] = ok ? a.v[c] : 0.0;
    }
    __syncthreads();
    double s = 0.0;
    if (row < a.n) {
        const int64_t li = row >> shift;
        const double rx = a.loc.x[li], ry = a.loc.y[li], rz = three_d ? a.loc.z[li] : 0.0;
        const int rvar = (int) (row & 1);
        const int cend = (int) min<int64_t>(kChunk, a.n - c0);
        for (int e = g; e < cend; e += 4) {
            const int64_t c = c0 + e;
            const int pair = shift ? (rvar * 2 + (int) (c & 1)) : 0;
            const double d = distance(rx, ry, rz, sx[e], sy[e], sz[e], a.prm.metric, three_d) / a.prm.range;
            const double cov = (d == 0.0) ? a.prm.sig[pair]
                                          : matern_scaled(d, a.prm.con[pair], a.prm.sig[pair], a.prm.nu[pair]);
            s += cov * sv[e];
        }
    }
    sp[g][r] = s;
    __syncthreads();
    if (t < kBlk) {
        const int64_t rr = (int64_t) blockIdx.x * kBlk + t;
        a.partial[(int64_t) blockIdx.y * a.npad + rr] = ((sp[0][t] + sp[1][t]) + sp[2][t]) + sp[3][t];
    }
}

// out[i] = base[i] + scale * sum_cb partial[cb][i]  (fixed chunk order), for i < npad.
__global__ void __launch_bounds__(kThreads) matvec_reduce_kernel(double *out, const double *base, double scale,
                                                                 const double *partial, int nchunks, int64_t n,
                                                                 int64_t npad) {
    const int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    if (i >= npad) return;
    double s = 0.0;
    for (int cb = 0; cb < nchunks; ++cb) s += partial[(int64_t) cb * npad + i];
    const double b = base ? base[i] : 0.0;
    out[i] = (i < n) ? b + scale * s : 0.0;
}

// Fixed-order dot products: block b sums indices b, b + G, b + 2G, ... then the
// host adds the G block sums in order.
constexpr int kDotBlocks = 256;

__global__ void __launch_bounds__(kThreads) dot_kernel(const double *x, const double *y, int64_t n, double *partial) {
    __shared__ double red[kThreads];
    double s = 0.0;
    const int64_t stride = (int64_t) kDotBlocks * kThreads;
    for (int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) s += x[i] * y[i];
    s = wg_sum(s, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// y = a * x + b * y
__global__ void __launch_bounds__(kThreads) axpby_kernel(double *y, const double *x, double a, double b, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    if (i < n) y[i] = a * x[i] + b * y[i];
}

void launch_cov_matvec(double *partial, const double *v, int64_t n, int64_t npad, const MaternParams &prm,
                       const double *x, const double *y, const double *z, hipStream_t s) {
    MatvecArgs a;
    a.partial = partial;
    a.v = v;
    a.n = n;
    a.npad = npad;
    a.prm = prm;
    a.loc = Locs{x, y, z};
    a.three_d = z != nullptr;
    const unsigned rows = (unsigned) (npad / kBlk);
    const unsigned chunks = (unsigned) ((n + kChunk - 1) / kChunk);
    hipLaunchKernelGGL(cov_matvec_kernel, dim3(rows, chunks), dim3(kThreads), 0, s, a);
}

int matvec_chunks(int64_t n) { return (int) ((n + kChunk - 1) / kChunk); }

void launch_matvec_reduce(double *out, const double *base, double scale, const double *partial, int nchunks,
                          int64_t n, int64_t npad, hipStream_t s) {
    hipLaunchKernelGGL(matvec_reduce_kernel, dim3((unsigned) ((npad + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       s, out, base, scale, partial, nchunks, n, npad);
}

int dot_blocks() { return kDotBlocks; }

void launch_dot(const double *x, const double *y, int64_t n, double *partial, hipStream_t s) {
    hipLaunchKernelGGL(dot_kernel, dim3(kDotBlocks), dim3(kThreads), 0, s, x, y, n, partial);
}

void launch_axpby(double *y, const double *x, double a, double b, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(axpby_kernel, dim3((unsigned) ((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, y, x, a,
                       b, n);
}

int64_t init_extent(const InitJob &j) {
    return std::max(j.sync ? std::max(j.sync_ints, j.winv_words) : 0, j.pending ? j.npad + 1 : 0);
}

void launch_init(const InitJob &job, hipStream_t s) {
    const int64_t n = init_extent(job);
    hipLaunchKernelGGL(init_kernel, dim3((unsigned) ((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, job);
}

void launch_init_batch(const InitJob *jobs, int count, int64_t most, hipStream_t s) {
    hipLaunchKernelGGL(init_batch_kernel, dim3((unsigned) ((most + kThreads - 1) / kThreads), count), dim3(kThreads), 0,
                       s, jobs);
}

void launch_forward(const TileMap &map, bool mixed, const double *winv, double *z, double *pending, double *partials,
                    int *info, hipStream_t s) {
    hipLaunchKernelGGL(mixed ? forward_kernel<true> : forward_kernel<false>, dim3((unsigned) map.blocks()), dim3(kThreads), 0,
                       s, map, winv, z, pending, partials, info);
}

void launch_forward_batch(const BatchJob *jobs, int njobs, int ts, int max_nt, hipStream_t s) {
    hipLaunchKernelGGL(forward_batch_kernel, dim3((unsigned) (njobs * max_nt * (ts / kBlk))), dim3(kThreads), 0, s, jobs,
                       njobs);
}

void launch_backward(const TileMap &map, bool mixed, const double *winv, double *z, double *pending, int *info,
                     hipStream_t s) {
    hipLaunchKernelGGL(mixed ? backward_kernel<true> : backward_kernel<false>, dim3((unsigned) map.blocks()), dim3(kThreads), 0,
                       s, map, winv, z, pending, info);
}

void launch_trmv(const TileMap &map, const double *e, double *out, hipStream_t s) {
    hipLaunchKernelGGL(trmv_kernel, dim3((unsigned) map.blocks()), dim3(kTrmvThreads), 0, s, map, e, out);
}

void launch_cov_gemv(double *out, int64_t rows, int64_t cols, const MaternParams &prm, const double *x1,
                     const double *y1, const double *z1, const double *x2, const double *y2, const double *z2,
                     const double *xv, const double *tabs, const double *word, hipStream_t s) {
    if (rows <= 0) return;
    CovGemvArgs a;
    a.out = out;
    a.rows = rows;
    a.cols = cols;
    a.prm = prm;
    a.l1 = Locs{x1, y1, z1};
    a.l2 = Locs{x2, y2, z2};
    a.x = xv;
    a.tabs = tabs;
    a.word = word;
    a.three_d = (z1 != nullptr && z2 != nullptr);
    static void (*const kernels[2][kTabSlots + 1])(CovGemvArgs) = {
        {cov_gemv_kernel<0, false>, cov_gemv_kernel<1, false>, cov_gemv_kernel<2, false>, cov_gemv_kernel<3, false>},
        {cov_gemv_kernel<0, true>, cov_gemv_kernel<1, true>, cov_gemv_kernel<2, true>, cov_gemv_kernel<3, true>}};
    hipLaunchKernelGGL(kernels[prm.metric == 1][prm.ntab], dim3((unsigned) rows), dim3(kThreads), 0, s, a);
}

void launch_dlarnv_normal(double *e, int64_t n, uint64_t seed48, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(dlarnv_normal_kernel, dim3((unsigned) ((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                       e, n, seed48);
}

void launch_copy_pad(double *dst, const double *src, int64_t n, int64_t npad, hipStream_t s) {
    if (npad <= 0) return;
    hipLaunchKernelGGL(copy_pad_kernel, dim3((unsigned) ((npad + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                       dst, src, n, npad);
}

// ------------------------------------------------------------------------
// Sigma v from the FP64 lower tiles (refinement of mixed plans).  One
// workgroup per tile (i, j); the tile is read once: wave w walks the columns
// in groups of four, c = 4 w + 16 p + u, lane l holds rows l + 64 m of a
// 512-row chunk.  The row
// products T v_j go to prow, the column products T' v_i (off the diagonal) to
// pcol; both are summed in a fixed order, so results are reproducible.
// ------------------------------------------------------------------------
constexpr int kRowsPerLane = 8;
constexpr int kChunkRows = 64 * kRowsPerLane;

__global__ void __launch_bounds__(kThreads) sigma_tile_matvec_kernel(const double *__restrict__ sig64,
                                                                     const int2 *__restrict__ pairs, int ts,
                                                                     const double *__restrict__ v,
                                                                     double *__restrict__ prow,
                                                                     double *__restrict__ pcol) {
    __shared__ double s_acc[kChunkRows];
    __shared__ double s_col[kMaxTs];
    const int2 ij = pairs[blockIdx.x];
    const int i = ij.x, j = ij.y;
    const int64_t tid = (int64_t) i * (i + 1) / 2 + j;
    const double *T = sig64 + tid * ts * ts;
    const double *vi = v + (int64_t) i * ts;
    const double *vj = v + (int64_t) j * ts;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const bool offdiag = i != j;
    for (int c = threadIdx.x; c < ts; c += kThreads) s_col[c] = 0.0;
    __syncthreads();
    for (int r0 = 0; r0 < ts; r0 += kChunkRows) {
        double acc[kRowsPerLane], vr[kRowsPerLane];
#pragma unroll
        for (int m = 0; m < kRowsPerLane; ++m) {
            const int r = r0 + lane + 64 * m;
            vr[m] = r < ts ? vi[r] : 0.0;
            acc[m] = 0.0;
        }
        // four consecutive columns per wave and pass, so that 32 loads per
        // lane are in flight; their four column dot products are reduced
        // across the wave together (7 shuffles instead of 24)
        constexpr int kPass = 4;
        constexpr int kStride = kPass * (kThreads / 64);
        const int cmain = ts - ts % kStride;
        for (int c0 = w * kPass; c0 < cmain; c0 += kStride) {
            double vc[kPass], dot[kPass];
#pragma unroll
            for (int u = 0; u < kPass; ++u) {
                vc[u] = vj[c0 + u];
                dot[u] = 0.0;
            }
            const double *col = T + (int64_t) c0 * ts + r0 + lane;
#pragma unroll
            for (int m = 0; m < kRowsPerLane; ++m) {
                if (r0 + lane + 64 * m < ts) {
#pragma unroll
                    for (int u = 0; u < kPass; ++u) {
                        const double t = __builtin_nontemporal_load(col + (int64_t) u * ts + 64 * m);
                        acc[m] += t * vc[u];
                        dot[u] += t * vr[m];
                    }
                }
            }
            if (offdiag) {
                // lanes with bit 5 clear keep columns 0, 1, set 2, 3; then bit
                // 4 picks one of the two: lane 16 q ends with column q
                const bool h32 = lane & 32, h16 = lane & 16;
                const double k0 = (h32 ? dot[2] : dot[0]) + __shfl_xor(h32 ? dot[0] : dot[2], 32, 64);
                const double k1 = (h32 ? dot[3] : dot[1]) + __shfl_xor(h32 ? dot[1] : dot[3], 32, 64);
                double d = (h16 ? k1 : k0) + __shfl_xor(h16 ? k0 : k1, 16, 64);
#pragma unroll
                for (int off = 8; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
                if ((lane & 15) == 0) s_col[c0 + (lane >> 4)] += d;
            }
        }
        for (int c = cmain + w; c < ts; c += kThreads / 64) {
            const double vc = vj[c];
            const double *col = T + (int64_t) c * ts + r0 + lane;
            double dot = 0.0;
#pragma unroll
            for (int m = 0; m < kRowsPerLane; ++m) {
                if (r0 + lane + 64 * m < ts) {
                    const double t = __builtin_nontemporal_load(col + 64 * m);
                    acc[m] += t * vc;
                    dot += t * vr[m];
                }
            }
            if (offdiag) {
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
                if (lane == 0) s_col[c] += dot;
            }
        }
        // the four waves' row partials, added in wave order
        for (int q = 0; q < kThreads / 64; ++q) {
            if (w == q) {
#pragma unroll
                for (int m = 0; m < kRowsPerLane; ++m) {
                    const int e = lane + 64 * m;
                    s_acc[e] = (q == 0 ? 0.0 : s_acc[e]) + acc[m];
                }
            }
            __syncthreads();
        }
        for (int e = threadIdx.x; e < kChunkRows && r0 + e < ts; e += kThreads) prow[tid * ts + r0 + e] = s_acc[e];
        __syncthreads();
    }
    if (offdiag)
        for (int c = threadIdx.x; c < ts; c += kThreads) pcol[tid * ts + c] = s_col[c];
}

__global__ void __launch_bounds__(kThreads) sigma_reduce_kernel(double *out, const double *base, double scale,
                                                                const double *__restrict__ prow,
                                                                const double *__restrict__ pcol, int nt, int ts,
                                                                int64_t n, int64_t npad) {
    const int64_t g = (int64_t) blockIdx.x * kThreads + threadIdx.x;
    if (g >= npad) return;
    const int i = (int) (g / ts), r = (int) (g % ts);
    double acc = 0.0;
    for (int j = 0; j <= i; ++j) acc += prow[((int64_t) i * (i + 1) / 2 + j) * ts + r];
    for (int j = i + 1; j < nt; ++j) acc += pcol[((int64_t) j * (j + 1) / 2 + i) * ts + r];
    out[g] = g < n ? (base ? base[g] : 0.0) + scale * acc : 0.0;
}

void launch_sigma_tile_matvec(const double *sig64, const int2 *pairs, int npairs, int ts, const double *v,
                              double *prow, double *pcol, hipStream_t s) {
    if (npairs <= 0) return;
    hipLaunchKernelGGL(sigma_tile_matvec_kernel, dim3((unsigned) npairs), dim3(kThreads), 0, s, sig64, pairs, ts, v,
                       prow, pcol);
}

void launch_sigma_reduce(double *out, const double *base, double scale, const double *prow, const double *pcol,
                         int nt, int ts, int64_t n, int64_t npad, hipStream_t s) {
    if (npad <= 0) return;
    hipLaunchKernelGGL(sigma_reduce_kernel, dim3((unsigned) ((npad + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                       out, base, scale, prow, pcol, nt, ts, n, npad);
}

// partials[2b] = sum of log L_ii (L_ii > 0) over 64-row block b, partials[2b+1] = 0.
__global__ void __launch_bounds__(kBlk) diag_logdet_kernel(TileMap map, double *partials) {
    const int b = blockIdx.x, nsb = map.ts / kBlk;
    const double d = tile_f64(map, b / nsb, b / nsb)[(int64_t) ((b % nsb) * kBlk + threadIdx.x) * (map.ts + 1)];
    const double ld = wave_sum(d > 0.0 ? log(d) : 0.0);
    if (threadIdx.x == 0) {
        partials[2 * b] = ld;
        partials[2 * b + 1] = 0.0;
    }
}

void launch_diag_logdet(const TileMap &map, double *partials, hipStream_t s) {
    hipLaunchKernelGGL(diag_logdet_kernel, dim3((unsigned) map.blocks()), dim3(kBlk), 0, s, map, partials);
}

}  // namespace egs
