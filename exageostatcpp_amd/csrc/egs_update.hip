// Trailing SYRK/GEMM update of the tiled Cholesky on gfx950, the kernel that
// carries ~95% of the factorization flops (the reference's Chameleon runs the
// same tile update C_ij -= L_ik L_jk^T as dsyrk/dgemm tasks).
//
// One workgroup of 256 threads (4 waves) owns a 96 x 192 block of C_ij and
// contracts over K = ts with v_mfma_f64_16x16x4f64; two workgroups share a CU:
//   * wave w covers all 96 rows and columns 48 w .. +48, i.e. 6 x 3 independent
//     16 x 16 accumulators (72 FP64 values per lane);
//   * A and B are staged through LDS in K-chunks of 16 columns, double
//     buffered; a chunk's loads stay in flight in registers for a whole chunk,
//     and the operands of four K columns are read from LDS while the four
//     before are multiplied;
//   * C -= acc goes out as FP64 atomic adds at the L2 (each element is added to
//     once per launch, so the sum has one rounding and no order): nothing waits
//     for C, where a read-modify-write spent 20 us per workgroup on it.
// Bound: FP64 MFMA, 64 cycles per instruction and SIMD (77.8 TF/s measured).
// Measured, all tiles of a step: 210 tiles of 960: 59.2 -> 65.0 TF/s, 861
// tiles 62.4 -> 67.2, 351 tiles of 384 49.1 -> 56.1 (one 192 x 192 block of 8
// waves per CU, whose C traffic nothing overlapped, before).
// The operand panel is either the tile arena itself or a contiguous FP64 copy
// of panel k (PanelRef), so the inner loop has no type dispatch.
#include "egs_common.hpp"
#include "egs_kernels.hpp"

namespace egs {

namespace {

constexpr int kBR = 96;            // block rows
constexpr int kBC = 192;           // block columns
constexpr int kKC = 16;            // K chunk
constexpr int kNT = 256;           // threads per workgroup

typedef double f64x2 __attribute__((ext_vector_type(2)));

// Where the operand tiles of panel k live: in the tile arena itself (FP64 plan)
// or in a contiguous FP64 copy of the panel (mixed plans), tile i of the panel
// at pbase + (i - k - 1) * pstride.
struct PanelRef {
    const char *pbase;
    int64_t pstride;
    int contiguous;
};

__device__ __forceinline__ const double *panel_tile(const TileMap &map, const PanelRef &pr, int i, int k) {
    if (pr.contiguous) return reinterpret_cast<const double *>(pr.pbase + (int64_t) (i - k - 1) * pr.pstride);
    return reinterpret_cast<const double *>(map.base + map.off[i * map.nt + k]);
}

// kPanels = 2: with the panels k and k + 1 of an FP64 plan, one after the other.
template <int kPanels>
__global__ void __launch_bounds__(kNT, 2) update192_kernel(TileMap map, PanelRef pr, const int2 *pairs, int k) {
    __shared__ __align__(16) double sA[2][kKC * kBR];
    __shared__ __align__(16) double sB[2][kKC * kBC];
    const int ts = map.ts;
    const int nbr = ts / kBR;
    const int nsub = nbr * (ts / kBC);
    const int bid = xcd_remap((int) blockIdx.x, (int) gridDim.x);
    const int pair = bid / nsub;
    const int sub = bid % nsub;
    const int sbm = sub % nbr, sbn = sub / nbr;
    const int2 ij = pairs[pair];
    if (ij.x == ij.y && (sbm + 1) * kBR <= sbn * kBC) return;   // strictly upper block of a diagonal tile
    if (sbm * kBR >= map.blocks(ij.x) * kBlk || sbn * kBC >= map.blocks(ij.y) * kBlk) return;   // padding

    const double *A = panel_tile(map, pr, ij.x, k) + sbm * kBR;
    const double *B = panel_tile(map, pr, ij.y, k) + sbn * kBC;
    const double *A2 = kPanels == 2 ? panel_tile(map, pr, ij.x, k + 1) + sbm * kBR : nullptr;
    const double *B2 = kPanels == 2 ? panel_tile(map, pr, ij.y, k + 1) + sbn * kBC : nullptr;
    const int per_panel = ts / kKC;

    const int t = threadIdx.x;
    const int lane = t & 63, w = t >> 6;
    const int lr = lane & 15, lk = lane >> 4;

    // staging in 16-byte vectors (ts and the blocks are multiples of 64 rows):
    // of A rows 2 (t % 16) + 32 q of column t / 16, of B rows 2 (t % 32) + 64 q
    // of columns t / 32 and t / 32 + 8
    const uint32_t ga = (uint32_t) (2 * (t & 15) + (t >> 4) * ts);
    const uint32_t gb = (uint32_t) (2 * (t & 31) + (t >> 5) * ts);
    const int la = 2 * (t & 15) + (t >> 4) * kBR;
    const int lb = 2 * (t & 31) + (t >> 5) * kBC;
    f64x2 ra[3], rb[6];
    auto issue = [&](int c) {
        const bool second = kPanels == 2 && c >= per_panel;
        const int64_t at = (int64_t) (second ? c - per_panel : c) * kKC * ts;
        const double *Ac = (second ? A2 : A) + at;
        const double *Bc = (second ? B2 : B) + at, *Bd = Bc + (int64_t) (kKC / 2) * ts;
#pragma unroll
        for (int q = 0; q < 3; ++q) ra[q] = *reinterpret_cast<const f64x2 *>(Ac + ga + 32 * q);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            rb[q] = *reinterpret_cast<const f64x2 *>(Bc + gb + 64 * q);
            rb[3 + q] = *reinterpret_cast<const f64x2 *>(Bd + gb + 64 * q);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<f64x2 *>(&sA[buf][la + 32 * q]) = ra[q];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            *reinterpret_cast<f64x2 *>(&sB[buf][lb + 64 * q]) = rb[q];
            *reinterpret_cast<f64x2 *>(&sB[buf][lb + 64 * q + (kKC / 2) * kBC]) = rb[3 + q];
        }
    };

    f64x4 acc[6][3];
#pragma unroll
    for (int mi = 0; mi < 6; ++mi)
#pragma unroll
        for (int ni = 0; ni < 3; ++ni) acc[mi][ni] = f64x4{0.0, 0.0, 0.0, 0.0};

    // operands of K columns kk .. kk + 3 of a chunk, in two register sets
    const int fa = lk * kBR + lr, fb = lk * kBC + w * 48 + lr;
    double a[2][6], b[2][3];
    auto read = [&](int set, int buf, int kk) {
#pragma unroll
        for (int ni = 0; ni < 3; ++ni) b[set][ni] = sB[buf][kk * kBC + fb + ni * 16];
#pragma unroll
        for (int mi = 0; mi < 6; ++mi) a[set][mi] = sA[buf][kk * kBR + fa + mi * 16];
        __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of the products before theirs
    };
    auto multiply = [&](int set, int m0, int m1) {
#pragma unroll
        for (int mi = m0; mi < m1; ++mi)
#pragma unroll
            for (int ni = 0; ni < 3; ++ni) acc[mi][ni] = mfma_f64(b[set][ni], a[set][mi], acc[mi][ni]);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int nchunks = kPanels * per_panel;
    issue(0);
    stage(0);
    issue(1);
    __syncthreads();
    read(0, 0, 0);
    for (int c = 0; c + 1 < nchunks; ++c) {
        const int buf = c & 1;
        read(1, buf, 4);
        multiply(0, 0, 6);
        read(0, buf, 8);
        multiply(1, 0, 2);
        stage(buf ^ 1);
        multiply(1, 2, 4);
        if (c + 2 < nchunks) issue(c + 2);
        multiply(1, 4, 6);
        read(1, buf, 12);
        multiply(0, 0, 6);
        __syncthreads();   // chunk c + 1 is staged, and every wave has read chunk c
        read(0, buf ^ 1, 0);
        multiply(1, 0, 6);
    }
    const int buf = (nchunks - 1) & 1;
    read(1, buf, 4);
    multiply(0, 0, 6);
    read(0, buf, 8);
    multiply(1, 0, 6);
    read(1, buf, 12);
    multiply(0, 0, 6);
    multiply(1, 0, 6);

    // C -= acc.  Lane l, element v of acc[mi][ni] is
    // C[mi*16 + l%16][w*48 + ni*16 + l/16 + 4v]  (FP64 MFMA output order).
    // This workgroup alone updates these elements: the adds are done at this
    // XCD's L2 (workgroup scope).
    double *C = tile_f64(map, ij.x, ij.y);
    const uint32_t cbase = (uint32_t) ((sbm * kBR + lr) + (sbn * kBC + w * 48 + lk) * ts);
#pragma unroll
    for (int mi = 0; mi < 6; ++mi)
#pragma unroll
        for (int ni = 0; ni < 3; ++ni)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                [[clang::atomic(no_remote_memory, no_fine_grained_memory)]] {
                    __hip_atomic_fetch_add(&C[cbase + (uint32_t) (mi * 16 + (ni * 16 + 4 * v) * ts)], -acc[mi][ni][v],
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
}

}  // namespace

bool update192_supported(int ts) { return ts % kBC == 0; }

void launch_update192(const TileMap &map, const double *p64, const int2 *pairs, int npairs, int k, int panels,
                      hipStream_t s) {
    if (npairs <= 0) return;
    const unsigned blocks = (unsigned) npairs * (unsigned) ((map.ts / kBR) * (map.ts / kBC));
    const PanelRef pr{reinterpret_cast<const char *>(p64), (int64_t) map.ts * map.ts * (int64_t) sizeof(double),
                      p64 != nullptr};
    hipLaunchKernelGGL(panels == 2 ? update192_kernel<2> : update192_kernel<1>, dim3(blocks), dim3(kNT), 0, s, map, pr,
                       pairs, k);
}

}  // namespace egs
