// Shared device/host definitions for the gfx950 kernels of exageostatcpp_amd.
//
// Matrix storage: the covariance matrix of dimension n (= locations x variables)
// is held as lower tiles of ts x ts elements (ts = the dense tile size rounded up
// to a multiple of 64).  Each tile is column-major with leading dimension ts and
// owns its own block of one HBM arena, so every tile can carry its own storage
// precision.  The matrix is padded to npad = nt * ts with the identity, which
// keeps it SPD, leaves log|Sigma| unchanged and lets every kernel work on full
// 64-row blocks without bounds checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace egs {

constexpr int kBlk = 64;        // sub-block edge used by every factorization kernel
constexpr int kThreads = 256;   // 4 waves of 64 lanes per workgroup

enum StoragePrecision : uint8_t { kStoreF64 = 0, kStoreF32 = 1 };
enum ComputeClass : uint8_t { kComputeF64 = 0, kComputeF32 = 1, kComputeBF16 = 2 };

// Location of every lower tile in the arena.  off[i * nt + j] is the byte offset
// of tile (i, j), i >= j; store[i * nt + j] its storage precision.  Of the last
// tile row only the first last_blocks 64-row blocks hold rows of the matrix; the
// factorization and the solves leave out the blocks that are all padding (which
// is its own factor): up to a tile's worth of work per row and column (400
// locations in tiles of 384: 310 -> 247 us; 6,001 in tiles of 960: 4.32 -> 3.83
// ms; 10,007 in tiles of 960: 10.7 -> 9.6 ms).
struct TileMap {
    char *base;
    const int64_t *off;
    const uint8_t *store;
    int nt;
    int ts;
    int last_blocks;

    // 64-row blocks of tile row i, and of the whole matrix, that are not padding
    __host__ __device__ int blocks(int i) const { return i == nt - 1 ? last_blocks : ts / kBlk; }
    __host__ __device__ int blocks() const { return (nt - 1) * (ts / kBlk) + last_blocks; }
};

__device__ __forceinline__ double *tile_f64(const TileMap &m, int i, int j) {
    return reinterpret_cast<double *>(m.base + m.off[i * m.nt + j]);
}
__device__ __forceinline__ float *tile_f32(const TileMap &m, int i, int j) {
    return reinterpret_cast<float *>(m.base + m.off[i * m.nt + j]);
}

// What a launch only reads, the same for the whole wave (the tile table, a job's
// record), through scalar loads: it stays out of the vector registers, and
// waiting for it does not wait for the vector loads in flight.
template <typename T> __device__ __forceinline__ T scalar_load(const T *p) {
    typedef const __attribute__((address_space(4))) uint32_t *Words;
    if constexpr (sizeof(T) % 4 != 0 || alignof(T) < 4) return *p;
    const Words q = reinterpret_cast<Words>(reinterpret_cast<uintptr_t>(p));
    union U {
        uint32_t w[sizeof(T) / 4];
        T v;
        __device__ U() {}
    } u;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) u.w[i] = q[i];
    return u.v;
}

// What workgroups of one launch hand each other goes past the L2s, each of which
// belongs to an XCD: stored and loaded at agent scope.  A word that holds ~0
// (kPending) has not been stored yet, so that the value is its own flag; a NaN of
// that pattern is stored as another one.
constexpr unsigned long long kPending = ~0ull;

__device__ __forceinline__ double load_shared(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool is_pending(double v) {
    return __builtin_bit_cast(unsigned long long, v) == kPending;
}
__device__ __forceinline__ void store_shared(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_word(double *p, double v) {
    store_shared(p, is_pending(v) ? __builtin_bit_cast(double, 0x7ff8000000000000ull) : v);
}

// Every wait for another workgroup of a launch ends: after kPatience requests
// (of half a microsecond and more: several seconds, where the longest wait that
// was measured is a few milliseconds) the wave sets *lost and goes on with what is
// there, and every other wait of the launch follows within kLook requests.  The
// host reads lost with the results.
struct Patience {
    int *lost;
    unsigned polls = 0;

    __device__ __forceinline__ bool over() {
        constexpr unsigned kPatience = 1u << 23, kLook = 1u << 10;
        if ((++polls & (kLook - 1)) != 0) return false;
        if (polls >= kPatience) __hip_atomic_store(lost, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_amdgcn_readfirstlane(__hip_atomic_load(lost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
    }
};

// Workgroups are dispatched to the 8 XCDs of an MI355X round-robin (workgroup w
// runs on XCD w % 8), and each XCD has its own L2.  xcd_remap gives XCD x a
// contiguous range of the logical block order, so blocks that share operand
// rows (consecutive logical blocks) meet in the same L2.  It is a bijection
// of [0, n).
__device__ __forceinline__ int xcd_remap(int w, int n) {
    constexpr int kXcd = 8;
    const int q = n / kXcd, r = n % kXcd;
    const int x = w % kXcd, i = w / kXcd;
    return x * q + min(x, r) + i;
}

// The same idea for blocks of uneven cost: groups of g consecutive logical
// blocks (one tile's blocks) are dealt to the XCDs in turn, XCD x taking
// groups x, x + 8, x + 16, ...  A group's blocks meet in one L2, and every
// XCD gets a share of each part of the order, so a run of expensive tiles
// does not all land on one XCD (with xcd_remap's contiguous ranges the last
// XCD took every tile at the end of the list).  Workgroups past the last full
// round of 8 g keep their index.  A bijection of [0, n).
__device__ __forceinline__ int xcd_deal(int w, int n, int g) {
    constexpr int kXcd = 8;
    const int full = n / (kXcd * g) * (kXcd * g);
    if (w >= full) return w;
    const int x = w % kXcd, i = w / kXcd;
    return (i / g) * (kXcd * g) + x * g + i % g;
}

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// D[i][j] += sum_k X[i][k] Y[k][j] on a 16x16x4 tile.  Lane l supplies X[l%16][l/16]
// and Y[l/16][l%16].  Result element v (0..3) of lane l is D[l/16 + 4*v][l%16] for
// the FP64 instruction and D[4*(l/16) + v][l%16] for the FP32 one (both measured
// on gfx950).
__device__ __forceinline__ f64x4 mfma_f64(double x, double y, f64x4 acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f32(float x, float y, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc, 0, 0, 0);
}

}  // namespace egs
