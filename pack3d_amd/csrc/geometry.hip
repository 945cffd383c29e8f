// Integer geometry kernels: layout construction, validation, reverse
// adjacency and repack transport.  Every output is bit-exact with the CPU
// construction of amilworks/Pack3D (src/pack3d/geometry.py).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "index.hpp"

namespace p3d {
namespace {

constexpr int kThreads = 256;

inline unsigned grid1d(int64_t n) { return (unsigned)cdiv(n, kThreads); }

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill_i64(int64_t* p, int64_t n, int64_t v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Number of points q of the box [0,E0) x [0,E1) x [0,E2) whose Morton code
// is smaller than that of p.  Codes interleave bit b of axis a at bit 3b+a
// (geometry.py:118-126).  Scanning code bits from the top, every 1 bit of p
// contributes the points that agree with p above it, hold 0 there and are
// free below; per axis that set is an aligned power-of-two interval clipped
// to the box, so the count is a product of three clipped lengths.
__device__ int32_t morton_rank(const int32_t p[3], const int32_t E[3], int nbits) {
    int32_t rank = 0;
    for (int b = nbits - 1; b >= 0; --b) {
        for (int a = 2; a >= 0; --a) {
            if (!((p[a] >> b) & 1)) continue;
            int32_t count = 1;
            for (int c = 0; c < 3 && count; ++c) {
                int32_t prefix;
                int k;
                if (c == a) {
                    prefix = (p[a] >> (b + 1)) << 1;
                    k = b;
                } else if (c < a) {
                    prefix = p[c] >> (b + 1);
                    k = b + 1;
                } else {
                    prefix = p[c] >> b;
                    k = b;
                }
                int32_t room = E[c] - (prefix << k);
                int32_t span = 1 << k;
                count = room <= 0 ? 0 : count * (room < span ? room : span);
            }
            rank += count;
        }
    }
    return rank;
}

struct LayoutDims {
    int64_t g[3], blk[3], r[3];
    int64_t n, volume;
    int morton, nbits;
};

// Per raster token t: packed row, order, coordinates and raster->packed map
// (geometry.py:241-252).  Morton keys block_code*(max_slot+1)+slot_code are
// ordered lexicographically by (block code, slot code) and every block holds
// every slot, so the packed row is rank(block) * volume + rank(slot).
__global__ void k_layout_map(LayoutDims d, int64_t* order, int64_t* coords, int32_t* map) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= d.n) return;
    // N < 2^31: 32-bit arithmetic for rows (not for entries of the coordinate table).
    const int32_t Y = (int32_t)d.g[1], X = (int32_t)d.g[2], t32 = (int32_t)t;
    const int32_t x = t32 % X, zy = t32 / X, y = zy % Y, z = zy / Y;
    int32_t packed = t32;
    if (d.morton) {
        const int32_t blk[3] = {(int32_t)d.blk[0], (int32_t)d.blk[1], (int32_t)d.blk[2]};
        const int32_t bc[3] = {z / blk[0], y / blk[1], x / blk[2]};
        const int32_t sc[3] = {z % blk[0], y % blk[1], x % blk[2]};
        const int32_t be[3] = {(int32_t)d.g[0] / blk[0], Y / blk[1], X / blk[2]};
        packed = morton_rank(bc, be, d.nbits) * (int32_t)d.volume + morton_rank(sc, blk, d.nbits);
    }
    if (map) map[t] = packed;
    order[packed] = t;
    const int64_t at = coord_start(packed);
    coords[at + 0] = z;
    coords[at + 1] = y;
    coords[at + 2] = x;
}

// Lanes per row of the row-wise table kernels: two rows share a wave up to 32
// columns, one wave takes a row of up to 64, and rows of up to 128 columns put
// elements l and l + 64 in lane l (two registers).  One wave per row rather
// than one thread per element keeps every per-row quantity (coordinates,
// permutation, row start) uniform and the column's offset loop-invariant, so
// no element pays a 64-bit division.
template <int COLS>
struct RowLanes {
    static constexpr int LANES = COLS < 64 ? COLS : 64;
    static constexpr int REGS = COLS > 64 ? 2 : 1;
    static constexpr int ROWS = 64 / LANES;  // rows per wave
};

// Calls f(integral constant) with the smallest of 32, 64 and 128 columns that
// holds `width`.
template <typename F>
void with_columns(int width, F f) {
    if (width <= 32) f(std::integral_constant<int, 32>{});
    else if (width <= 64) f(std::integral_constant<int, 64>{});
    else f(std::integral_constant<int, 128>{});
}

// Blocks of 4 waves over n rows, each wave walking its rows with a grid stride.
template <int COLS>
unsigned row_blocks(int64_t n) {
    return (unsigned)std::min<int64_t>(cdiv(n, 4 * RowLanes<COLS>::ROWS), 4096);
}

// The sorting kernels take four rows per wave, 16 lanes each.
unsigned sort_blocks(int64_t n) { return (unsigned)std::min<int64_t>(cdiv(n, 16), 4096); }

// Neighbour column k is offset ((dz+rz)(2ry+1)+(dy+ry))(2rx+1)+(dx+rx), the
// itertools.product order of geometry.py:254-259; absent neighbours are -1.
// Bound by its stores (4 N W bytes).  At 131,072 rows of 125 columns: 61 us as
// one thread per element, 30 us as one wave per row.
template <int COLS>
__global__ __launch_bounds__(256) void k_layout_neighbors(LayoutDims d, int32_t width, const int64_t* coords,
                                                          const int32_t* map, int32_t* nb) {
    typedef RowLanes<COLS> R;
    const int lane = threadIdx.x & 63, k0 = lane % R::LANES;
    const int Z = (int)d.g[0], Y = (int)d.g[1], X = (int)d.g[2];
    const int wy = 2 * (int)d.r[1] + 1, wx = 2 * (int)d.r[2] + 1;
    int oz[R::REGS], oy[R::REGS], ox[R::REGS];
#pragma unroll
    for (int r = 0; r < R::REGS; ++r) {
        const int k = k0 + 64 * r;
        oz[r] = k / (wy * wx) - (int)d.r[0];
        oy[r] = (k / wx) % wy - (int)d.r[1];
        ox[r] = k % wx - (int)d.r[2];
    }
    const int64_t step = (int64_t)gridDim.x * 4 * R::ROWS;
    for (int64_t i = ((int64_t)blockIdx.x * 4 + threadIdx.x / 64) * R::ROWS + lane / R::LANES; i < d.n; i += step) {
        const int cz = (int)coords[3 * i], cy = (int)coords[3 * i + 1], cx = (int)coords[3 * i + 2];
#pragma unroll
        for (int r = 0; r < R::REGS; ++r) {
            const int k = k0 + 64 * r;
            if (k >= width) continue;
            const int z = cz + oz[r], y = cy + oy[r], x = cx + ox[r];
            const bool inside = (unsigned)z < (unsigned)Z && (unsigned)y < (unsigned)Y && (unsigned)x < (unsigned)X;
            int v = -1;
            if (inside) {
                v = (z * Y + y) * X + x;  // N < 2^31
                if (map) v = map[v];
            }
            nb[i * width + k] = v;
        }
    }
}

__global__ void k_iota_i32(int32_t* p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int32_t)i;
}

// ----------------------------------------------------------- validation
template <typename I>
__global__ void k_check_neighbors(const I* nb, int64_t count, int64_t n, int32_t* out,
                                  int32_t* degree, int32_t* flags) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    int64_t v = (int64_t)nb[e];
    bool bad = v < -1 || v >= n;
    out[e] = bad ? -1 : (int32_t)v;
    if (bad) atomicAdd(&flags[0], 1);
    else if (v >= 0) atomicAdd(&degree[v], 1);
}

template <typename I>
__global__ void k_check_blocks(const I* blocks, int64_t count, int64_t n, int32_t* out,
                               int32_t* cover, int32_t* flags) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    int64_t v = (int64_t)blocks[e];
    bool bad = v < -1 || v >= n;
    out[e] = bad ? -1 : (int32_t)v;
    if (bad) atomicAdd(&flags[1], 1);
    else if (v >= 0) atomicAdd(&cover[v], 1);
}

// v of the lane at distance XOR M within a 16-lane row, on the VALU (DPP).
template <int CTRL>
__device__ __forceinline__ int32_t dpp_i32(int32_t v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int M>
__device__ __forceinline__ int32_t lane_xor(int32_t v) {
    static_assert(M == 1 || M == 2 || M == 3 || M == 4 || M == 7 || M == 15, "no such permutation");
    if constexpr (M == 1) return dpp_i32<0xB1>(v);        // quad_perm 1,0,3,2
    else if constexpr (M == 2) return dpp_i32<0x4E>(v);   // quad_perm 2,3,0,1
    else if constexpr (M == 3) return dpp_i32<0x1B>(v);   // quad_perm 3,2,1,0
    else if constexpr (M == 7) return dpp_i32<0x141>(v);  // row_half_mirror
    else if constexpr (M == 15) return dpp_i32<0x140>(v); // row_mirror
    else return lane_xor<3>(lane_xor<7>(v));
}

// Ascending sort of the 16 R values of each 16-lane row, by any input order,
// to element R l + r in register r of lane l: bitonic merges whose first
// exchange mirrors the second run, so every run ascends.  With the low bits
// of the index in the registers, 18 of the 28 exchanges of 128 values are
// plain min / max pairs and the other 10 stay within a DPP row: about 50 VALU
// operations per value and no LDS.  131,072 rows of 125 values: 81 us with a
// row per wave through __shfl_xor, 58 us with a row per wave and one value
// per register on DPP and the row swaps, 33 us like this.
template <int R, int J>
__device__ __forceinline__ void halve_regs(int32_t (&a)[R]) {
    if constexpr (J >= 1) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (!(r & J)) {
                const int32_t lo = min(a[r], a[r | J]), hi = max(a[r], a[r | J]);
                a[r] = lo;
                a[r | J] = hi;
            }
        halve_regs<R, J / 2>(a);
    }
}
template <int R, int J>  // J: lane distance
__device__ __forceinline__ void halve_lanes(int32_t (&a)[R]) {
    if constexpr (J >= 1) {
        const bool upper = __lane_id() & J;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int32_t p = lane_xor<J>(a[r]);
            a[r] = upper ? max(a[r], p) : min(a[r], p);
        }
        halve_lanes<R, J / 2>(a);
    }
}
template <int R, int K>  // merge within the registers: runs of K / 2 -> K
__device__ __forceinline__ void merge_regs(int32_t (&a)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (!(r & (K / 2))) {
            const int q = r ^ (K - 1);
            const int32_t lo = min(a[r], a[q]), hi = max(a[r], a[q]);
            a[r] = lo;
            a[q] = hi;
        }
    halve_regs<R, K / 4>(a);
}
template <int R, int L>  // merge runs of L / 2 lanes -> L
__device__ __forceinline__ void merge_lanes(int32_t (&a)[R]) {
    const bool upper = __lane_id() & (L / 2);
    int32_t b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int32_t p = lane_xor<L - 1>(a[R - 1 - r]);
        b[r] = upper ? max(a[r], p) : min(a[r], p);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = b[r];
    halve_lanes<R, L / 4>(a);
    halve_regs<R, R / 2>(a);
}
template <int R>
__device__ __forceinline__ void sort_rows(int32_t (&a)[R]) {
    static_assert(R == 2 || R == 4 || R == 8, "registers per lane");
    merge_regs<R, 2>(a);
    if constexpr (R >= 4) merge_regs<R, 4>(a);
    if constexpr (R >= 8) merge_regs<R, 8>(a);
    merge_lanes<R, 2>(a);
    merge_lanes<R, 4>(a);
    merge_lanes<R, 8>(a);
    merge_lanes<R, 16>(a);
}

// Sorts each row and looks for equal valid neighbours.
template <int COLS>
__global__ __launch_bounds__(256) void k_check_duplicates(const int32_t* nb, int64_t n, int32_t width,
                                                          int32_t* flags) {
    constexpr int R = COLS / 16;
    const int lane = threadIdx.x & 63, e = lane & 15;
    const int64_t step = (int64_t)gridDim.x * 16;
    bool any = false;
    // Every lane of a wave runs the same number of rounds (the sort reads its
    // whole 16-lane row): rows past the end hold no valid entry.
    for (int64_t first = ((int64_t)blockIdx.x * 4 + threadIdx.x / 64) * 4; first < n; first += step) {
        const int64_t row = first + (lane >> 4);
        int32_t a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = e + 16 * r;
            a[r] = row < n && k < width ? nb[row * width + k] : INT_MAX;
            if (a[r] < 0) a[r] = INT_MAX;
        }
        sort_rows<R>(a);
        const int32_t next = __shfl_down(a[0], 1);
        any = any || (e < 15 && a[R - 1] != INT_MAX && a[R - 1] == next);
#pragma unroll
        for (int r = 0; r + 1 < R; ++r) any = any || (a[r] != INT_MAX && a[r] == a[r + 1]);
    }
    if (__ballot(any) && lane == 0) atomicAdd(&flags[2], 1);
}

// degree may be null (the bucketed check finds the largest degree by itself).
__global__ void k_check_cover(const int32_t* cover, const int32_t* degree, int64_t n, int32_t* flags) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool miss = t < n && cover[t] != 1;
    const int most = wave_max_i(degree && t < n ? degree[t] : 0);
    const unsigned long long misses = __ballot(miss);
    if ((threadIdx.x & 63) == 0) {
        if (misses) atomicAdd(&flags[3], __popcll(misses));
        if (most) atomicMax(&flags[5], most);
    }
}

__global__ void k_check_groups(const int32_t* blocks, int64_t fine, int32_t slots, int32_t pool,
                               int64_t groups, int32_t* flags) {
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= groups) return;
    int64_t end = min(fine, (g + 1) * pool);
    bool any = false;
    for (int64_t f = g * pool; f < end && !any; ++f)
        for (int s = 0; s < slots; ++s) any = any || blocks[f * slots + s] >= 0;
    if (!any) atomicAdd(&flags[4], 1);
}

// ------------------------------------------------------ reverse adjacency
__global__ void k_reverse_scatter(const int32_t* nb, int64_t count, int32_t width, int32_t* cursor,
                                  int32_t* reverse, int32_t rwidth) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    int32_t j = nb[e];
    if (j < 0) return;
    int32_t slot = atomicAdd(&cursor[j], 1);
    if (slot < rwidth) reverse[(int64_t)j * rwidth + slot] = (int32_t)(e / width);
}

// Reverse rows out[i] = the valid entries of source row i (row perm[i] where a
// permutation is given, each entry relabelled by `inverse`), ascending, padded
// with -1: the order that the stable argsort of geometry.py:90 produces.  The
// source is a table whose row i lists, in any order, the rows that reach i:
// a reverse table filled in arbitrary order (in place), the neighbour table of
// a symmetric graph (a complete stencil), or the reverse table that a repack
// relabels.  None of these needs the edges to be scattered by destination:
// 38 us for 131,072 rows of 125 entries (131 MB read and written) against
// 1,530 us through p3d_reverse_adjacency.
template <int COLS>
__global__ __launch_bounds__(256) void k_reverse_rows(const int32_t* rows, int64_t n, int32_t width,
                                                      const int64_t* perm, const int64_t* inverse, int32_t* out,
                                                      int32_t rwidth) {
    constexpr int R = COLS / 16;
    typedef __attribute__((ext_vector_type(R))) int32_t Regs;
    __shared__ __align__(16) int32_t sorted[4][4][COLS];
    const int lane = threadIdx.x & 63, e = lane & 15, q = lane >> 4;
    int32_t* mine = sorted[threadIdx.x / 64][q];
    const int64_t step = (int64_t)gridDim.x * 16;
    for (int64_t first = ((int64_t)blockIdx.x * 4 + threadIdx.x / 64) * 4; first < n; first += step) {
        const int64_t row = first + q;
        const int64_t src = row < n ? (perm ? perm[row] : row) : 0;
        int32_t a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = e + 16 * r;
            int32_t v = row < n && k < width ? rows[src * width + k] : -1;
            if (v >= 0 && inverse) v = (int32_t)inverse[v];
            a[r] = v < 0 ? INT_MAX : v;
        }
        sort_rows<R>(a);
        Regs v;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = a[r] == INT_MAX ? -1 : a[r];
        // Through LDS, so that consecutive lanes store consecutive entries.
        wave_lds_sync();
        *reinterpret_cast<Regs*>(mine + R * e) = v;
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = e + 16 * r;
            if (row < n && k < rwidth) out[row * rwidth + k] = mine[k];
        }
    }
}

// ------------------------------------------------- bucketed transposition
// The reverse adjacency of an arbitrary graph, without a global atomic per
// edge: edges are grouped by destination bucket (kBucketRows consecutive rows)
// with one workgroup per chunk of the table counting and placing its edges
// through LDS counters, and one atomic per (chunk, bucket) pair reserving
// their space; then one workgroup per bucket fills its reverse rows in LDS,
// sorts them and writes them out.  At 131,072 rows of 125 columns the table
// took 565 us for the in-degrees (16 M global atomics) and 1,530 us for the
// reverse rows (16 M returning atomics and scattered 4-byte stores); this
// takes 28 + 73 + 30 (count, scatter, degrees) and 58 us.
constexpr int kBucketRows = 128;     // a bucket's reverse rows: up to 64 KB of LDS
constexpr int kMaxBuckets = 8192;    // LDS counters of a chunk: 32 KB; n up to 2^20 rows
constexpr int kBucketThreads = 1024;

struct Buckets {
    int32_t n_buckets;
    int32_t *count, *cursor, *start;  // [n_buckets], [n_buckets], [n_buckets + 1]
    uint32_t* edges;                  // (row within the bucket) << 24 | source row
};

inline int64_t bucket_count(int64_t n) { return cdiv(n, kBucketRows); }

int64_t bucket_bytes(int64_t n, int32_t width) {
    if (n < 1 || width < 1 || width > 128 || n * width >= ((int64_t)1 << 31) || bucket_count(n) > kMaxBuckets) return 0;
    return (3 * bucket_count(n) + 1 + n * width) * (int64_t)sizeof(int32_t);
}

Buckets buckets_in(void* work, int64_t n) {
    Buckets b;
    b.n_buckets = (int32_t)bucket_count(n);
    b.count = reinterpret_cast<int32_t*>(work);
    b.cursor = b.count + b.n_buckets;
    b.start = b.cursor + b.n_buckets;
    b.edges = reinterpret_cast<uint32_t*>(b.start + b.n_buckets + 1);
    return b;
}

// Edges per workgroup: at least 2,048 on small tables, and on large ones as
// many as fit in LDS beside two words per bucket (each chunk pays up to one
// atomic per bucket, and longer runs per bucket store whole lines).
inline int32_t edge_chunk(int64_t count, int64_t n) {
    const int64_t most = bucket_count(n) <= 2048 ? 32768 : 22528;  // 128 + 16 KB, 88 + 64 KB
    return (int32_t)std::min<int64_t>(most, std::max<int64_t>(2048, cdiv(count, 512)));
}

// Converts and range-checks the table, and counts its valid edges per bucket.
template <typename I>
__global__ __launch_bounds__(kBucketThreads) void k_bucket_count(const I* nb, int64_t count, int64_t chunk, int64_t n,
                                                                 int32_t* out, Buckets b, int32_t* flags) {
    extern __shared__ int32_t hist[];
    for (int i = threadIdx.x; i < b.n_buckets; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    const int64_t end = min(count, ((int64_t)blockIdx.x + 1) * chunk);
    int wrong = 0;
    for (int64_t e = (int64_t)blockIdx.x * chunk + threadIdx.x; e < end; e += blockDim.x) {
        const int64_t v = (int64_t)nb[e];
        const bool bad = v < -1 || v >= n;
        out[e] = bad ? -1 : (int32_t)v;
        wrong += bad;
        if (!bad && v >= 0) atomicAdd(&hist[(int)v / kBucketRows], 1);
    }
    if (wrong) atomicAdd(&flags[0], wrong);
    __syncthreads();
    for (int i = threadIdx.x; i < b.n_buckets; i += blockDim.x)
        if (hist[i]) atomicAdd(&b.count[i], hist[i]);
}

// Exclusive prefix sums of the bucket counts (one workgroup).
__global__ __launch_bounds__(1024) void k_bucket_scan(Buckets b) {
    __shared__ int32_t part[1024];
    const int per = (b.n_buckets + 1023) / 1024, first = threadIdx.x * per;
    int32_t sum = 0;
    for (int i = first; i < min(first + per, b.n_buckets); ++i) sum += b.count[i];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int32_t add = (int)threadIdx.x >= o ? part[threadIdx.x - o] : 0;
        __syncthreads();
        part[threadIdx.x] += add;
        __syncthreads();
    }
    int32_t at = part[threadIdx.x] - sum;
    for (int i = first; i < min(first + per, b.n_buckets); ++i) {
        b.start[i] = b.cursor[i] = at;
        at += b.count[i];
    }
    if (threadIdx.x == 1023) b.start[b.n_buckets] = part[1023];
}

// Places each edge into its bucket's range.  The workgroup counts its chunk's
// edges per bucket, reserves their places with one atomic per bucket, groups
// the chunk by bucket in LDS, and writes each bucket's run with consecutive
// lanes: stored straight from the edge loop, the 4-byte stores of a random
// token order hit one cache line each (154 us against 73 us).
__global__ __launch_bounds__(kBucketThreads) void k_bucket_scatter(const int32_t* nb, int64_t count, int32_t chunk,
                                                                   int32_t width, Buckets b) {
    extern __shared__ int32_t place[];     // [n_buckets]: count, then end of the run in `group`
    int32_t* base = place + b.n_buckets;   // [n_buckets]: where the run goes in b.edges
    uint32_t* group = reinterpret_cast<uint32_t*>(base + b.n_buckets);  // [chunk]
    __shared__ int32_t part[kBucketThreads];
    for (int i = threadIdx.x; i < b.n_buckets; i += blockDim.x) place[i] = 0;
    __syncthreads();
    const int64_t begin = (int64_t)blockIdx.x * chunk, end = min(count, begin + chunk);
    for (int64_t e = begin + threadIdx.x; e < end; e += blockDim.x) {
        const int32_t v = nb[e];
        if (v >= 0) atomicAdd(&place[v / kBucketRows], 1);
    }
    __syncthreads();
    // Exclusive prefix sums over the buckets, kBucketThreads runs of them.
    const int per = (b.n_buckets + kBucketThreads - 1) / kBucketThreads;
    const int first = min((int)threadIdx.x * per, b.n_buckets), last = min(first + per, b.n_buckets);
    int32_t sum = 0;
    for (int i = first; i < last; ++i) {
        if (place[i]) base[i] = atomicAdd(&b.cursor[i], place[i]);
        sum += place[i];
    }
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < kBucketThreads; o <<= 1) {
        const int32_t add = (int)threadIdx.x >= o ? part[threadIdx.x - o] : 0;
        __syncthreads();
        part[threadIdx.x] += add;
        __syncthreads();
    }
    int32_t at = part[threadIdx.x] - sum;
    for (int i = first; i < last; ++i) {
        const int32_t c = place[i];
        place[i] = at;
        at += c;
    }
    __syncthreads();
    for (int64_t e = begin + threadIdx.x; e < end; e += blockDim.x) {
        const int32_t v = nb[e];
        if (v < 0) continue;
        const uint32_t source = (uint32_t)e / (uint32_t)width;  // count < 2^31
        group[atomicAdd(&place[v / kBucketRows], 1)] = (uint32_t)(v % kBucketRows) << 24 | source;
    }
    __syncthreads();
    // place[i] is now the end of bucket i's run and the start of bucket i + 1's.
    // A quarter wave writes a run: 16 lanes, 64 bytes.
    for (int i = threadIdx.x / 16; i < b.n_buckets; i += kBucketThreads / 16) {
        const int32_t from = i ? place[i - 1] : 0, to = place[i];
        for (int32_t j = from + (threadIdx.x & 15); j < to; j += 16) b.edges[base[i] + j - from] = group[j];
    }
}

// Largest in-degree -> flags[5].
__global__ __launch_bounds__(256) void k_bucket_degree(Buckets b, int32_t* flags) {
    __shared__ int32_t degree[kBucketRows];
    for (int i = threadIdx.x; i < kBucketRows; i += blockDim.x) degree[i] = 0;
    __syncthreads();
    const int32_t end = b.start[blockIdx.x + 1];
    for (int32_t e = b.start[blockIdx.x] + threadIdx.x; e < end; e += blockDim.x) atomicAdd(&degree[b.edges[e] >> 24], 1);
    __syncthreads();
    if (threadIdx.x < 64) {
        int most = 0;
        for (int i = threadIdx.x; i < kBucketRows; i += 64) most = max(most, degree[i]);
        most = wave_max_i(most);
        if (threadIdx.x == 0 && most) atomicMax(&flags[5], most);
    }
}

// The reverse rows of one bucket: slots taken by LDS atomics in any order, each
// row sorted in place, and the table written out as one run.  A slot past
// rwidth (the caller's bound was not the largest in-degree) is dropped.
template <int COLS>
__global__ __launch_bounds__(512) void k_bucket_reverse(Buckets b, int64_t n, int32_t* reverse, int32_t rwidth) {
    constexpr int R = COLS / 16;
    extern __shared__ int32_t table[];
    int32_t* cursor = table + kBucketRows * rwidth;
    for (int i = threadIdx.x; i < kBucketRows; i += blockDim.x) cursor[i] = 0;
    for (int i = threadIdx.x; i < kBucketRows * rwidth; i += blockDim.x) table[i] = INT_MAX;
    __syncthreads();
    const int32_t end = b.start[blockIdx.x + 1];
    for (int32_t e = b.start[blockIdx.x] + threadIdx.x; e < end; e += blockDim.x) {
        const uint32_t edge = b.edges[e], row = edge >> 24;
        const int32_t slot = atomicAdd(&cursor[row], 1);
        if (slot < rwidth) table[row * rwidth + slot] = (int32_t)(edge & 0xffffffu);
    }
    __syncthreads();
    const int e = threadIdx.x & 15;
    for (int row = threadIdx.x / 16; row < kBucketRows; row += blockDim.x / 16) {
        int32_t a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = e + 16 * r < rwidth ? table[row * rwidth + e + 16 * r] : INT_MAX;
        sort_rows<R>(a);
        wave_lds_sync();  // the row's lanes have all read it
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (R * e + r < rwidth) table[row * rwidth + R * e + r] = a[r] == INT_MAX ? -1 : a[r];
    }
    __syncthreads();
    const int64_t row0 = (int64_t)blockIdx.x * kBucketRows;
    const int count = (int)min((int64_t)kBucketRows, n - row0) * rwidth;
    for (int i = threadIdx.x; i < count; i += blockDim.x) reverse[row0 * rwidth + i] = table[i];
}

// ---------------------------------------------------------------- repack
__global__ void k_invert(const int64_t* perm, int64_t n, int64_t* inverse, int32_t* flags) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t v = perm[i];
    if (v < 0 || v >= n) {
        atomicAdd(&flags[0], 1);
        return;
    }
    unsigned long long prev = atomicCAS(reinterpret_cast<unsigned long long*>(inverse + v),
                                        (unsigned long long)(-1LL), (unsigned long long)i);
    if (prev != (unsigned long long)(-1LL)) atomicAdd(&flags[0], 1);
}

__device__ __forceinline__ int32_t relabel(int32_t old, const int64_t* inverse) {
    return old >= 0 ? (int32_t)inverse[old] : -1;
}

template <int COLS>
__global__ __launch_bounds__(256) void k_repack_rows(const int64_t* perm, int64_t n, const int32_t* nb, int32_t width,
                                                     const int64_t* inverse, int32_t* nb_out) {
    typedef RowLanes<COLS> R;
    const int lane = threadIdx.x & 63, k0 = lane % R::LANES;
    const int64_t step = (int64_t)gridDim.x * 4 * R::ROWS;
    for (int64_t i = ((int64_t)blockIdx.x * 4 + threadIdx.x / 64) * R::ROWS + lane / R::LANES; i < n; i += step) {
        const int64_t src = perm[i];
        const bool ok = src >= 0 && src < n;
#pragma unroll
        for (int r = 0; r < R::REGS; ++r) {
            const int k = k0 + 64 * r;
            if (k < width) nb_out[i * width + k] = ok ? relabel(nb[src * width + k], inverse) : -1;
        }
    }
}

__global__ void k_repack_tokens(const int64_t* perm, int64_t n, const int64_t* order, const int64_t* coords,
                                const int32_t* map, const int64_t* inverse, int64_t* order_out,
                                int64_t* coords_out, int32_t* map_out, int32_t* flags) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t src = perm[i];
    bool ok = src >= 0 && src < n;
    order_out[i] = ok ? order[src] : -1;
    for (int a = 0; a < 3; ++a) coords_out[3 * i + a] = ok ? coords[3 * src + a] : -1;
    if (map_out) {
        const int32_t to = (int32_t)inverse[map ? map[i] : i];
        map_out[i] = to;
        if (__ballot(to != (int32_t)i) && (threadIdx.x & 63) == 0) flags[1] = 1;  // every writer stores 1
    }
}

__global__ void k_relabel(const int32_t* in, int64_t count, const int64_t* inverse, int32_t* out) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < count) out[e] = relabel(in[e], inverse);
}

__global__ void k_check_layout(LayoutDims d, const int64_t* order, const int64_t* coords,
                               int32_t* seen, int32_t* flags) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    int64_t t = order[i];
    if (t < 0 || t >= d.n) {
        atomicAdd(&flags[0], 1);
        return;
    }
    if (atomicAdd(&seen[t], 1) != 0) atomicAdd(&flags[0], 1);
    int64_t x = t % d.g[2], y = (t / d.g[2]) % d.g[1], z = t / (d.g[2] * d.g[1]);
    if (coords[3 * i] != z || coords[3 * i + 1] != y || coords[3 * i + 2] != x) atomicAdd(&flags[0], 1);
}

// ------------------------------------------------------ stencil match
// raster index -> packed row from a layout's order (order[i] = raster index of
// row i; map starts at -1); entries outside [0, n) and raster indices that
// appear twice (order is then no permutation, and some raster index is left
// without a row) are counted in flags[0].
__global__ void k_scatter_order(const int64_t* order, int64_t n, int32_t* map, int32_t* flags) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t t = order[i];
    if (t < 0 || t >= n) {
        atomicAdd(&flags[0], 1);
        return;
    }
    if (atomicExch(&map[t], (int32_t)i) != -1) atomicAdd(&flags[0], 1);
}

// Counts in flags[1] the entries of nb [N, W] that differ from the complete
// product-order stencil of radius d.r on grid d.g, evaluated at each row's
// raster coordinate (the table build_layout makes, geometry.py:253-259).
__global__ void k_compare_stencil(LayoutDims d, int64_t width, const int64_t* order, const int32_t* map,
                                  const int32_t* nb, int32_t* flags) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= d.n * width) return;
    int64_t i = e / width;
    int64_t k = e - i * width;
    int64_t t = order[i];
    if (t < 0 || t >= d.n) return;  // counted by k_scatter_order
    int64_t c[3] = {t / (d.g[2] * d.g[1]), (t / d.g[2]) % d.g[1], t % d.g[2]};
    int64_t wy = 2 * d.r[1] + 1, wx = 2 * d.r[2] + 1;
    int64_t off[3] = {k / (wy * wx) - d.r[0], (k / wx) % wy - d.r[1], k % wx - d.r[2]};
    int64_t raster = 0;
    bool inside = true;
    for (int a = 0; a < 3; ++a) {
        int64_t v = c[a] + off[a];
        inside = inside && v >= 0 && v < d.g[a];
        raster = raster * d.g[a] + (inside ? v : 0);
    }
    int32_t expect = inside ? map[raster] : -1;
    if (nb[e] != expect) atomicAdd(&flags[1], 1);
}

void reverse_rows(const int32_t* rows, int64_t n, int32_t width, const int64_t* perm, const int64_t* inverse,
                  int32_t* reverse, int32_t rwidth, hipStream_t s) {
    with_columns(std::max(width, rwidth), [&](auto c) {
        k_reverse_rows<decltype(c)::value><<<sort_blocks(n), 256, 0, s>>>(rows, n, width, perm, inverse, reverse, rwidth);
    });
}

void check_rows_and_cover(const int32_t* nb, int64_t n, int32_t width, const int32_t* blocks, int64_t fine,
                          int32_t slots, int32_t pool_size, const int32_t* degree, const int32_t* cover, int32_t* flags,
                          hipStream_t s) {
    with_columns(width, [&](auto c) {
        k_check_duplicates<decltype(c)::value><<<sort_blocks(n), 256, 0, s>>>(nb, n, width, flags);
    });
    k_check_cover<<<grid1d(n), kThreads, 0, s>>>(cover, degree, n, flags);
    const int64_t groups = cdiv(fine, pool_size);
    k_check_groups<<<grid1d(groups), kThreads, 0, s>>>(blocks, fine, slots, pool_size, groups, flags);
}

}  // namespace
}  // namespace p3d

using namespace p3d;

extern "C" int p3d_build_layout(const int64_t grid[3], const int64_t block[3], const int64_t radius[3],
                                int32_t morton, int64_t* order, int64_t* coords,
                                int32_t* raster_to_packed, int32_t* neighbors, int32_t* blocks,
                                void* stream) {
    LayoutDims d{};
    d.n = 1;
    d.volume = 1;
    int64_t width = 1;
    for (int a = 0; a < 3; ++a) {
        P3D_REQUIRE(grid[a] >= 1 && block[a] >= 1 && radius[a] >= 0, "invalid grid, block or radius");
        P3D_REQUIRE(grid[a] % block[a] == 0, "grid must be divisible by block_shape");
        d.g[a] = grid[a];
        d.blk[a] = block[a];
        d.r[a] = radius[a];
        d.n *= grid[a];
        d.volume *= block[a];
        width *= 2 * radius[a] + 1;
    }
    P3D_REQUIRE(d.volume <= 64 && width <= 128, "layout exceeds supported block or neighborhood width");
    P3D_REQUIRE(d.n * width < ((int64_t)1 << 31), "geometry exceeds the 32-bit kernel indexing limit");
    P3D_REQUIRE(order && coords && neighbors && blocks, "null output");
    P3D_REQUIRE(!morton || raster_to_packed, "morton layouts need the raster->packed map");
    d.morton = morton != 0;
    for (int a = 0; a < 3; ++a)
        while (std::max(grid[a] / block[a], block[a]) > (int64_t)1 << d.nbits) ++d.nbits;
    hipStream_t s = as_stream(stream);
    k_layout_map<<<grid1d(d.n), kThreads, 0, s>>>(d, order, coords, raster_to_packed);
    with_columns((int)width, [&](auto c) {
        k_layout_neighbors<decltype(c)::value><<<row_blocks<decltype(c)::value>(d.n), 256, 0, s>>>(
            d, (int32_t)width, coords, morton ? raster_to_packed : nullptr, neighbors);
    });
    k_iota_i32<<<grid1d(d.n), kThreads, 0, s>>>(blocks, d.n);
    return check_launch("p3d_build_layout");
}

extern "C" int p3d_geometry_check(const void* neighbors, int32_t nb_is64, int64_t n, int32_t width,
                                  const void* blocks, int32_t blocks_is64, int64_t fine, int32_t slots,
                                  int32_t pool_size, int32_t* neighbors32, int32_t* blocks32,
                                  int32_t* degree, int32_t* cover, int32_t* flags, void* stream) {
    P3D_REQUIRE(n >= 1 && width >= 1 && width <= 128 && fine >= 1 && slots >= 1 && slots <= 64,
                "invalid geometry shape");
    P3D_REQUIRE(pool_size >= 1 && pool_size <= 32, "pool_size must be an integer in [1,32]");
    hipStream_t s = as_stream(stream);
    k_fill_i32<<<1, 64, 0, s>>>(flags, 8, 0);
    k_fill_i32<<<grid1d(n), kThreads, 0, s>>>(degree, n, 0);
    k_fill_i32<<<grid1d(n), kThreads, 0, s>>>(cover, n, 0);
    int64_t cnb = n * width, cbl = fine * slots;
    if (nb_is64)
        k_check_neighbors<<<grid1d(cnb), kThreads, 0, s>>>((const int64_t*)neighbors, cnb, n, neighbors32, degree, flags);
    else
        k_check_neighbors<<<grid1d(cnb), kThreads, 0, s>>>((const int32_t*)neighbors, cnb, n, neighbors32, degree, flags);
    if (blocks_is64)
        k_check_blocks<<<grid1d(cbl), kThreads, 0, s>>>((const int64_t*)blocks, cbl, n, blocks32, cover, flags);
    else
        k_check_blocks<<<grid1d(cbl), kThreads, 0, s>>>((const int32_t*)blocks, cbl, n, blocks32, cover, flags);
    check_rows_and_cover(neighbors32, n, width, blocks32, fine, slots, pool_size, degree, cover, flags, s);
    return check_launch("p3d_geometry_check");
}

extern "C" int p3d_bucket_bytes(int64_t n, int32_t width, int64_t* bytes) {
    P3D_REQUIRE(bytes, "null output");
    *bytes = bucket_bytes(n, width);
    return P3D_OK;
}

extern "C" int p3d_geometry_check_bucketed(const void* neighbors, int32_t nb_is64, int64_t n, int32_t width,
                                           const void* blocks, int32_t blocks_is64, int64_t fine, int32_t slots,
                                           int32_t pool_size, int32_t* neighbors32, int32_t* blocks32,
                                           int32_t* cover, void* work, int32_t* flags, void* stream) {
    P3D_REQUIRE(bucket_bytes(n, width) > 0 && fine >= 1 && slots >= 1 && slots <= 64, "invalid geometry shape");
    P3D_REQUIRE(pool_size >= 1 && pool_size <= 32, "pool_size must be an integer in [1,32]");
    P3D_REQUIRE(neighbors && blocks && neighbors32 && blocks32 && cover && work && flags, "null argument");
    hipStream_t s = as_stream(stream);
    const Buckets b = buckets_in(work, n);
    const int64_t cnb = n * width, cbl = fine * slots, chunk = edge_chunk(cnb, n);
    const unsigned chunks = (unsigned)cdiv(cnb, chunk);
    const size_t lds = (size_t)b.n_buckets * sizeof(int32_t);
    k_fill_i32<<<1, 64, 0, s>>>(flags, 8, 0);
    k_fill_i32<<<grid1d(n), kThreads, 0, s>>>(cover, n, 0);
    k_fill_i32<<<grid1d(b.n_buckets), kThreads, 0, s>>>(b.count, b.n_buckets, 0);
    if (nb_is64)
        k_bucket_count<<<chunks, kBucketThreads, lds, s>>>((const int64_t*)neighbors, cnb, chunk, n, neighbors32, b, flags);
    else
        k_bucket_count<<<chunks, kBucketThreads, lds, s>>>((const int32_t*)neighbors, cnb, chunk, n, neighbors32, b, flags);
    if (blocks_is64)
        k_check_blocks<<<grid1d(cbl), kThreads, 0, s>>>((const int64_t*)blocks, cbl, n, blocks32, cover, flags);
    else
        k_check_blocks<<<grid1d(cbl), kThreads, 0, s>>>((const int32_t*)blocks, cbl, n, blocks32, cover, flags);
    k_bucket_scan<<<1, 1024, 0, s>>>(b);
    k_bucket_scatter<<<chunks, kBucketThreads, 2 * lds + (size_t)chunk * 4, s>>>(neighbors32, cnb, (int32_t)chunk, width, b);
    k_bucket_degree<<<b.n_buckets, 256, 0, s>>>(b, flags);
    check_rows_and_cover(neighbors32, n, width, blocks32, fine, slots, pool_size, nullptr, cover, flags, s);
    return check_launch("p3d_geometry_check_bucketed");
}

extern "C" int p3d_reverse_bucketed(void* work, int64_t n, int32_t width, int32_t* reverse, int32_t rwidth,
                                    void* stream) {
    P3D_REQUIRE(bucket_bytes(n, width) > 0 && rwidth >= 1 && rwidth <= 128, "invalid reverse adjacency shape");
    P3D_REQUIRE(work && reverse, "null argument");
    const Buckets b = buckets_in(work, n);
    const size_t lds = (size_t)kBucketRows * (rwidth + 1) * sizeof(int32_t);
    with_columns(rwidth, [&](auto c) {
        k_bucket_reverse<decltype(c)::value><<<b.n_buckets, 512, lds, as_stream(stream)>>>(b, n, reverse, rwidth);
    });
    return check_launch("p3d_reverse_bucketed");
}

extern "C" int p3d_reverse_rows(const int32_t* rows, int64_t n, int32_t width, const int64_t* perm,
                                const int64_t* inverse, int32_t* reverse, int32_t rwidth, void* stream) {
    P3D_REQUIRE(n >= 1 && width >= 1 && width <= 128 && rwidth >= 1 && rwidth <= 128, "invalid reverse adjacency shape");
    P3D_REQUIRE(rows && reverse, "null argument");
    reverse_rows(rows, n, width, perm, inverse, reverse, rwidth, as_stream(stream));
    return check_launch("p3d_reverse_rows");
}

extern "C" int p3d_reverse_adjacency(const int32_t* neighbors, int64_t n, int32_t width, int32_t* cursor,
                                     int32_t* reverse, int32_t rwidth, void* stream) {
    P3D_REQUIRE(n >= 1 && width >= 1 && rwidth >= 1 && rwidth <= 128, "invalid reverse adjacency shape");
    hipStream_t s = as_stream(stream);
    k_fill_i32<<<grid1d(n), kThreads, 0, s>>>(cursor, n, 0);
    k_fill_i32<<<grid1d(n * rwidth), kThreads, 0, s>>>(reverse, n * rwidth, -1);
    k_reverse_scatter<<<grid1d(n * width), kThreads, 0, s>>>(neighbors, n * width, width, cursor, reverse, rwidth);
    reverse_rows(reverse, n, rwidth, nullptr, nullptr, reverse, rwidth, s);
    return check_launch("p3d_reverse_adjacency");
}

extern "C" int p3d_repack(const int64_t* perm, int64_t n, const int32_t* neighbors, int32_t width,
                          const int32_t* blocks, int64_t fine, int32_t slots, const int64_t* order,
                          const int64_t* coords, const int32_t* raster_map, int64_t* inverse,
                          int32_t* neighbors_out, int32_t* blocks_out, int64_t* order_out,
                          int64_t* coords_out, int32_t* raster_map_out, int32_t* flags, void* stream) {
    P3D_REQUIRE(n >= 1 && width >= 1 && width <= 128 && fine >= 1 && slots >= 1, "invalid repack shape");
    hipStream_t s = as_stream(stream);
    k_fill_i32<<<1, 64, 0, s>>>(flags, 8, 0);
    k_fill_i64<<<grid1d(n), kThreads, 0, s>>>(inverse, n, -1);
    k_invert<<<grid1d(n), kThreads, 0, s>>>(perm, n, inverse, flags);
    // A rejected permutation leaves some inverse entries at -1; clamp them so
    // the gathers below stay in bounds (the caller raises on flags[0]).
    with_columns(width, [&](auto c) {
        k_repack_rows<decltype(c)::value><<<row_blocks<decltype(c)::value>(n), 256, 0, s>>>(perm, n, neighbors, width,
                                                                                         inverse, neighbors_out);
    });
    k_relabel<<<grid1d(fine * slots), kThreads, 0, s>>>(blocks, fine * slots, inverse, blocks_out);
    k_repack_tokens<<<grid1d(n), kThreads, 0, s>>>(perm, n, order, coords, raster_map, inverse, order_out,
                                                  coords_out, raster_map_out, flags);
    return check_launch("p3d_repack");
}

extern "C" int p3d_check_layout(const int64_t grid[3], const int64_t* order, const int64_t* coords,
                                int32_t* scratch, int32_t* flags, void* stream) {
    LayoutDims d{};
    d.n = grid[0] * grid[1] * grid[2];
    for (int a = 0; a < 3; ++a) d.g[a] = grid[a];
    P3D_REQUIRE(d.n >= 1, "empty grid");
    hipStream_t s = as_stream(stream);
    k_fill_i32<<<1, 64, 0, s>>>(flags, 8, 0);
    k_fill_i32<<<grid1d(d.n), kThreads, 0, s>>>(scratch, d.n, 0);
    k_check_layout<<<grid1d(d.n), kThreads, 0, s>>>(d, order, coords, scratch, flags);
    return check_launch("p3d_check_layout");
}

extern "C" int p3d_stencil_match(const int64_t grid[3], const int64_t radius[3], const int64_t* order,
                                 const int32_t* neighbors, int32_t width, int32_t* raster_to_packed,
                                 int32_t* flags, void* stream) {
    LayoutDims d{};
    d.n = 1;
    int64_t w = 1;
    for (int a = 0; a < 3; ++a) {
        P3D_REQUIRE(grid[a] >= 1 && radius[a] >= 0, "invalid grid or radius");
        d.g[a] = grid[a];
        d.r[a] = radius[a];
        d.n *= grid[a];
        w *= 2 * radius[a] + 1;
    }
    P3D_REQUIRE(w == width, "neighbour width does not match the stencil radius");
    P3D_REQUIRE(d.n * w < ((int64_t)1 << 31), "geometry exceeds the 32-bit kernel indexing limit");
    P3D_REQUIRE(order && neighbors && raster_to_packed && flags, "null argument");
    hipStream_t s = as_stream(stream);
    k_fill_i32<<<1, 64, 0, s>>>(flags, 8, 0);
    k_fill_i32<<<grid1d(d.n), kThreads, 0, s>>>(raster_to_packed, d.n, -1);
    k_scatter_order<<<grid1d(d.n), kThreads, 0, s>>>(order, d.n, raster_to_packed, flags);
    k_compare_stencil<<<grid1d(d.n * w), kThreads, 0, s>>>(d, w, order, raster_to_packed, neighbors, flags);
    return check_launch("p3d_stencil_match");
}
