// Weight gradients of the PACK3D layer's linear maps (to_q, to_kv, gate and
// to_out of attention.py:64-67,85,89 of amilworks/Pack3D): for y = x W^T,
// dW[o][i] = sum over tokens n of dy[n][o] x[n][i], accumulated in fp32.
// The contraction runs over all tokens (262,144 at 64^3) while W is small
// (at most a few hundred rows), so the tokens are split across workgroups
// and each writes an fp32 partial; a second kernel sums the partials in a
// fixed order (deterministic).
//
// A workgroup owns 256 output rows (8 waves x 32) and a token range, taken 32
// tokens per stage (16 in fp32).  The pass is bound by the bytes in flight per
// CU, so the stages of dy [tokens x 256 rows] and of x [tokens x I] are copied to
// LDS by DMA, two stages ahead of the one that is multiplied: through registers,
// a stage at a time, 262,144 tokens took 253 us for 968 x 192 and 64 us for
// 192 x 192, now 153 and 46 us (32,768 tokens of 1,040 x 512: 90 -> 65 us).
// Three and four buffers of 32 tokens and two of 64 are alike.  The MFMA
// operands need 8 consecutive tokens of one column per lane; they come out of the
// row-major tiles through ds_read_b64_tr_b16, two 8-byte transposed reads per
// fragment, so nothing is transposed on the way in.
// Each wave then multiplies its 32 x 16-token A fragment with the I / 32
// shared x fragments: D = dy^T x, 32 rows by I columns per wave.
//
// In fp32 the operands (two tokens of one column per 64 lanes) are plain reads of
// two tile rows, and the pass is bound by the MFMA: 18,711 tokens of to_q, to_kv
// and the gate at width 192 take 89 us and to_out 51 us, where the library's four
// products, on a few dozen workgroups, took 403 us.
#include "attn_common.hpp"

namespace p3d {
namespace {

constexpr int kWgWaves = 8;
constexpr int kWgThreads = 64 * kWgWaves;
constexpr int kWgRows = 32 * kWgWaves;  // output rows per workgroup
constexpr int kWgTokMax = 64;           // splits are multiples of this many tokens
constexpr int kWgMaxCols = 256;         // input columns per workgroup

// Tiles of one stage in LDS: TOK rows of 256 dy columns, then TOK rows of x's
// columns rounded up to 128 or 256, in 16-byte pieces without padding (the DMA
// writes 64 pieces of a wave in a row).  Piece c of row r lies at c ^ swizzle(r),
// so that the rows a fragment reads together start in different banks: four rows
// of 64 bytes (16-bit types), two of 128 (fp32).
template <typename T, int IT>
struct WgCfg {
    static constexpr int EP = Piece<T>::N;
    static constexpr int TOK = sizeof(T) == 2 ? 32 : 16;
    static constexpr int BUFS = 3;
    static constexpr int AP = kWgRows / EP;                // pieces of a dy row
    static constexpr int XP = (IT <= 4 ? 128 : 256) / EP;  // and of an x row
    static constexpr int NA = TOK * AP / kWgThreads, NX = TOK * XP / kWgThreads;  // copies per thread
    static constexpr int STAGE = TOK * (AP + XP) * 16;     // bytes
    static_assert(NA * kWgThreads == TOK * AP && NX * kWgThreads == TOK * XP, "a stage is whole copies");
};
template <typename T>
__device__ __forceinline__ int wg_swizzle(int row) { return sizeof(T) == 2 ? 4 * (row & 3) : 8 * (row & 1); }

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));

// MFMA operand fragment (32x32x16 layout: lane L holds index L % 32 of the
// M or N dimension and contraction indices 8 (L / 32) .. + 8) from a
// row-major LDS tile whose rows are the contraction index (tokens): rows
// k0 + 8 (L / 32) + t, column c0 + L % 32.  ds_read_b64_tr_b16 hands lane
// B + 4a + e of each 16-lane block element e of the 8-byte windows addressed
// by lanes B + a + 4j (j = 0..3) as its values j, so lane L addresses row
// k0 + 8 (L / 32) + (L % 16) / 4 (four rows further for the second read) at
// column c0 + 16 ((L / 16) % 2) + 4 (L % 4).  pieces: of a tile row.
template <typename T>
__device__ __forceinline__ typename Mma<T>::Frag frag_tr(const T* tile, int pieces, int k0, int c0, int lane) {
    const int row = k0 + 8 * (lane >> 5) + ((lane & 15) >> 2);
    const int col = c0 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    const T* p = tile + (row * pieces + ((col / 8) ^ wg_swizzle<T>(row))) * 8 + col % 8;
    typedef __attribute__((address_space(3))) v4s* lds_v4s;
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)p);
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(p + 4 * pieces * 8));  // same swizzle
    const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(typename Mma<T>::Frag, v);
}

template <>
__device__ __forceinline__ float frag_tr<float>(const float* tile, int pieces, int k0, int c0, int lane) {
    const int row = k0 + (lane >> 5), col = c0 + (lane & 31);
    return tile[(row * pieces + ((col / 4) ^ wg_swizzle<float>(row))) * 4 + col % 4];
}

// dy as up to three column blocks of output rows: rows [0, end[0]) from
// src[0], [end[0], end[1]) from src[1], [end[1], O) from src[2], each with its
// own row stride (a single dy has end[0] = end[1] = O).
template <typename T>
struct WgSrc {
    const T* src[3];
    int64_t ld[3];
    int end[2];
};

// The tiles of dW (row blocks x column blocks) of each token range.  by_xcd:
// workgroups go to the eight XCDs in turn, so the tiles of a range, which read
// the same rows of dy and x, take ids 8 apart and share one XCD's L2 (ids past
// the last range leave at once).  32,768 rows of 1,040 x 512 (10 tiles): 71 us
// spread over the XCDs, 65 us so; 262,144 of 968 x 192 (4 tiles): 160 and 153
// us.  Fewer than 8 ranges would leave XCDs idle and keep the tiles spread.
struct WgGrid {
    int row_blocks, col_blocks, splits;
    bool by_xcd;
};

// Partial dW of token range [split * per, + per) for output rows [ob, ob + rpb)
// (rpb a multiple of 32, at most 256: the rows are spread evenly over the row
// blocks, so that a last block of a few rows does not cost a whole workgroup's
// pass) and input columns [cb * I, + I) of I_total, written to
// part[split][o][cb * I + i].
// BUFS stages of dynamic LDS.
template <typename T, int IT>
__global__ __launch_bounds__(kWgThreads) void k_wgrad(WgSrc<T> dy, const T* x, int64_t ldx, float* part, int64_t rows,
                                                      int O, int rpb, int64_t per, int I_total, WgGrid wg) {
    typedef Mma<T> M;
    typedef WgCfg<T, IT> C;
    constexpr int I = 32 * IT, EP = C::EP, NP = C::NA + C::NX;
    extern __shared__ __align__(16) unsigned char wg_smem[];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = wg.row_blocks * wg.col_blocks, id = blockIdx.x;
    const int split = wg.by_xcd ? id / 8 / tiles * 8 + id % 8 : id / tiles;
    const int tile = wg.by_xcd ? id / 8 % tiles : id % tiles;
    if (split >= wg.splits) return;  // the whole workgroup
    const int cb = tile / wg.row_blocks, ob = (tile - cb * wg.row_blocks) * rpb;
    const int64_t n0 = (int64_t)split * per, n1 = min(rows, n0 + per);
    x += (int64_t)cb * I;  // this workgroup's input columns
    const bool active = 32 * wave < rpb && ob + 32 * wave < O;  // wave-uniform

    // This thread's pieces of a stage: p-th copy's row, and its source in the
    // stage to come next (columns past the block's or x's last are read from it:
    // they only reach output rows and columns that are not stored).
    int prow[NP];
    const unsigned char* src[NP];
    int64_t step[NP];  // bytes per stage
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const bool isx = i >= C::NA;
        const int L = tid + (isx ? i - C::NA : i) * kWgThreads, pieces = isx ? C::XP : C::AP;
        prow[i] = L / pieces;
        const int c = ((L % pieces) ^ wg_swizzle<T>(prow[i])) * EP;
        if (isx) {
            src[i] = reinterpret_cast<const unsigned char*>(x + (n0 + prow[i]) * ldx + min(c, I - EP));
            step[i] = C::TOK * ldx * (int64_t)sizeof(T);
        } else {
            const int o = ob + min(c, min(rpb, O - ob) - EP);  // a piece of one source (the blocks are multiples of 8)
            const int sel = o < dy.end[0] ? 0 : (o < dy.end[1] ? 1 : 2);
            const int o_src = o - (sel == 0 ? 0 : dy.end[sel - 1]);
            src[i] = reinterpret_cast<const unsigned char*>(dy.src[sel] + (n0 + prow[i]) * dy.ld[sel] + o_src);
            step[i] = C::TOK * dy.ld[sel] * (int64_t)sizeof(T);
        }
    }
    // Copies stage t0 .. t0 + TOK - 1 into buffer buf: by LDS DMA, or through
    // registers with zeros past n1 where it is the range's partial last one.
    auto issue = [&](int64_t t0, int buf) __attribute__((always_inline)) {
        if (t0 >= n1) return;
        if (t0 + C::TOK <= n1) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                dma_copy16(src[i], lds_address(wg_smem) + buf * C::STAGE + (i * kWgThreads + wave * 64) * 16);
                src[i] += step[i];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            u32x4 v{0, 0, 0, 0};
            if (t0 + prow[i] < n1) v = *reinterpret_cast<const u32x4*>(src[i]);
            *reinterpret_cast<u32x4*>(wg_smem + buf * C::STAGE + (i * kWgThreads + tid) * 16) = v;
        }
    };

    f32x16 acc[IT];
#pragma unroll
    for (int t = 0; t < IT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    constexpr int AHEAD = C::BUFS - 1;  // stages being copied while one is multiplied
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) issue(n0 + i * C::TOK, i);
    int buf = 0;
    for (int64_t t0 = n0; t0 < n1; t0 += C::TOK) {
        // This wave's copies of the stage have landed (those of the stages after
        // it are still counted if all of them are whole), and after the barrier
        // every wave's; every wave is also done with the stage before, whose buffer
        // is copied into next.
        if (t0 + AHEAD * C::TOK <= n1)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((AHEAD - 1) * NP) : "memory");
        else
            dma_wait();
        __syncthreads();
        issue(t0 + AHEAD * C::TOK, (buf + AHEAD) % C::BUFS);
        const T* cur = reinterpret_cast<const T*>(wg_smem + buf * C::STAGE);
        // Waves past the block's last output row multiply columns of the dy tile
        // that are not stored: no branch around the MFMAs, whose accumulators would
        // otherwise be copied between register files at the join.
#pragma unroll
        for (int ks = 0; ks < C::TOK / M::KS; ++ks) {
            const typename M::Frag fa = frag_tr<T>(cur, C::AP, M::KS * ks, 32 * wave, lane);
#pragma unroll
            for (int t = 0; t < IT; ++t)
                acc[t] = M::mfma(fa, frag_tr<T>(cur + C::TOK * C::AP * EP, C::XP, M::KS * ks, 32 * t, lane), acc[t]);
        }
        buf = (buf + 1) % C::BUFS;
    }
    if (!active) return;
    // D row acc_row(r, g) is output row ob + 32 wave + that; column lane % 32 of tile t is input 32 t + lane % 32.
    float* out = part + (int64_t)split * O * I_total + (int64_t)cb * I;
#pragma unroll
    for (int t = 0; t < IT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int o = ob + 32 * wave + acc_row(r, g);
            if (o < O) out[(int64_t)o * I_total + 32 * t + (lane & 31)] = acc[t][r];
        }
}

// dw[e] = sum over splits of part[s][e] in a fixed order (deterministic),
// rounded once to dw's type: thread group j of a block (64 elements x G
// groups) sums splits j, j + G, ... in increasing order, eight loads issued
// together, then the groups are added pairwise.  16 groups where there are
// more than 64 splits (256 of a 192 x 192 gradient, 38 MB: 18 us with 4 groups
// and one load at a time, 9 us), else 4, whose threads all have work (25 of a
// 1,040 x 512 gradient, 53 MB: 9 us against 24 us with 16 groups).
constexpr int kRedElems = 64;
template <typename TO, int G>
__global__ __launch_bounds__(kRedElems * G) void k_wgrad_reduce(const float* part, TO* dw, int64_t count, int splits) {
    __shared__ float sums[G][kRedElems];
    const int le = threadIdx.x % kRedElems, grp = threadIdx.x / kRedElems;
    const int64_t e = (int64_t)blockIdx.x * kRedElems + le;
    float s = 0.f;
    if (e < count)
        for (int k = grp; k < splits; k += 8 * G) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = part[(int64_t)min(k + i * G, splits - 1) * count + e];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k + i * G < splits) s += v[i];
        }
    sums[grp][le] = s;
    __syncthreads();
#pragma unroll
    for (int h = G / 2; h >= 1; h /= 2) {
        if (grp < h) sums[grp][le] += sums[grp + h][le];
        __syncthreads();
    }
    if (grp == 0 && e < count) dw[e] = from_f32<TO>(sums[0][le]);
}

template <typename TO>
void launch_reduce(const float* part, TO* dw, int64_t count, int splits, hipStream_t s) {
    const unsigned blocks = (unsigned)cdiv(count, kRedElems);
    if (splits > 64)
        k_wgrad_reduce<TO, 16><<<blocks, kRedElems * 16, 0, s>>>(part, dw, count, splits);
    else
        k_wgrad_reduce<TO, 4><<<blocks, kRedElems * 4, 0, s>>>(part, dw, count, splits);
}

// Input widths the kernel takes: a multiple of 32 up to 256 (one column
// block), or a multiple of 256 up to 2048 (column blocks of 256).
inline bool wgrad_cols_ok(int I) {
    return (I >= 32 && I % 32 == 0 && I <= kWgMaxCols) || (I > kWgMaxCols && I % kWgMaxCols == 0 && I <= 2048);
}

template <typename T>
int launch_wgrad(const WgSrc<T>& dy, const void* x, int64_t ldx, void* dw, int dw_dtype, float* part, int64_t rows,
                 int O, int I, int splits, hipStream_t s) {
    const int64_t per = cdiv(cdiv(rows, splits), kWgTokMax) * kWgTokMax;
    const int used = (int)cdiv(rows, per);
    // Past 256 input columns the columns go to blocks of 256, each
    // with its own accumulators; dy is read once per block.
    const int cbs = I > kWgMaxCols ? I / kWgMaxCols : 1, Ib = I / cbs;
    const int nrb = (int)cdiv(O, kWgRows), rpb = 32 * (int)cdiv(cdiv(O, nrb), 32);
    const WgGrid wg{nrb, cbs, used, nrb * cbs > 1 && used >= 8};
    const unsigned grid = (unsigned)(nrb * cbs * (wg.by_xcd ? cdiv(used, 8) * 8 : used));
    switch (Ib / 32) {
#define CASE(IT)                                                                                                  \
    case IT:                                                                                                      \
        k_wgrad<T, IT><<<grid, kWgThreads, WgCfg<T, IT>::BUFS * WgCfg<T, IT>::STAGE, s>>>(                       \
            dy, (const T*)x, ldx, part, rows, O, rpb, per, I, wg);                                                       \
        break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
        default: return fail(P3D_EUNSUPPORTED, "in_features must be a multiple of 32, at most 256");
    }
    const int64_t count = (int64_t)O * I;
    if (dw_dtype == P3D_F32)
        launch_reduce(part, (float*)dw, count, used, s);
    else  // the inputs' own type
        launch_reduce(part, (T*)dw, count, used, s);
    return check_launch("p3d_weight_grad");
}

}  // namespace
}  // namespace p3d

using namespace p3d;

extern "C" int p3d_weight_grad(const void* dy, int64_t ldy, const void* x, int64_t ldx, float* dw, float* workspace,
                               int64_t rows, int32_t out_features, int32_t in_features, int32_t splits, int32_t dtype,
                               void* stream) {
    P3D_REQUIRE(dy && x && dw && workspace, "null pointer argument");
    P3D_REQUIRE(dtype >= P3D_F32 && dtype <= P3D_BF16, "unknown dtype");
    P3D_REQUIRE(rows >= 1 && splits >= 1, "need at least one row and one split");
    P3D_REQUIRE(out_features >= 8 && out_features % 8 == 0, "out_features must be a positive multiple of 8");
    P3D_REQUIRE(wgrad_cols_ok(in_features),
                "in_features must be a multiple of 32 up to 256, or a multiple of 256 up to 2048");
    P3D_REQUIRE(ldy >= out_features && ldy % 8 == 0 && ldx >= in_features && ldx % 8 == 0,
                "row strides must cover the rows and keep 16-byte alignment");
    P3D_REQUIRE(aligned16(dy) && aligned16(x), "dy and x must be 16-byte aligned");
    P3D_REQUIRE(cdiv(out_features, kWgRows) < 65536 && splits < 65536, "grid too large");
    if (dtype == P3D_F32) {
        const WgSrc<float> src{{(const float*)dy, nullptr, nullptr}, {ldy, 0, 0}, {out_features, out_features}};
        return launch_wgrad<float>(src, x, ldx, dw, P3D_F32, workspace, rows, out_features, in_features, splits,
                                   as_stream(stream));
    }
    if (dtype == P3D_F16) {
        const WgSrc<_Float16> src{{(const _Float16*)dy, nullptr, nullptr}, {ldy, 0, 0}, {out_features, out_features}};
        return launch_wgrad<_Float16>(src, x, ldx, dw, P3D_F32, workspace, rows, out_features, in_features, splits,
                                      as_stream(stream));
    }
    const WgSrc<__bf16> src{{(const __bf16*)dy, nullptr, nullptr}, {ldy, 0, 0}, {out_features, out_features}};
    return launch_wgrad<__bf16>(src, x, ldx, dw, P3D_F32, workspace, rows, out_features, in_features, splits,
                                as_stream(stream));
}

extern "C" int p3d_weight_grad3(const void* dy0, int64_t ld0, int32_t out0, const void* dy1, int64_t ld1,
                                int32_t out1, const void* dy2, int64_t ld2, int32_t out2, const void* x, int64_t ldx,
                                void* dw, int32_t dw_dtype, float* workspace, int64_t rows, int32_t in_features,
                                int32_t splits, int32_t dtype, void* stream) {
    P3D_REQUIRE(dy0 && dy1 && dy2 && x && dw && workspace, "null pointer argument");
    P3D_REQUIRE(dtype >= P3D_F32 && dtype <= P3D_BF16, "unknown dtype");
    P3D_REQUIRE(dw_dtype == P3D_F32 || dw_dtype == dtype, "dw is fp32 or of the inputs' type");
    P3D_REQUIRE(rows >= 1 && splits >= 1, "need at least one row and one split");
    P3D_REQUIRE(out0 >= 8 && out1 >= 8 && out2 >= 8 && out0 % 8 == 0 && out1 % 8 == 0 && out2 % 8 == 0 &&
                    (int64_t)out0 + out1 + out2 < (1 << 24),
                "out features must be positive multiples of 8");
    P3D_REQUIRE(wgrad_cols_ok(in_features),
                "in_features must be a multiple of 32 up to 256, or a multiple of 256 up to 2048");
    P3D_REQUIRE(ld0 >= out0 && ld1 >= out1 && ld2 >= out2 && ld0 % 8 == 0 && ld1 % 8 == 0 && ld2 % 8 == 0 &&
                    ldx >= in_features && ldx % 8 == 0,
                "row strides must cover the rows and keep 16-byte alignment");
    P3D_REQUIRE(aligned16(dy0) && aligned16(dy1) && aligned16(dy2) && aligned16(x), "dy and x must be 16-byte aligned");
    const int O = out0 + out1 + out2;
    P3D_REQUIRE(cdiv(O, kWgRows) < 65536 && splits < 65536, "grid too large");
    if (dtype == P3D_F32) {
        const WgSrc<float> src{{(const float*)dy0, (const float*)dy1, (const float*)dy2}, {ld0, ld1, ld2},
                               {out0, out0 + out1}};
        return launch_wgrad<float>(src, x, ldx, dw, dw_dtype, workspace, rows, O, in_features, splits,
                                   as_stream(stream));
    }
    if (dtype == P3D_F16) {
        const WgSrc<_Float16> src{{(const _Float16*)dy0, (const _Float16*)dy1, (const _Float16*)dy2},
                                  {ld0, ld1, ld2},
                                  {out0, out0 + out1}};
        return launch_wgrad<_Float16>(src, x, ldx, dw, dw_dtype, workspace, rows, O, in_features, splits,
                                      as_stream(stream));
    }
    const WgSrc<__bf16> src{{(const __bf16*)dy0, (const __bf16*)dy1, (const __bf16*)dy2}, {ld0, ld1, ld2},
                            {out0, out0 + out1}};
    return launch_wgrad<__bf16>(src, x, ldx, dw, dw_dtype, workspace, rows, O, in_features, splits, as_stream(stream));
}
