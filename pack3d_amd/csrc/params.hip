// Small passes around the 16-bit training step that carry little data each and
// were one torch launch (or several) apiece: sums of partial parameter
// gradients with their cast, the gate's pair softmax and its backward, weight
// casts, and the transposed concatenation of the input projections' weights.
// Each is bound by its launch and one or two memory round trips, so what counts
// is how many there are and that every load of a thread is in flight at once.  A
// 16-bit training step went from 52 launches to 32; in one of 32,768 tokens at
// dim 512 the parameter sums and casts fell from 150 to 25 us, the gate's backward
// (a fill, a strided copy, a product and a softmax backward) to 9 us, the gate and
// bias casts to 4.
#include <algorithm>

#include "common.hpp"

namespace p3d {
namespace {

// Store x into a tensor of a runtime dtype.
__device__ __forceinline__ void store_any(void* p, int64_t i, int dtype, float x) {
    if (dtype == P3D_F32) reinterpret_cast<float*>(p)[i] = x;
    else if (dtype == P3D_F16) reinterpret_cast<_Float16*>(p)[i] = (_Float16)x;
    else reinterpret_cast<__bf16*>(p)[i] = (__bf16)x;
}

// ------------------------------------------------------------- row sums
constexpr int kMaxJobs = 8;
constexpr int kSumThreads = 1024;

struct SumJobs {
    p3d_sum_job job[kMaxJobs];
    int first_block[kMaxJobs + 1];
    int cols_per_block[kMaxJobs];
    int count;
};

// dst[c] = sum over rows of src[r * stride + c], in a fixed order: a block
// takes CW columns and 1024 / CW groups of consecutive rows (each thread's
// loads issued eight at a time), then adds the groups in order.
__global__ __launch_bounds__(kSumThreads) void k_sum_rows(SumJobs a) {
    __shared__ float part[kSumThreads];
    int j = 0;
    while (j + 1 < a.count && (int)blockIdx.x >= a.first_block[j + 1]) ++j;
    const p3d_sum_job& job = a.job[j];
    const int cw = a.cols_per_block[j], groups = kSumThreads / cw;
    const int lc = threadIdx.x % cw, grp = threadIdx.x / cw;
    const int64_t c = (int64_t)((int)blockIdx.x - a.first_block[j]) * cw + lc;
    float sum = 0.f;
    if (c < job.cols) {
        const int64_t per = (job.rows + groups - 1) / groups;
        const int64_t first = grp * per, last = min(first + per, job.rows);
        const float* p = job.src + c;
        for (int64_t r = first; r < last; r += 8) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = p[min(r + i, last - 1) * job.stride];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (r + i < last) sum += v[i];
        }
    }
    part[threadIdx.x] = sum;
    __syncthreads();
    // Pairwise over the groups: groups is a power of two.
    for (int h = groups / 2; h >= 1; h /= 2) {
        if (grp < h) part[threadIdx.x] += part[threadIdx.x + h * cw];
        __syncthreads();
    }
    if (grp == 0 && c < job.cols) store_any(job.dst, c, job.dtype, part[lc]);
}

// ----------------------------------------------------------------- gate
// The second probability of the softmax over a logit pair (attention.py:85):
// computed in fp32 from 16-bit logits.
__device__ __forceinline__ void pair_softmax(float l0, float l1, float& y0, float& y1) {
    const float m = fmaxf(l0, l1), e0 = expf(l0 - m), e1 = expf(l1 - m), inv = 1.f / (e0 + e1);
    y0 = e0 * inv;
    y1 = e1 * inv;
}

template <typename T>
__global__ __launch_bounds__(256) void k_gate_fwd(const T* logits, void* gate, int gate_dtype, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    typedef __attribute__((ext_vector_type(2))) T T2;
    const T2 l = reinterpret_cast<const T2*>(logits)[i];
    float y0, y1;
    pair_softmax(to_f32(l[0]), to_f32(l[1]), y0, y1);
    store_any(gate, i, gate_dtype, y1);
}

// dlogits of the pair softmax from the gradient dgate of its second entry:
// d(1) = y1 (dg - y1 dg) = y0 y1 dg, d(0) = -y0 y1 dg.  dgate is [B, H, N]
// (any strides, tokens contiguous in use); a thread takes one token, so that
// its reads run along the tokens and its writes are one row of logits.  Each
// block also writes the column sums of its unrounded dlogits, the gradient of
// the bias that the logits hold, to part[block][2 H].  Grid y takes kGateHeads
// heads each, whose sums fit in LDS.
constexpr int kGateHeads = 2048;
template <typename T>
__global__ __launch_bounds__(256) void k_gate_bwd(const T* logits, p3d_view dgate, int dgate_dtype, T* dlogits,
                                                  float* part, int H, int64_t N, int64_t tokens) {
    extern __shared__ float red[];  // [4 waves][HB]
    const int h0 = blockIdx.y * kGateHeads, HB = min(kGateHeads, H - h0);
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool ok = t < tokens;
    const int64_t b = ok ? t / N : 0, n = ok ? t - b * N : 0;
    typedef __attribute__((ext_vector_type(2))) T T2;
    const T2* l = reinterpret_cast<const T2*>(logits) + (ok ? t : 0) * H + h0;
    T2* d = reinterpret_cast<T2*>(dlogits) + (ok ? t : 0) * H + h0;
    for (int h = 0; h < HB; ++h) {
        const T2 x = l[h];
        float y0, y1;
        pair_softmax(to_f32(x[0]), to_f32(x[1]), y0, y1);
        const float g = load_any(dgate.data, b * dgate.sb + (int64_t)(h0 + h) * dgate.sh + n * dgate.sn, dgate_dtype);
        const float v = ok ? y0 * y1 * g : 0.f;
        T2 o;
        o[0] = from_f32<T>(-v);
        o[1] = from_f32<T>(v);
        if (ok) d[h] = o;
        const float sum = wave_sum(v);
        if ((threadIdx.x & 63) == 0) red[(threadIdx.x >> 6) * HB + h] = sum;
    }
    __syncthreads();
    float* mine = part + ((int64_t)blockIdx.x * H + h0) * 2;
    for (int h = threadIdx.x; h < HB; h += 256) {
        const float s = (red[h] + red[HB + h]) + (red[2 * HB + h] + red[3 * HB + h]);
        mine[2 * h] = -s;
        mine[2 * h + 1] = s;
    }
}

// ---------------------------------------------------------------- casts
struct CastJobs {
    p3d_cast_job job[kMaxJobs];
    int first_block[kMaxJobs + 1];
    int count;
};

constexpr int kCastPerBlock = 2048;  // 8 elements per thread

__global__ __launch_bounds__(256) void k_cast(CastJobs a) {
    int j = 0;
    while (j + 1 < a.count && (int)blockIdx.x >= a.first_block[j + 1]) ++j;
    const p3d_cast_job& job = a.job[j];
    const int64_t base = (int64_t)((int)blockIdx.x - a.first_block[j]) * kCastPerBlock;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t e = base + i * 256 + threadIdx.x;
        v[i] = load_any(job.src, min(e, job.count - 1), job.src_dtype);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t e = base + i * 256 + threadIdx.x;
        if (e < job.count) store_any(job.dst, e, job.dst_dtype, v[i]);
    }
}

// ------------------------------------------------- concatenated transpose
// wt[c][k] = W[k][c] of the concatenated rows of three [out_i, dim] matrices,
// zero for k in [out_0 + out_1 + out_2, k_pad): 32 x 32 tiles through LDS.
struct CatDev {
    const uint16_t* w[3];
    int end[3];  // first row past matrix i
    int dim, k_pad;
    uint16_t* wt;
};
__global__ __launch_bounds__(256) void k_concat_transpose(CatDev a) {
    __shared__ uint16_t tile[32][33];
    const int k0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int x = threadIdx.x & 31, y0 = threadIdx.x >> 5;
#pragma unroll
    for (int y = y0; y < 32; y += 8) {
        const int k = k0 + y, c = c0 + x;
        uint16_t v = 0;
        if (k < a.end[2] && c < a.dim) {
            const int i = k < a.end[0] ? 0 : (k < a.end[1] ? 1 : 2), start = i == 0 ? 0 : a.end[i - 1];
            v = a.w[i][(int64_t)(k - start) * a.dim + c];
        }
        tile[y][x] = v;
    }
    __syncthreads();
#pragma unroll
    for (int y = y0; y < 32; y += 8) {
        const int c = c0 + y, k = k0 + x;
        if (c < a.dim && k < a.k_pad) a.wt[(int64_t)c * a.k_pad + k] = tile[x][y];
    }
}

bool known(int dtype) { return dtype >= P3D_F32 && dtype <= P3D_BF16; }

}  // namespace
}  // namespace p3d

using namespace p3d;

extern "C" int p3d_sum_rows(const p3d_sum_job* jobs, int32_t count, void* stream) {
    P3D_REQUIRE(jobs && count >= 1 && count <= kMaxJobs, "need 1 to 8 jobs");
    SumJobs a{};
    a.count = count;
    int64_t blocks = 0;
    for (int j = 0; j < count; ++j) {
        const p3d_sum_job& job = jobs[j];
        P3D_REQUIRE(job.src && job.dst && job.rows >= 1 && job.cols >= 1 && known(job.dtype), "bad sum job");
        a.job[j] = job;
        // At most about 32 rows per thread: tall tables take few columns and
        // many row groups per block, short ones whole lines.
        a.cols_per_block[j] = job.rows <= 512 ? 64 : (job.rows <= 2048 ? 16 : 4);
        a.first_block[j] = (int)blocks;
        blocks += cdiv(job.cols, a.cols_per_block[j]);
    }
    P3D_REQUIRE(blocks < (1 << 30), "too many columns");
    a.first_block[count] = (int)blocks;
    k_sum_rows<<<(unsigned)blocks, kSumThreads, 0, as_stream(stream)>>>(a);
    return check_launch("p3d_sum_rows");
}

extern "C" int p3d_gate_fwd(const void* logits, int32_t dtype, void* gate, int32_t gate_dtype, int64_t count,
                            void* stream) {
    P3D_REQUIRE(logits && gate && count >= 1 && known(gate_dtype), "bad gate arguments");
    P3D_REQUIRE(dtype == P3D_F16 || dtype == P3D_BF16, "dtype must be fp16 or bf16");
    P3D_REQUIRE(cdiv(count, 256) < (1LL << 31), "launch grid too large");
    hipStream_t s = as_stream(stream);
    const unsigned blocks = (unsigned)cdiv(count, 256);
    if (dtype == P3D_F16)
        k_gate_fwd<_Float16><<<blocks, 256, 0, s>>>((const _Float16*)logits, gate, gate_dtype, count);
    else
        k_gate_fwd<__bf16><<<blocks, 256, 0, s>>>((const __bf16*)logits, gate, gate_dtype, count);
    return check_launch("p3d_gate_fwd");
}

extern "C" int p3d_gate_bwd(const void* logits, int32_t dtype, p3d_view dgate, int32_t dgate_dtype, void* dlogits,
                            float* part, int32_t batch, int32_t heads, int64_t tokens, void* stream) {
    P3D_REQUIRE(logits && dgate.data && dlogits && part && batch >= 1 && heads >= 1 && heads <= (1 << 24) && tokens >= 1 &&
                    known(dgate_dtype),
                "bad gate arguments");
    P3D_REQUIRE(dtype == P3D_F16 || dtype == P3D_BF16, "dtype must be fp16 or bf16");
    const int64_t all = batch * tokens;
    P3D_REQUIRE(cdiv(all, 256) < (1LL << 31), "launch grid too large");
    hipStream_t s = as_stream(stream);
    const dim3 blocks((unsigned)cdiv(all, 256), (unsigned)cdiv(heads, kGateHeads));
    const size_t lds = (size_t)4 * std::min(heads, kGateHeads) * sizeof(float);
    if (dtype == P3D_F16)
        k_gate_bwd<_Float16><<<blocks, 256, lds, s>>>((const _Float16*)logits, dgate, dgate_dtype, (_Float16*)dlogits,
                                                      part, heads, tokens, all);
    else
        k_gate_bwd<__bf16><<<blocks, 256, lds, s>>>((const __bf16*)logits, dgate, dgate_dtype, (__bf16*)dlogits, part,
                                                    heads, tokens, all);
    return check_launch("p3d_gate_bwd");
}

extern "C" int p3d_cast(const p3d_cast_job* jobs, int32_t count, void* stream) {
    P3D_REQUIRE(jobs && count >= 1 && count <= kMaxJobs, "need 1 to 8 jobs");
    CastJobs a{};
    a.count = count;
    int64_t blocks = 0;
    for (int j = 0; j < count; ++j) {
        const p3d_cast_job& job = jobs[j];
        P3D_REQUIRE(job.src && job.dst && job.count >= 1 && known(job.src_dtype) && known(job.dst_dtype), "bad cast job");
        a.job[j] = job;
        a.first_block[j] = (int)blocks;
        blocks += cdiv(job.count, kCastPerBlock);
    }
    P3D_REQUIRE(blocks < (1 << 30), "too many elements");
    a.first_block[count] = (int)blocks;
    k_cast<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(a);
    return check_launch("p3d_cast");
}

extern "C" int p3d_concat_transpose(const void* w0, int32_t out0, const void* w1, int32_t out1, const void* w2,
                                    int32_t out2, int32_t dim, void* wt, int32_t k_pad, void* stream) {
    P3D_REQUIRE(w0 && w1 && w2 && wt && out0 >= 1 && out1 >= 1 && out2 >= 1 && dim >= 1, "bad transpose arguments");
    P3D_REQUIRE((int64_t)out0 + out1 + out2 <= k_pad && k_pad <= (1 << 20) && dim <= (1 << 20), "k_pad must hold every row");
    const CatDev a{{(const uint16_t*)w0, (const uint16_t*)w1, (const uint16_t*)w2},
                   {out0, out0 + out1, out0 + out1 + out2}, dim, k_pad, (uint16_t*)wt};
    k_concat_transpose<<<dim3((unsigned)cdiv(k_pad, 32), (unsigned)cdiv(dim, 32)), 256, 0, as_stream(stream)>>>(a);
    return check_launch("p3d_concat_transpose");
}
