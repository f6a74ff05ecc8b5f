// gfx950 kernels for the rest of the decode step around the MoE layer
// (crates/llmpager-cuda/kernels/decode.cu: RMSNorm, scale-add, KV append,
// NeoX RoPE, GQA decode attention over f32 or f16 caches, bf16 row gather)
// and for MLA absorbed decode (kernels/mla.cu: interleaved RoPE, attention
// over the shared latent cache, batched bf16 GEMV, strided copy), behind
// 1:1 launchers with the reference's argument meaning.  The arithmetic is
// this build's own: decode attention is split over positions (one workgroup
// per (block of query heads of a kv head, split), partial records merged by a
// second kernel), and config 5's batched MLA decode over bf16 latent caches runs on MFMA.
#include "lp_device.h"

using namespace lp;
using namespace lpk;

namespace {

template <typename T>
__device__ __forceinline__ T* dptr(uint64_t a) {
    return reinterpret_cast<T*>(a);
}

// Sum / max over a workgroup of nw waves (red: nw floats of LDS).  Ends with a
// barrier, so LDS written before the call is visible after it.
__device__ __forceinline__ float block_sum(float v, float* red) {
    for (int o = 32; o >= 1; o >>= 1) v += shfl_xor(v, o);
    const int nw = (int)(blockDim.x >> 6);
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.0f;
    for (int w = 0; w < nw; ++w) t += red[w];
    __syncthreads();
    return t;
}

__device__ __forceinline__ float block_max(float v, float* red) {
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, shfl_xor(v, o));
    const int nw = (int)(blockDim.x >> 6);
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = -INFINITY;
    for (int w = 0; w < nw; ++w) t = fmaxf(t, red[w]);
    __syncthreads();
    return t;
}

__device__ __forceinline__ float half_bits_to_f32(uint32_t h) { return f16_bits_to_f32(h & 0xffffu); }

__device__ __forceinline__ uint16_t f32_to_half_bits(float f) {
    return __builtin_bit_cast(uint16_t, (_Float16)f);  // round to nearest even
}

}  // namespace

// ---------------------------------------------------------------------------
// RMSNorm per row (decode.cu:17-41): y[r] = x[r] * 1/sqrt(mean(x[r]^2) + eps)
// * w; w is shared by all rows; y may be x.  Rows of up to 1024 elements take
// a wave each (four per workgroup, no barrier), longer ones a workgroup; a
// row whose pieces are 16-byte aligned and at most 4 per thread is read once,
// with w, in one round of loads and kept in registers.  (One workgroup per
// row whatever its width, element by element and twice: 5.1 us on average
// over a decode layer's 1 x 2048, 32 x 128 and 4 x 128 norms, 2.6 now.)
// ---------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(256) lp_rmsnorm(const RmsNormArgs a) {
    __shared__ float red[4];
    const int per = a.wave_rows ? 64 : 256, i0 = a.wave_rows ? lane_id() : (int)threadIdx.x;
    const int row = a.wave_rows ? (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6) : (int)blockIdx.x;
    if (row >= a.rows) return;  // whole waves; with a workgroup per row, none
    const uint64_t xp = a.x + (uint64_t)row * (uint32_t)a.n * 4u, yp = a.y + (uint64_t)row * (uint32_t)a.n * 4u;
    auto total = [&](float v) {
        if (!a.wave_rows) return block_sum(v, red);
        for (int o = 32; o >= 1; o >>= 1) v += shfl_xor(v, o);
        return v;
    };
    if ((a.n & 3) == 0 && ((xp | yp | a.w) & 15) == 0 && a.n <= 16 * per) {
        float4 x[4], w[4];
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = i0 + j * per;
            x[j] = w[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (4 * i < a.n) {
                x[j] = gptr<float4>(xp)[i];
                w[j] = gptr<float4>(a.w)[i];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc = __builtin_fmaf(x[j].x, x[j].x, acc);
            acc = __builtin_fmaf(x[j].y, x[j].y, acc);
            acc = __builtin_fmaf(x[j].z, x[j].z, acc);
            acc = __builtin_fmaf(x[j].w, x[j].w, acc);
        }
        const float inv = 1.0f / sqrtf(total(acc) / (float)a.n + a.eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = i0 + j * per;
            if (4 * i < a.n)
                gptr_w<float4>(yp)[i] = make_float4(x[j].x * inv * w[j].x, x[j].y * inv * w[j].y,
                                                    x[j].z * inv * w[j].z, x[j].w * inv * w[j].w);
        }
        return;
    }
    const float* x = dptr<const float>(xp);
    const float* w = dptr<const float>(a.w);
    float* y = dptr<float>(yp);
    float acc = 0.0f;
    for (int i = i0; i < a.n; i += per) acc = __builtin_fmaf(x[i], x[i], acc);
    const float inv = 1.0f / sqrtf(total(acc) / (float)a.n + a.eps);
    for (int i = i0; i < a.n; i += per) y[i] = x[i] * inv * w[i];
}

// a += s * b (decode.cu:44-53)
extern "C" __global__ void __launch_bounds__(256) lp_scale_add(const ScaleAddArgs a) {
    float* pa = dptr<float>(a.a);
    const float* pb = dptr<const float>(a.b);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x)
        pa[i] = __builtin_fmaf(a.s, pb[i], pa[i]);
}

// The token's k / v ([kv_heads, head_dim]) into caches [kv_heads, max_seq,
// head_dim] at `pos` (decode.cu:57-77, 242-261); f16 caches round to
// nearest even.
extern "C" __global__ void __launch_bounds__(256) lp_kv_append_f32(const KvAppendArgs a) {
    const int total = a.kv_heads * a.head_dim;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int h = i / a.head_dim, d = i - h * a.head_dim;
        const size_t dst = ((size_t)h * a.max_seq + a.pos) * a.head_dim + d;
        dptr<float>(a.kcache)[dst] = dptr<const float>(a.k)[i];
        dptr<float>(a.vcache)[dst] = dptr<const float>(a.v)[i];
    }
}

extern "C" __global__ void __launch_bounds__(256) lp_kv_append_f16(const KvAppendArgs a) {
    const int total = a.kv_heads * a.head_dim;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int h = i / a.head_dim, d = i - h * a.head_dim;
        const size_t dst = ((size_t)h * a.max_seq + a.pos) * a.head_dim + d;
        dptr<uint16_t>(a.kcache)[dst] = f32_to_half_bits(dptr<const float>(a.k)[i]);
        dptr<uint16_t>(a.vcache)[dst] = f32_to_half_bits(dptr<const float>(a.v)[i]);
    }
}

// NeoX rotate-half RoPE in place over [heads, head_dim] (decode.cu:145-167):
// pair (i, i + hd/2) rotates by pos * base^(-2i/hd).  Library powf / cosf /
// sinf (the reference's fast-math intrinsics are approximations of these).
extern "C" __global__ void __launch_bounds__(256) lp_rope(const RopeArgs a) {
    const int half = a.head_dim >> 1;
    for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < a.heads * half; idx += gridDim.x * blockDim.x) {
        const int h = idx / half, i = idx - h * half;
        const float freq = powf(a.base, -2.0f * (float)i / (float)a.head_dim);
        const float ang = (float)a.pos * freq;
        const float c = cosf(ang), s = sinf(ang);
        float* p = dptr<float>(a.x) + (size_t)h * a.head_dim;
        const float x1 = p[i], x2 = p[i + half];
        p[i] = x1 * c - x2 * s;
        p[i + half] = x1 * s + x2 * c;
    }
}

// out[n] = f32(table[row, :n]) (decode.cu:328-339)
extern "C" __global__ void __launch_bounds__(256) lp_bf16_row_to_f32(const RowArgs a) {
    const uint16_t* src = dptr<const uint16_t>(a.table) + (size_t)a.row * a.n;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x)
        dptr<float>(a.out)[i] = bf16_to_f32(src[i]);
}

// Interleaved RoPE with a frequency table (mla.cu:22-45): pairs (2i, 2i+1) of
// the slice at `offset` in each of n_vecs vectors rotate by pos * inv_freq[i],
// both factors scaled by mscale.
extern "C" __global__ void __launch_bounds__(256) lp_mla_rope(const MlaRopeArgs a) {
    const float* fr = dptr<const float>(a.inv_freq);
    for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < a.n_vecs * a.half; idx += gridDim.x * blockDim.x) {
        const int v = idx / a.half, i = idx - v * a.half;
        const float ang = (float)a.pos * fr[i];
        const float c = cosf(ang) * a.mscale, s = sinf(ang) * a.mscale;
        float* p = dptr<float>(a.x) + (size_t)v * a.stride + a.offset + 2 * i;
        const float x1 = p[0], x2 = p[1];
        p[0] = x1 * c - x2 * s;
        p[1] = x1 * s + x2 * c;
    }
}

// Batched bf16 GEMV (mla.cu:120-148): y_b = W_b x_b, W_b = w + b w_stride
// [rows, cols] row-major, x_b = x + b x_stride, y_b = y + b y_stride (strides
// in elements).  One wave per row, lanes over 8-column chunks (16-byte loads
// when the row and x_b are 16-byte aligned), butterfly reduction.  Grid
// (ceil(rows / 4), batch).
extern "C" __global__ void __launch_bounds__(256) lp_bf16_gemv_batch(const Bf16GemvBatchArgs a) {
    const int b = blockIdx.y;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = lane_id();
    if (row >= a.rows) return;
    const uint16_t* w = dptr<const uint16_t>(a.w) + (size_t)b * a.w_stride + (size_t)row * a.cols;
    const float* x = dptr<const float>(a.x) + (size_t)b * a.x_stride;
    float acc = 0.0f;
    const bool vec = (a.cols & 7) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    if (vec) {
        for (int ch = lane; ch < (a.cols >> 3); ch += 64) {
            const uint4 wv = *reinterpret_cast<const uint4*>(w + ch * 8);
            const float4 xa = *reinterpret_cast<const float4*>(x + ch * 8);
            const float4 xb = *reinterpret_cast<const float4*>(x + ch * 8 + 4);
            acc = __builtin_fmaf(bf16_to_f32(wv.x & 0xffffu), xa.x, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.x >> 16), xa.y, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.y & 0xffffu), xa.z, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.y >> 16), xa.w, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.z & 0xffffu), xb.x, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.z >> 16), xb.y, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.w & 0xffffu), xb.z, acc);
            acc = __builtin_fmaf(bf16_to_f32(wv.w >> 16), xb.w, acc);
        }
    } else {
        for (int c = lane; c < a.cols; c += 64) acc = __builtin_fmaf(bf16_to_f32(w[c]), x[c], acc);
    }
    for (int o = 32; o >= 1; o >>= 1) acc += shfl_xor(acc, o);
    if (lane == 0) dptr<float>(a.y)[(size_t)b * a.y_stride + row] = acc;
}

// dst[v dst_stride + dst_off + i] = src[v src_stride + src_off + i]
// (mla.cu:153-166)
extern "C" __global__ void __launch_bounds__(256) lp_strided_copy(const StridedCopyArgs a) {
    for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < a.n_vecs * a.n; idx += gridDim.x * blockDim.x) {
        const int v = idx / a.n, i = idx - v * a.n;
        dptr<float>(a.dst)[(size_t)v * a.dst_stride + a.dst_off + i] =
            dptr<const float>(a.src)[(size_t)v * a.src_stride + a.src_off + i];
    }
}

// ---------------------------------------------------------------------------
// Decode attention, one query per head, split over positions (attn_decode_f32
// / _f16kv, decode.cu:172-325; mla_attn_decode_f32, mla.cu:51-111).  Grid
// (kv heads x blocks of kAttnHeads query heads of one kv head, splits), 256
// threads.
//
// One token's attention is a chain of memory round trips, not bytes (3 MB at
// 1,500 positions of 4 kv heads), so a workgroup brings a chunk of rows'
// keys and values in by one burst of coalesced loads, fp32 in LDS, and all
// query heads of the kv head use them: each row is read once for the group,
// the next chunk's while this one is worked on.
//   scores   attn_scores: LDS reads bound it, so each piece serves several
//            products; the rows are padded by 16 bytes;
//   softmax  online over the chunks, each head's scores in half a wave;
//   context  thread (4 columns, kAttnHeads / slots heads): rows from LDS,
//            probabilities of four rows at a time, broadcast.
// One split writes out[h] = acc / sum; more write records {max, sum,
// acc[out_dim]} that lp_attn_combine merges.  Measured, whole calls (us),
// with a thread per key row and a workgroup per query head, with one row and
// head per thread and chunks loaded when they are needed, and as it is:
// 32 heads on 4 kv heads of 128 f16, 1,500 rows 35.1, 13.0, 12.7 (100 rows 9.8,
// 11.0, 9.3); MLA, 16 heads of 576 / 512 in a cache of 4,096 (its scratch
// holds seven records), 700 rows 40.2, 66.9, 38.8 and 1,500 rows 65.4, 108.9,
// 61.9.
// ---------------------------------------------------------------------------
namespace {

// Rows of a cache from element `at` as fp32 in LDS, row stride rs floats,
// columns past n zero.  A vector piece is 16 bytes; NP pieces per thread are
// loaded (load) before the first is stored (store).
template <bool F16, int NP>
struct AttnStage {
    static constexpr int kPer = F16 ? 8 : 4;
    uint64_t src;  // address of the first row
    float* dst;
    int row_bytes, rs, n, n4, rows, pieces;
    int per, dr, dm;  // pieces of a row; 256 pieces further: rows, pieces
    int r0, m0;       // this thread's first piece not yet stored: row, piece
    bool vec;
    u32x4_t u[NP];
    __device__ __forceinline__ AttnStage(float* d, int rs_, uint64_t base, size_t at, int row_stride, int n_, int n4_)
        : src(base + at * (F16 ? 2 : 4)), dst(d), row_bytes(row_stride * (F16 ? 2 : 4)), rs(rs_), n(n_), n4(n4_) {
        vec = (n & (kPer - 1)) == 0 && (src & 15) == 0 && (row_bytes & 15) == 0;
        per = max(n / kPer, 1);
        dr = 256 / per, dm = 256 - dr * per;
    }
    // the rows to bring in: rows_ of them, `skip` past those before
    __device__ __forceinline__ void next(int skip, int rows_) {
        src += (uint64_t)(uint32_t)skip * (uint32_t)row_bytes;
        rows = rows_;
        pieces = vec ? rows * per : 0;
        r0 = (int)threadIdx.x / per, m0 = (int)threadIdx.x - r0 * per;
    }
    __device__ __forceinline__ void step(int& r, int& m) const {
        r += dr, m += dm;
        if (m >= per) ++r, m -= per;
    }
    __device__ __forceinline__ void load(int i0) {
        int r = r0, m = m0;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            if (i0 + 256 * j >= pieces) break;  // uniform
            u[j] = *gptr<u32x4_t>(src + (uint64_t)((uint32_t)min(r, rows - 1) * (uint32_t)row_bytes + 16u * (uint32_t)m));
            step(r, m);
        }
    }
    __device__ __forceinline__ void store(int i0) {
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            if (i0 + 256 * j >= pieces) break;
            if (r0 < rows) {
                float* o = dst + r0 * rs + m0 * kPer;
                if constexpr (F16) {
                    reinterpret_cast<float4*>(o)[0] =
                        make_float4(half_bits_to_f32(u[j][0]), half_bits_to_f32(u[j][0] >> 16), half_bits_to_f32(u[j][1]),
                                    half_bits_to_f32(u[j][1] >> 16));
                    reinterpret_cast<float4*>(o)[1] =
                        make_float4(half_bits_to_f32(u[j][2]), half_bits_to_f32(u[j][2] >> 16), half_bits_to_f32(u[j][3]),
                                    half_bits_to_f32(u[j][3] >> 16));
                } else {
                    *reinterpret_cast<u32x4_t*>(o) = u[j];
                }
            }
            step(r0, m0);
        }
    }
    // the whole of it from the second round on (the first is in flight)
    __device__ __forceinline__ void finish() {
        store(0);
        for (int i = 256 * NP; i < pieces; i += 256 * NP) {
            load(i);
            store(i);
        }
        if (vec) return;
        for (int i = threadIdx.x; i < rows * 4 * n4; i += 256) {  // no 16-byte pieces
            const int r = i / (4 * n4), c = i - r * 4 * n4;
            const uint64_t row = src + (uint64_t)r * (uint32_t)row_bytes;
            float v = 0.0f;
            if (c < n) {
                if constexpr (F16)
                    v = half_bits_to_f32(gptr<uint16_t>(row)[c]);
                else
                    v = gptr<float>(row)[c];
            }
            dst[r * rs + c] = v;
        }
    }
};

// A chunk's scores before their scale, pr[head][row] for rows 0 .. 16 R - 1:
// thread (part tid % 8, head quad, rg = tid / 16) multiplies the row pieces
// part, part + 8, ... of rows rg + 16 r with its four heads', so that a piece
// read from LDS serves R or four products (LDS reads bound this pass).
template <int R>
__device__ __forceinline__ void attn_scores(const float* qs, const float* kt, int krs, int d4, float* pr) {
    static_assert(kAttnHeads == 8, "two quads of heads");
    const int part = threadIdx.x & 7, h4 = ((threadIdx.x >> 3) & 1) * 4, rg = threadIdx.x >> 4;
    float acc[4][R];
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[h][r] = 0.0f;
    const float4* q4 = reinterpret_cast<const float4*>(qs) + h4 * d4;
    for (int i = part; i < d4; i += 8) {
        float4 k[R];
#pragma unroll
        for (int r = 0; r < R; ++r) k[r] = reinterpret_cast<const float4*>(kt + (rg + 16 * r) * krs)[i];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const float4 y = q4[h * d4 + i];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                acc[h][r] = __builtin_fmaf(y.x, k[r].x, acc[h][r]);
                acc[h][r] = __builtin_fmaf(y.y, k[r].y, acc[h][r]);
                acc[h][r] = __builtin_fmaf(y.z, k[r].z, acc[h][r]);
                acc[h][r] = __builtin_fmaf(y.w, k[r].w, acc[h][r]);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float v = acc[h][r];  // over the eight lanes: quad permutations, then the halves of eight
            v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, false));
            v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, false));
            v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));
            if (part == ((h * R + r) & 7)) pr[(h4 + h) * kAttnRows + rg + 16 * r] = v;
        }
}

// HPT: query heads per thread in the context pass (1 up to 128 columns, 2 up
// to 256, 4 up to 512, 8 up to 1024).  NK, NV: pieces of keys and values per
// thread in flight (18: the whole of an MLA chunk, 32 rows of 576 f32).
template <bool F16, int HPT, int NK, int NV>
__device__ __forceinline__ void attn_split_body(const AttnArgs& a) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, sp = blockIdx.y;
    const int blocks = (a.group + kAttnHeads - 1) / kAttnHeads;
    const int kvh = blockIdx.x / blocks, h0 = kvh * a.group + (blockIdx.x - kvh * blocks) * kAttnHeads;
    const int nh = min(kAttnHeads, (kvh + 1) * a.group - h0);
    const int d4 = (a.dot_dim + 3) >> 2, o4 = (a.out_dim + 3) >> 2;
    const int krs = attn_row_floats(a.dot_dim), vrs = a.shared_kv ? krs : attn_row_floats(a.out_dim);
    float* qs = reinterpret_cast<float*>(lds);  // [kAttnHeads][4 d4]
    float* pr = qs + kAttnHeads * 4 * d4;       // [kAttnHeads][kAttnRows]
    float* al = pr + kAttnHeads * kAttnRows;    // [kAttnHeads]: the chunk's rescaling
    float* kt = al + kAttnHeads;                // [rows][krs]
    float* vt = a.shared_kv ? kt : kt + a.rows * krs;
    // the block's query heads: rows of dot_dim floats one behind the other
    const uint64_t q = a.q + (uint64_t)h0 * (uint32_t)a.dot_dim * 4u;
    const bool qvec = (a.dot_dim & 3) == 0 && (q & 15) == 0;
    constexpr int NQ = 8;  // up to 8 heads of 1024 columns by 16-byte pieces
    float4 qv[NQ];
    if (qvec) {
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const int i = tid + 256 * j;
            qv[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (i < nh * d4) qv[j] = gptr<float4>(q)[i];
        }
    }
    const size_t kv_off = (size_t)kvh * a.kv_stride;
    const int p0 = sp * a.span, p1 = min(a.seq_len, p0 + a.span);
    const int pl = tid & 31, hl = tid >> 5;  // score pass: row, head
    float m = -INFINITY, l = 0.0f;           // head hl's running max and sum (in its 32 lanes alike)
    // context pass: columns 4 c .. 4 c + 3, heads hs, hs + slots, ...
    const int quads = o4 <= 32 ? 32 : o4 <= 64 ? 64 : o4 <= 128 ? 128 : 256;
    const int c = tid & (quads - 1), hs = tid / quads, slots = 256 / quads;
    float4 acc[HPT];
#pragma unroll
    for (int j = 0; j < HPT; ++j) acc[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // a chunk's loads go out before the previous chunk is worked on
    const size_t at = kv_off + (size_t)p0 * a.row_stride;
    AttnStage<F16, NK> K(kt, krs, a.k, at, a.row_stride, a.dot_dim, d4);
    AttnStage<F16, NV> V(vt, vrs, a.v, at, a.row_stride, a.out_dim, o4);
    auto issue = [&](int skip, int n) {
        K.next(skip, n);
        V.next(skip, a.shared_kv ? 0 : n);
        K.load(0);
        V.load(0);
    };
    issue(0, min(a.rows, p1 - p0));
    if (qvec) {
#pragma unroll
        for (int j = 0; j < NQ; ++j)
            if (tid + 256 * j < kAttnHeads * d4) reinterpret_cast<float4*>(qs)[tid + 256 * j] = qv[j];
    } else {
        for (int i = tid; i < kAttnHeads * 4 * d4; i += 256) {
            const int h = i / (4 * d4), d = i - h * 4 * d4;
            qs[i] = h < nh && d < a.dot_dim ? gptr<float>(q)[h * a.dot_dim + d] : 0.0f;
        }
    }
    for (int p = p0; p < p1; p += a.rows) {
        const int n = min(a.rows, p1 - p);
        if (p > p0) __syncthreads();  // the previous chunk's rows are read
        K.finish();
        V.finish();
        __syncthreads();
        if (p + a.rows < p1) issue(a.rows, min(a.rows, p1 - p - a.rows));
        // partial dot products: rows rg, rg + 16, ... of the chunk against four
        // heads, every eighth piece of the row; the eight parts meet in lanes
        if (n > 32)
            attn_scores<4>(qs, kt, krs, d4, pr);
        else if (n > 16)
            attn_scores<2>(qs, kt, krs, d4, pr);
        else
            attn_scores<1>(qs, kt, krs, d4, pr);
        __syncthreads();
        float s0 = pl < n ? pr[hl * kAttnRows + pl] * a.scale : -INFINITY;
        float s1 = pl + 32 < n ? pr[hl * kAttnRows + pl + 32] * a.scale : -INFINITY;
        float mx = fmaxf(s0, s1);
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) mx = fmaxf(mx, shfl_xor(mx, o));
        const float mn = fmaxf(m, mx);
        // every score so far -inf: nothing to rescale, nothing added
        const float alpha = mn == -INFINITY ? 1.0f : expf(m - mn);
        const float e0 = mn == -INFINITY ? 0.0f : expf(s0 - mn);
        const float e1 = mn == -INFINITY ? 0.0f : expf(s1 - mn);
        float sum = e0 + e1;
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) sum += shfl_xor(sum, o);
        l = __builtin_fmaf(l, alpha, sum);
        m = mn;
        pr[hl * kAttnRows + pl] = e0;
        pr[hl * kAttnRows + pl + 32] = e1;
        if (pl == 0) al[hl] = alpha;
        __syncthreads();
        if (c < o4) {
#pragma unroll
            for (int j = 0; j < HPT; ++j) {
                const float f = al[(hs + j * slots) & (kAttnHeads - 1)];
                acc[j] = make_float4(acc[j].x * f, acc[j].y * f, acc[j].z * f, acc[j].w * f);
            }
            auto add = [&](float4& o, float w, const float4& v) {
                o.x = __builtin_fmaf(w, v.x, o.x);
                o.y = __builtin_fmaf(w, v.y, o.y);
                o.z = __builtin_fmaf(w, v.z, o.z);
                o.w = __builtin_fmaf(w, v.w, o.w);
            };
            const float* vc = vt + 4 * c;
            int r = 0;
#pragma unroll 2
            for (; r + 4 <= n; r += 4) {
                float4 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const float4*>(vc + (r + i) * vrs);
#pragma unroll
                for (int j = 0; j < HPT; ++j) {
                    const float4 w = *reinterpret_cast<const float4*>(
                        pr + ((hs + j * slots) & (kAttnHeads - 1)) * kAttnRows + r);
                    add(acc[j], w.x, v[0]);
                    add(acc[j], w.y, v[1]);
                    add(acc[j], w.z, v[2]);
                    add(acc[j], w.w, v[3]);
                }
            }
            for (; r < n; ++r)
#pragma unroll
                for (int j = 0; j < HPT; ++j)
                    add(acc[j], pr[((hs + j * slots) & (kAttnHeads - 1)) * kAttnRows + r],
                        *reinterpret_cast<const float4*>(vc + r * vrs));
        }
    }
    // each head's max and sum to the threads that hold its columns
    __syncthreads();
    if (pl == 0) pr[2 * hl] = m, pr[2 * hl + 1] = l;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < HPT; ++j) {
        const int h = hs + j * slots;
        if (h >= nh || c >= o4) continue;
        const float f = a.splits == 1 ? 1.0f / pr[2 * h + 1] : 1.0f;
        float* o = a.splits == 1 ? dptr<float>(a.out) + (size_t)(h0 + h) * a.out_dim
                                 : dptr<float>(a.scratch) + (size_t)(h0 + h) * a.scratch_stride +
                                       (size_t)sp * (a.out_dim + 2) + 2;
        const float v[4] = {acc[j].x * f, acc[j].y * f, acc[j].z * f, acc[j].w * f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * c + i < a.out_dim) o[4 * c + i] = v[i];
        if (a.splits > 1 && c == 0) {
            o[-2] = pr[2 * h];
            o[-1] = pr[2 * h + 1];
        }
    }
}

template <bool F16>
__device__ __forceinline__ void attn_split(const AttnArgs& a) {
    if (a.out_dim <= 128)
        attn_split_body<F16, 1, 8, 8>(a);
    else
        attn_split_body<F16, 2, 8, 8>(a);
}

template <bool F16>
__device__ __forceinline__ void attn_split_wide(const AttnArgs& a) {
    if (a.out_dim <= 512)
        attn_split_body<F16, 4, 18, 8>(a);
    else
        attn_split_body<F16, 8, 8, 8>(a);
}

}  // namespace

// Up to 256 columns of out, and wider rows (kernels of their own: their
// registers would halve the narrow ones' occupancy).
extern "C" __global__ void __launch_bounds__(256) lp_attn_split_f32(const AttnArgs a) { attn_split<false>(a); }
extern "C" __global__ void __launch_bounds__(256) lp_attn_split_f16(const AttnArgs a) { attn_split<true>(a); }
extern "C" __global__ void __launch_bounds__(256) lp_attn_split_wide_f32(const AttnArgs a) { attn_split_wide<false>(a); }
extern "C" __global__ void __launch_bounds__(256) lp_attn_split_wide_f16(const AttnArgs a) { attn_split_wide<true>(a); }

// Merge of the split records: out[h][d] = sum_s e^(m_s - M) acc_s[d] /
// sum_s e^(m_s - M) l_s, M = max_s m_s.  Grid (heads, ceil(out_dim / 64)),
// 256 threads: the weights to LDS, one split per thread, then thread (column
// d, group g) sums the splits g, g + 4, ... and the groups meet in LDS, so
// that the records come in a few bursts instead of one dependent load per
// split.
extern "C" __global__ void __launch_bounds__(256) lp_attn_combine(const AttnArgs a) {
    __shared__ float wsh[kAttnMaxSplits];
    __shared__ float red[4];
    __shared__ float part[4][64];
    const int h = blockIdx.x, tid = threadIdx.x;
    const float* base = dptr<const float>(a.scratch) + (size_t)h * a.scratch_stride;
    const int rec = a.out_dim + 2;
    const float ms = tid < a.splits ? base[(size_t)tid * rec] : -INFINITY;
    const float ls = tid < a.splits ? base[(size_t)tid * rec + 1] : 0.0f;
    const float M = block_max(ms, red);
    const float w = ms == -INFINITY ? 0.0f : expf(ms - M);
    const float den = block_sum(w * ls, red);
    if (tid < a.splits) wsh[tid] = ms == -INFINITY ? -1.0f : w;  // -1: an empty split
    __syncthreads();
    const int d = blockIdx.y * 64 + (tid & 63), g = tid >> 6;
    float num = 0.0f;
    if (d < a.out_dim) {
        const float* col = base + 2 + d;
#pragma unroll 8
        for (int s = g; s < a.splits; s += 4) {
            const float v = col[(size_t)s * rec], ws = wsh[s];
            num = ws < 0.0f ? num : __builtin_fmaf(ws, v, num);
        }
    }
    part[g][tid & 63] = num;
    __syncthreads();
    if (g == 0 && d < a.out_dim)
        dptr<float>(a.out)[(size_t)h * a.out_dim + d] =
            ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])) / den;
}

// ---------------------------------------------------------------------------
// Batched MLA decode over bf16 latent caches (config 5), on MFMA.  Grid
// (splits, batch), 4 waves.  Split s of sequence b walks its positions in
// chunks of 64 cache rows with an online softmax over the chunks:
//   scores  S[h][r] = scale * q_h . row_r: v_mfma_f32_16x16x32_bf16 with
//           the query as A (heads as M; its fp32 values split into bf16
//           hi + lo, two MFMAs per step, so the query keeps 16 significant
//           bits) and 16 cache rows per wave as B, loaded as 16-byte row
//           pieces straight into registers (the next chunk's loads are in
//           flight while this chunk's softmax and context are computed);
//   softmax per head over the chunk, the running max and sum rescaled;
//   context ctx[h][d] += sum_r p[h][r] row_r[d]: the same MFMA with the
//           probabilities (hi + lo) as A and the chunk as B (each wave a
//           quarter of the c_dim columns): the rows go to LDS as they are
//           (one 16-byte store per lane and step during the score pass) and
//           the B operand comes back column-wise through the transposing
//           LDS read (ds_read_b64_tr_b16: each 16-lane group reads a 4-row x
//           16-column block, lane i receiving column i's four values).
// A workgroup's time is its chain of chunks, and at the capacity's split a
// batch of shorter sequences leaves part of the workgroups without rows and
// the others with the longest chain: where a split has several chunks
// the same workgroups are shared out by the lengths (the _bal kernels,
// mla_share; kernels of their own, as the test costs the others 0.25 us).
// 16 sequences of 1,024 to 4,096 rows in caches of 4,096: 29.2 us a call by
// the capacity's split, 26.7 by lengths; all 4,096 long (the split that the
// capacity gives): 31.8 and 31.2.  The query's loads of the capacity's
// sequence go out before the lengths arrive (and again if it is another).
// The cache rows are read once from HBM.  Each split ends with a partial
// record {max[16], sum[16], acc[16][c_dim]}; lp_mla_combine merges them.
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ uint32_t pack_bf16(uint32_t lo, uint32_t hi) { return lo | (hi << 16); }

typedef short v4i16_t __attribute__((ext_vector_type(4)));

// e^x for the batched MLA's softmax (x <= 0 there): the hardware base-2
// exponential of x log2(e), within a few ulp (the bf16 cache bounds the
// result's precision far below that); -inf gives 0.
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

// hi / lo bf16 images of eight fp32 values, element order = value order
__device__ __forceinline__ void split8(const float (&v)[8], uint4& hi, uint4& lo) {
    uint32_t h[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        h[i] = f32_to_bf16_rne(v[i]);
        l[i] = f32_to_bf16_rne(v[i] - bf16_to_f32(h[i]));
    }
    hi = make_uint4(pack_bf16(h[0], h[1]), pack_bf16(h[2], h[3]), pack_bf16(h[4], h[5]), pack_bf16(h[6], h[7]));
    lo = make_uint4(pack_bf16(l[0], l[1]), pack_bf16(l[2], l[3]), pack_bf16(l[4], l[5]), pack_bf16(l[6], l[7]));
}

__device__ __forceinline__ f32x4_t mfma_bf16(const uint4& a, const uint4& b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// The sharing by lengths, one sequence per lane (batch <= 64): the fewest
// chunks `per` for which every sequence's splits of `per` chunks (at least
// one each) fit the launch's batch x splits workgroups; the capacity's split
// always fits.  Sequence b's splits, and their records, are [incl - splits,
// incl) of lane b.  False: no shorter chain than the capacity's split.
struct MlaShare {
    int per, splits, incl;
};
__device__ __forceinline__ bool mla_share(const MlaBatchArgs& a, int len, MlaShare& o) {
    const int cap = a.span / kMlaRows, n = a.batch * a.splits;
    const int chunks = lane_id() < a.batch ? max(1, (min(len, a.max_seq) + kMlaRows - 1) / kMlaRows) : 0;
    const int total = __builtin_amdgcn_readlane(wave_incl_scan(chunks), 63);
    for (int per = (total + n - 1) / n; per < cap; ++per) {
        const int s = (chunks + per - 1) / per, incl = wave_incl_scan(s);
        if (__builtin_amdgcn_readlane(incl, 63) <= n) {
            o = {per, s, incl};
            return true;
        }
    }
    return false;
}

__device__ __forceinline__ int mla_len(const MlaBatchArgs& a) {
    return lane_id() < a.batch ? gptr<int>(a.seq_lens)[lane_id()] : 0;
}

template <int STEPS, bool BAL>
__device__ __forceinline__ void mla_split_body(const MlaBatchArgs& a) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int QK = 32 * STEPS;
    int b = blockIdx.y, sp = blockIdx.x, span = a.span, rec = b * a.splits + sp;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const int n = lane & 15, kb = lane >> 4;
    const int H = a.heads, CD = a.c_dim;
    const int tpw = CD >> 6;  // 16-column tiles per wave (a quarter of c_dim)
    uint4* qhi = reinterpret_cast<uint4*>(lds);
    uint4* qlo = qhi + STEPS * 64;
    const int rsb = mla_row_bytes(CD);
    uint8_t* ct = lds + 2 * STEPS * 1024;  // the chunk's first c_dim columns: [kMlaRows][rsb]
    const uint32_t ct_addr = lds_addr_of(ct);
    float* sl = reinterpret_cast<float*>(ct + kMlaRows * rsb);  // [16][64]
    // a length past the cache is cut to the cache (rows beyond max_seq
    // belong to the next sequence, or to no allocation at all)
    int seq;
    if constexpr (BAL)
        seq = mla_len(a);
    else
        seq = dptr<const int>(a.seq_lens)[b];
    // the query's loads behind the lengths', before any of them is waited for
    constexpr int kUnits = (STEPS * 64 + 255) / 256;  // query pieces per thread
    float4 v4[kUnits][2];
    auto load_q = [&](int bq) {
        const uint64_t q = a.q + (uint64_t)bq * H * QK * 4;
#pragma unroll
        for (int r = 0; r < kUnits; ++r) {
            const int u = tid + 256 * r, j = u >> 6, l = u & 63, m = l & 15, k8 = l >> 4;
            v4[r][0] = v4[r][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (u < STEPS * 64 && m < H) {
                const LP_GLOBAL float4* src = gptr<float4>(q + ((uint64_t)m * QK + 32 * j + 8 * k8) * 4);
                v4[r][0] = src[0];
                v4[r][1] = src[1];
            }
        }
    };
    load_q(b);
    if constexpr (BAL) {
        MlaShare sh;
        if (mla_share(a, seq, sh)) {
            const int w = rec, b0 = b;
            b = __popcll(__ballot(sh.incl <= w));  // 64 past the last split
            if (b >= a.batch) return;              // the whole workgroup
            sp = w - (__builtin_amdgcn_readlane(sh.incl, b) - __builtin_amdgcn_readlane(sh.splits, b));
            span = sh.per * kMlaRows;
            if (b != b0) load_q(b);
        }
        seq = __builtin_amdgcn_readlane(seq, b);
    }
    seq = min(seq, a.max_seq);
    const int p0 = sp * span;
    const int p1 = min(seq, p0 + span);
    const int nchunks = p1 > p0 ? (p1 - p0 + kMlaRows - 1) / kMlaRows : 0;
    // the query's hi / lo images in A order: step j, lane (m, kb) holds
    // q[m][32 j + 8 kb .. + 7]; heads past H are zero
    // the sequence's valid rows through a raw buffer: rows past p1 read zero
    const uint64_t cb = a.cache + (uint64_t)b * a.cache_stride;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(uniform_u64(cb)), (short)0,
        __builtin_amdgcn_readfirstlane(p1 > 0 ? p1 * QK * 2 : 0), kBufferWord3);
    auto load_chunk = [&](uint4 (&B)[STEPS], int c) {
        const int row = p0 + c * kMlaRows + 16 * wave + n;
        const uint32_t off = (uint32_t)row * (QK * 2) + 16u * (uint32_t)kb;
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
            B[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + 64u * j), 0, 0));
    };
    float m_run = -INFINITY, l_run = 0.0f;  // head n (every kb lane holds the same)
    f32x4_t acc[kMlaMaxC / 64];
#pragma unroll
    for (int c = 0; c < kMlaMaxC / 64; ++c) acc[c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // one register buffer: a chunk's rows are dead once its scores are made,
    // so the next chunk's loads go into the same registers at that point
    auto chunk = [&](uint4 (&Bc)[STEPS], int c) {
        // scores of rows 16 wave + n; the chunk's first c_dim columns stored
        // row by row for the context pass
        f32x4_t s4 = {0.0f, 0.0f, 0.0f, 0.0f};
        const int rl = 16 * wave + n;
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            s4 = mfma_bf16(qhi[j * 64 + lane], Bc[j], s4);
            s4 = mfma_bf16(qlo[j * 64 + lane], Bc[j], s4);
            const int col = 32 * j + 8 * kb;
            if (col < CD) *reinterpret_cast<uint4*>(ct + (size_t)rl * rsb + col * 2) = Bc[j];
        }
        if (c + 1 < nchunks) load_chunk(Bc, c + 1);
        const bool rvalid = p0 + c * kMlaRows + rl < p1;
#pragma unroll
        for (int v = 0; v < 4; ++v) sl[(4 * kb + v) * kMlaRows + rl] = rvalid ? s4[v] * a.scale : -INFINITY;
        __syncthreads();
        // online softmax: lane (head n, kb) takes rows 32 s + 8 kb + i
        float sv[16];
        float mx = -INFINITY;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sv[8 * s + i] = sl[n * kMlaRows + 32 * s + 8 * kb + i];
                mx = fmaxf(mx, sv[8 * s + i]);
            }
        mx = fmaxf(mx, shfl_xor(mx, 16));
        mx = fmaxf(mx, shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const bool none = m_new == -INFINITY;  // every row so far masked
        const float alpha = none ? 1.0f : exp_hw(m_run - m_new);
        float ps = 0.0f;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            sv[t] = none ? 0.0f : exp_hw(sv[t] - m_new);
            ps += sv[t];
        }
        ps += shfl_xor(ps, 16);
        ps += shfl_xor(ps, 32);
        l_run = __builtin_fmaf(l_run, alpha, ps);
        m_run = m_new;
        float av[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) av[v] = __shfl(alpha, 4 * kb + v, 64);
        uint4 phi[2], plo[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float v8[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v8[i] = sv[8 * s + i];
            split8(v8, phi[s], plo[s]);
        }
        // context over this wave's columns: lane (n, kb) needs rows
        // 32 s + 8 kb .. + 7 of column n; lane i of group kb points the
        // transposing read at row 32 s + 8 kb + i / 4, columns 4 (i % 4) .. + 3
        // of the 16-column tile (and 4 rows further for the second half)
        const int li = lane & 15;
#pragma unroll
        for (int t = 0; t < kMlaMaxC / 64; ++t) {
            if (t < tpw) {  // uniform
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[t][v] *= av[v];
                const int col0 = wave * (CD >> 2) + 16 * t;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint32_t pa = ct_addr + (uint32_t)((32 * s + 8 * kb + (li >> 2)) * rsb) +
                                        (uint32_t)((col0 + 4 * (li & 3)) * 2);
                    const v4i16_t r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        reinterpret_cast<__attribute__((address_space(3))) v4i16_t*>((uintptr_t)pa));
                    const v4i16_t r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        reinterpret_cast<__attribute__((address_space(3))) v4i16_t*>((uintptr_t)(pa + 4u * rsb)));
                    const uint4 bt = make_uint4(pack_bf16((uint16_t)r0[0], (uint16_t)r0[1]),
                                                pack_bf16((uint16_t)r0[2], (uint16_t)r0[3]),
                                                pack_bf16((uint16_t)r1[0], (uint16_t)r1[1]),
                                                pack_bf16((uint16_t)r1[2], (uint16_t)r1[3]));
                    acc[t] = mfma_bf16(phi[s], bt, acc[t]);
                    acc[t] = mfma_bf16(plo[s], bt, acc[t]);
                }
            }
        }
        __syncthreads();  // the chunk's LDS is free for the next one
    };
    // the first chunk's rows behind the query's loads: they retire in order, so
    // the query images are made while the rows are in flight
    uint4 B0[STEPS];
    if (nchunks > 0) load_chunk(B0, 0);
#pragma unroll
    for (int r = 0; r < kUnits; ++r) {
        const int u = tid + 256 * r;
        if (u < STEPS * 64) {
            const float v[8] = {v4[r][0].x, v4[r][0].y, v4[r][0].z, v4[r][0].w,
                                v4[r][1].x, v4[r][1].y, v4[r][1].z, v4[r][1].w};
            split8(v, qhi[u], qlo[u]);
        }
    }
    __syncthreads();  // the query images
    for (int c = 0; c < nchunks; ++c) chunk(B0, c);
    // the partial record
    float* part = dptr<float>(a.part) + (size_t)rec * mla_part_floats(CD);
    if (wave == 0 && lane < 16) {
        part[lane] = m_run;
        part[16 + lane] = l_run;
    }
#pragma unroll
    for (int t = 0; t < kMlaMaxC / 64; ++t) {
        if (t < tpw) {
            const int col = wave * (CD >> 2) + 16 * t + n;
#pragma unroll
            for (int v = 0; v < 4; ++v) part[32 + (size_t)(4 * kb + v) * CD + col] = acc[t][v];
        }
    }
}

template <bool BAL>
__device__ __forceinline__ void mla_split(const MlaBatchArgs& a) {
    switch (a.qk_dim >> 5) {
        case 3: mla_split_body<3, BAL>(a); break;
        case 4: mla_split_body<4, BAL>(a); break;
        case 6: mla_split_body<6, BAL>(a); break;
        case 8: mla_split_body<8, BAL>(a); break;
        case 12: mla_split_body<12, BAL>(a); break;
        case 16: mla_split_body<16, BAL>(a); break;
        case 18: mla_split_body<18, BAL>(a); break;
        case 20: mla_split_body<20, BAL>(a); break;
        default: break;  // the host admits only these widths
    }
}

}  // namespace

extern "C" __global__ void __launch_bounds__(256) lp_mla_split(const MlaBatchArgs a) { mla_split<false>(a); }
extern "C" __global__ void __launch_bounds__(256) lp_mla_split_bal(const MlaBatchArgs a) { mla_split<true>(a); }

// ctx[b][h][d] from the splits' records.  Grid (heads, batch, c_dim / 64),
// 256 threads: the weights e^(m_s - M) / sum_s e^(m_s - M) l_s go to LDS once
// per workgroup, then thread (column d, group g) sums the splits s = g, g + 4,
// ... of its column (four loads in flight per step) and the four groups'
// sums meet in LDS.
namespace {

template <bool BAL>
__device__ __forceinline__ void mla_combine(const MlaBatchArgs& a) {
    __shared__ float wsh[kMlaMaxSplits];
    __shared__ float red[4];
    __shared__ float part_sum[4][64];
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
    const int CD = a.c_dim, PF = mla_part_floats(CD);
    const float* base = dptr<const float>(a.part) + (size_t)b * a.splits * PF;
    int splits = a.splits;
    int len = 0;
    if constexpr (BAL) len = mla_len(a);
    auto max_of = [&] { return tid < splits ? base[(size_t)tid * PF + h] : -INFINITY; };
    auto sum_of = [&] { return tid < splits ? base[(size_t)tid * PF + 16 + h] : 0.0f; };
    float ms = max_of(), ls = sum_of();  // the capacity's split, in flight beside the lengths
    if constexpr (BAL) {
        if (MlaShare sh; mla_share(a, len, sh)) {
            splits = __builtin_amdgcn_readlane(sh.splits, b);
            base = dptr<const float>(a.part) + (size_t)(__builtin_amdgcn_readlane(sh.incl, b) - splits) * PF;
            ms = max_of(), ls = sum_of();
        }
    }
    const float M = block_max(ms, red);
    const float w = ms == -INFINITY ? 0.0f : expf(ms - M);
    const float den = block_sum(w * ls, red);
    if (tid < splits) wsh[tid] = w / den;
    __syncthreads();
    const int d = blockIdx.z * 64 + (tid & 63), g = tid >> 6;
    const float* col = base + 32 + (size_t)h * CD + d;
    float num = 0.0f;
    int s = g;
    for (; s + 12 < splits; s += 16) {
        const float v0 = col[(size_t)s * PF], v1 = col[(size_t)(s + 4) * PF];
        const float v2 = col[(size_t)(s + 8) * PF], v3 = col[(size_t)(s + 12) * PF];
        num = __builtin_fmaf(wsh[s], v0, num);
        num = __builtin_fmaf(wsh[s + 4], v1, num);
        num = __builtin_fmaf(wsh[s + 8], v2, num);
        num = __builtin_fmaf(wsh[s + 12], v3, num);
    }
    for (; s < splits; s += 4) num = __builtin_fmaf(wsh[s], col[(size_t)s * PF], num);
    part_sum[g][tid & 63] = num;
    __syncthreads();
    if (g == 0)
        dptr<float>(a.ctx)[((size_t)b * a.heads + h) * CD + d] =
            (part_sum[0][tid] + part_sum[1][tid]) + (part_sum[2][tid] + part_sum[3][tid]);
}

}  // namespace

extern "C" __global__ void __launch_bounds__(256) lp_mla_combine(const MlaBatchArgs a) { mla_combine<false>(a); }
extern "C" __global__ void __launch_bounds__(256) lp_mla_combine_bal(const MlaBatchArgs a) { mla_combine<true>(a); }
