// Batches between decode and prefill: the grouped expert projections of more
// than 64 tokens that are too few per expert for the prefill GEMM, and the
// shared MLP of every batch above 64 tokens.
//
// With up to about 16 tokens per expert a layer still has to stream every
// expert's weights once (340 MB at H 2048 / I 768 / E 128), so HBM is the
// floor; what must not happen is a pass over the weights' arithmetic per few
// tokens.  The decode kernels spend a fifth of the matrix cores' rows on
// keeping four scales apart and take four tokens per pass (235 + 127 us for
// gate/up and down of 203 tokens, H 2048 / I 768 / 128 experts / top 8; 92 + 53
// here, traced).  Here a token tile is 16 tokens of one
// expert and an MFMA's K is exactly one 32-column sub-group:
//
//   v_mfma_f32_16x16x32_f16, A = 16 tokens, B = 16 weight rows.  The weights
//   enter as the stored nibbles n = q + 8 in the middle mantissa bits of
//   fp16, 1 + n / 64 (three shifts and four and-ors per eight weights); two
//   MFMAs of the tokens with the constant -72 / 64 seed the accumulators of
//   all four weight tiles, which leaves the sum of x q / 64.  The tokens are
//   fp16 hi + lo images (x 2^-e = hi + lo to 22 bits), so a product is exact
//   and a sub-group's sum is off by fp32 roundings only (those of sums about
//   15 times its size; the nibbles as subnormals, one AND each, come out of
//   the matrix core with 15 bits).  Then one fused multiply-add by the row's
//   scale: lane (n, kb) holds four tokens of row n, so a sub-group costs four
//   multiply-adds per 16 tokens.
//
// A wave owns four 16-row tiles (gate/up: 32 act columns, their gate and up
// rows, so a wave holds a whole sub-group of act and gives it its own
// exponent; down: 64 rows), a workgroup of four waves 128 act columns (256
// rows of down) for one block of up to 32 tokens of one expert (the tile
// list of the dispatch: a popular expert's blocks run side by side).
//
// Loads are by whole 128-byte lines: weights in pieces of 256 columns, one
// piece ahead in registers; a lane's 16 bytes are one sub-group of its row,
// and a 4 x 4 transposition over the four lanes of a row
// (v_permlane32_swap, v_permlane16_swap: four instructions per four
// sub-groups) turns them into one sub-group's words per lane.  The scales of
// 64 sub-groups sit in LDS, each row's line read once (read per stage from
// memory they cost as many cache lines as the weights).  Token rows pass
// through registers into two LDS slots of 128 columns, in operand order with
// a pad (no bank conflicts either way).
//
// act leaves gate/up as hi + lo images (2 I bytes each, no padding: together the
// bytes of the fp32 row that the other kernels keep) with one 16-bit exponent
// per (token, sub-group); down scales each staged piece to its row's largest
// exponent.
#include "lp_device.h"

using namespace lp;
using namespace lpk;

namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ ExpertEntry load_entry(uint64_t et, int u) {
    const LP_GLOBAL uint4* p = gptr<uint4>(et + (uint64_t)u * sizeof(ExpertEntry));
    const uint4 lo = p[0];
    ExpertEntry x{};
    x.blob = uniform_u64((uint64_t)lo.x | ((uint64_t)lo.y << 32));
    x.p0 = uni((int)lo.z);
    x.ntok = uni((int)lo.w);
    return x;
}

// A q4 word's stored nibbles n = q + 8 as fp16 1 + n / 64 in image order (0,
// 4, 1, 5, 2, 6, 3, 7).
__device__ __forceinline__ f16x8_t q4_word_to_f16(uint32_t b) {
    return __builtin_bit_cast(
        f16x8_t, u32x4_t{and_or(b << 4, 0x00F000F0u, 0x3C003C00u), and_or(b, 0x00F000F0u, 0x3C003C00u),
                         and_or(b >> 4, 0x00F000F0u, 0x3C003C00u), and_or(b >> 8, 0x00F000F0u, 0x3C003C00u)});
}

// Lane row kb's words 0..3 (x, y, z, w) are sub-group kb's: afterwards the
// four words are sub-groups 0..3's word kb.
__device__ __forceinline__ void transpose4(uint4& v) {
    const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    v = make_uint4(c[0], c[1], d[0], d[1]);
}

// 2^d as fp16 bits for d <= 0 (0 below 2^-24)
__device__ __forceinline__ uint32_t f16_pow2(int d) {
    return d >= -14 ? (uint32_t)(d + 15) << 10 : d >= -24 ? 1u << (d + 24) : 0u;
}

__device__ __forceinline__ uint32_t mul_f16x2(uint32_t v, f16x2_t f) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2_t, v) * f);
}

// Tokens tb .. tb + nt - 1 (nt <= 16 TT) of expert entry x against the
// wave's four row tiles from n0 (MODE 0: act columns, MODE 1: down rows).
template <int MODE, int RS, bool SV, int TT>
__device__ __forceinline__ void mid_tokens(const MidArgs& a, const ExpertEntry& x, int tb, int nt, int n0,
                                           uint8_t* lds) {
    const LayerView& L = a.L;
    const int K = MODE == 0 ? L.hidden : L.inter, NR = MODE == 0 ? L.inter : L.hidden;
    const int ng = K >> 5, nst = frag_ngp(K) >> 2, gpr = ng >> RS;
    const int lane = lane_id(), wave = uni((int)threadIdx.x >> 6), tid = (int)threadIdx.x;
    const int n = lane & 15, kb = lane >> 4;
    uint8_t* scl = lds;                                              // [4 waves x 64 rows] scales
    uint4* slots = reinterpret_cast<uint4*>(lds + kMidScaleBytes);   // [2][TT][hi, lo][kMidBlk]
    int* ex_l = reinterpret_cast<int*>(lds + kMidExOff);               // the tokens' exponents

    // --- token rows: thread (token tid / 16 of tile t, piece tid % 16 = word
    // p & 3 of sub-group p / 4) ---
    const int piece = tid & 15;
    int pos[TT], ex[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        pos[t] = x.p0 + tb + min(16 * t + (tid >> 4), nt - 1);  // rows past the block repeat its last token
        if (MODE == 0) pos[t] = gptr<int>(a.W.perm)[pos[t]] / L.top_k;
    }

    // --- weights: rows n of the wave's tiles; piece h of stage pair q is
    // sub-groups 8 q + 4 h + kb ---
    const uint32_t sbytes = (uint32_t)NR * (uint32_t)gpr * 2u;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(x.blob), (short)0,
        uni((int)((MODE == 0 ? max((uint32_t)L.gate_off, (uint32_t)L.up_off) : (uint32_t)L.down_off) + sbytes +
                  (uint32_t)NR * (uint32_t)ng * 16u)),
        kBufferWord3);
    auto row_of = [&](int t, int r) {  // row r of the wave's tile t
        return (uint32_t)min(MODE == 0 ? n0 + 16 * (t & 1) + r : n0 + 16 * t + r, NR - 1);
    };
    auto region = [&](int t) { return (uint32_t)(MODE == 0 ? (t < 2 ? L.gate_off : L.up_off) : L.down_off); };
    uint32_t wo[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) wo[t] = region(t) + sbytes + (row_of(t, n) * (uint32_t)ng + (uint32_t)kb) * 16u;
    struct Pair {
        uint4 w[2][4];
    };
    // stages past the last read what follows (zeros past the blob): unused
    auto load_w = [&](Pair& P, int q) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                P.w[h][t] = __builtin_bit_cast(
                    uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(wo[t] + 128u * (uint32_t)q + 64u * h), 0, 0));
    };
    // the scales of sub-groups 64 win .. of the wave's 64 rows, one f16 per
    // sub-group, kMidScaleRow bytes per row; read back by this wave alone
    auto load_scales = [&](int win) {
        uint8_t* dst = scl + wave * 64 * kMidScaleRow;
        if constexpr (SV) {
            // 16 lanes per row, 8 bytes (four sub-groups) each
            uint2 v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i)
                v[i] = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(
                               rs, (int)(region(i >> 2) + row_of(i >> 2, 4 * (i & 3) + kb) * (uint32_t)gpr * 2u +
                                         128u * (uint32_t)win + 8u * n), 0, 0));
#pragma unroll
            for (int i = 0; i < 16; ++i)
                *reinterpret_cast<uint2*>(dst + (4 * i + kb) * kMidScaleRow + 8 * n) = v[i];
        } else {
            // one sub-group per lane; zero past the last (its images are zero,
            // but a scale read past the row may be no number)
#pragma unroll 4
            for (int i = 0; i < 64; ++i) {
                const int g = 64 * win + lane;
                const uint32_t r = row_of(i >> 4, i & 15);
                const uint16_t v = __builtin_amdgcn_raw_buffer_load_b16(
                    rs, (int)(region(i >> 4) + (r * (uint32_t)gpr + (uint32_t)(min(g, ng - 1) >> RS)) * 2u), 0, 0);
                *reinterpret_cast<uint16_t*>(dst + i * kMidScaleRow + 2 * lane) = g < ng ? v : (uint16_t)0;
            }
        }
    };

    uint64_t row[TT];
    struct Rows {
        uint4 v[TT][2];
        int e[TT];
    };
    auto load_rows = [&](Rows& R, int st0) {
        const int st = min(st0, nst - 1);
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            // x's images end in zero sub-groups, act's rows in the next row:
            // pieces past their last sub-group repeat it, times zero
            const int g = 4 * st + (piece >> 2), gc = MODE == 1 && !SV ? min(g, ng - 1) : g;
            const uint64_t at = row[t] + 256u * (uint32_t)st - 64u * (uint32_t)(g - gc);
            R.v[t][0] = *gptr<uint4>(at);
            R.v[t][1] = *gptr<uint4>(at + a.lo_off);
            if (MODE == 1) R.e[t] = gc == g ? gptr<int16_t>(a.exps)[(size_t)pos[t] * ng + gc] : 16 * kExpNone;
        }
    };
    // into the slot (down: times 2^(sub-group exponent - row exponent))
    auto store_rows = [&](Rows& R, int slot) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t f = MODE == 1 ? f16_pow2(max(R.e[t] - ex[t], -127)) : 0u;
            const f16x2_t f2 = __builtin_bit_cast(f16x2_t, f | (f << 16));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint4 v = R.v[t][h];
                if (MODE == 1)
                    v = make_uint4(mul_f16x2(v.x, f2), mul_f16x2(v.y, f2), mul_f16x2(v.z, f2), mul_f16x2(v.w, f2));
                slots[((slot * TT + t) * 2 + h) * kMidBlk + piece * 17 + (tid >> 4)] = v;
            }
        }
    };

    Pair P0, P1;
    load_w(P0, 0);
    load_scales(0);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        row[t] = a.img + (uint64_t)(uint32_t)pos[t] * a.img_stride + 16u * (uint32_t)piece;
        if (MODE == 0) {
            ex[t] = gptr<int>(a.W.xexp)[pos[t]];
        } else {
            // the row's largest exponent over its 16 lanes
            int m = kExpNone;
            for (int c = piece; c < ng; c += 16) m = max(m, (int)gptr<int16_t>(a.exps)[(size_t)pos[t] * ng + c]);
#pragma unroll
            for (int o = 8; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
            ex[t] = m;
        }
    }
    Rows R;
    load_rows(R, 0);
    if (piece == 0)
#pragma unroll
        for (int t = 0; t < TT; ++t) ex_l[16 * t + (tid >> 4)] = ex[t];
    store_rows(R, 0);
    load_rows(R, 1);

    f32x4_t acc[4][TT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < TT; ++u) acc[t][u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // -72 / 64 in the weights' places
    const f16x8_t m8 = __builtin_bit_cast(f16x8_t, u32x4_t{0xBC80BC80u, 0xBC80BC80u, 0xBC80BC80u, 0xBC80BC80u});
    const uint8_t* srow = scl + (wave * 64 + n) * kMidScaleRow;

    auto compute = [&](uint4 (&w)[4], int st) {
#pragma unroll
        for (int t = 0; t < 4; ++t) transpose4(w[t]);
        const uint4* sl = slots + (st & 1) * TT * 2 * kMidBlk + kb * 17 + n;
        uint2 sc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            sc[t] = *reinterpret_cast<const uint2*>(srow + 16 * t * kMidScaleRow + 8 * (st & 15));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4_t seed[TT];
            f16x8_t hi[TT], lo[TT];
#pragma unroll
            for (int u = 0; u < TT; ++u) {
                hi[u] = __builtin_bit_cast(f16x8_t, sl[(2 * u) * kMidBlk + j * 68]);
                lo[u] = __builtin_bit_cast(f16x8_t, sl[(2 * u + 1) * kMidBlk + j * 68]);
                seed[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[u], m8, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                seed[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[u], m8, seed[u], 0, 0, 0);
            }
            f32x4_t c[4][TT];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f16x8_t q = q4_word_to_f16(j == 0 ? w[t].x : j == 1 ? w[t].y : j == 2 ? w[t].z : w[t].w);
#pragma unroll
                for (int u = 0; u < TT; ++u) {
                    c[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[u], q, seed[u], 0, 0, 0);
                    c[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[u], q, c[t][u], 0, 0, 0);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t sb = j < 2 ? sc[t].x : sc[t].y;
                const float s = f16_bits_to_f32((j & 1) ? sb >> 16 : sb & 0xffffu);
#pragma unroll
                for (int u = 0; u < TT; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[t][u][i] = __builtin_fmaf(s, c[t][u][i], acc[t][u][i]);
            }
        }
    };
    // Stage st's rows are in slot st & 1; the slot written here was last read
    // in stage st - 1, which every wave has left.  A stage pair's weights are
    // loaded at the start of the pair before it, after that stage's rows:
    // loads land in order, so the next wait for rows does not wait for them.
    auto step = [&](uint4 (&w)[4], int st, auto next) {
        __syncthreads();
        if (st > 0 && (st & 15) == 0) load_scales(st >> 4);  // the wave's own rows: no barrier
        store_rows(R, (st + 1) & 1);                         // past the last stage: stale rows, unread
        load_rows(R, st + 2);
        next();
        compute(w, st);
    };
    auto none = [] {};
    for (int q = 0; 2 * q < nst; q += 2) {
        step(P0.w[0], 2 * q, [&] { load_w(P1, q + 1); });
        if (2 * q + 1 < nst) step(P0.w[1], 2 * q + 1, none);
        if (2 * q + 2 < nst) {
            step(P1.w[0], 2 * q + 2, [&] { load_w(P0, q + 2); });
            if (2 * q + 3 < nst) step(P1.w[1], 2 * q + 3, none);
        }
    }

    // --- epilogues: lane (n, kb) holds tokens 16 u + 4 kb + i of row n ---
    if constexpr (MODE == 0) {
        // act = silu(gate) up of the wave's sub-group, columns n0 .. n0 + 31:
        // the wave's tiles through LDS (its own part of the token slots, free
        // after the barrier), so that lane (token n, word kb) finishes one
        // image word: eight columns, the exponent over the token's four lanes
        __syncthreads();
        float* ep = reinterpret_cast<float*>(slots) + wave * 64 * kMidEpRow;  // [64 rows][16 tokens]
        const bool live = n0 < NR;
#pragma unroll
        for (int u = 0; u < TT; ++u) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                *reinterpret_cast<f32x4_t*>(ep + (16 * t + n) * kMidEpRow + 4 * kb) = acc[t][u];
            const int tt = 16 * u + n, e = ex_l[tt] + 6;  // the weights' 1 / 64
            float v[8], m = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float g = __builtin_ldexpf(ep[(8 * kb + i) * kMidEpRow + n], e);
                const float up = __builtin_ldexpf(ep[(32 + 8 * kb + i) * kMidEpRow + n], e);
                v[i] = live ? g / (1.0f + expf(-g)) * up : 0.0f;
                m = fmaxf(m, fabsf(v[i]));
            }
            m = fmaxf(m, shfl_xor(m, 16));
            m = fmaxf(m, shfl_xor(m, 32));
            const int ae = m > 0.0f ? h16_exp(m) : 0;
            if (tt < nt && live) {
                float r[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float w = __builtin_ldexpf(v[i], -ae);
                    r[i] = w - (float)(_Float16)w;
                }
                const size_t p = (size_t)(x.p0 + tb + tt);
                LP_GLOBAL uint4* o = gptr_w<uint4>(a.out + p * (4u * (uint32_t)NR) + 2u * (uint32_t)n0);
                o[kb] = h16_word(v, ae);
                o[(NR >> 3) + kb] = h16_word(r, 0);
                if (kb == 0)
                    gptr_w<int16_t>(a.exps)[p * (size_t)(NR >> 5) + (n0 >> 5)] = (int16_t)(m > 0.0f ? ae : kExpNone);
            }
        }
    } else {
        LP_GLOBAL float* y = gptr_w<float>(a.out);
#pragma unroll
        for (int u = 0; u < TT; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int tt = 16 * u + 4 * kb + i;
                const int e = ex_l[tt] + 6;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int r = n0 + 16 * t + n;
                    if (tt < nt && r < NR)
                        y[(size_t)(x.p0 + tb + tt) * NR + r] = __builtin_ldexpf(acc[t][u][i], e);
                }
            }
    }
}

// Tokens tb .. tb + nt - 1 of a routed expert without a slot: zeros (gate/up:
// zero images, no exponent).
template <int MODE>
__device__ __forceinline__ void mid_missing(const MidArgs& a, const ExpertEntry& x, int chunk, int tb, int nt) {
    if (threadIdx.x == 0) atomicOr(gptr_w<int>(a.W.meta) + 1, kErrMissingExpert);
    const int NR = MODE == 0 ? a.L.inter : a.L.hidden;
    for (int t = tb; t < tb + nt; ++t) {
        const size_t p = (size_t)(x.p0 + t);
        if (MODE == 0) {
            const int ng = NR >> 5, g = 4 * chunk + (int)(threadIdx.x & 15) / 4;
            // four sub-groups of 64 bytes, hi and lo
            if (threadIdx.x < 32 && g < ng)
                gptr_w<uint4>(a.out + p * (4u * (uint32_t)NR) + (threadIdx.x >> 4) * 2u * (uint32_t)NR +
                              256u * (uint32_t)chunk)[threadIdx.x & 15] = make_uint4(0u, 0u, 0u, 0u);
            if (threadIdx.x < 4 && 4 * chunk + (int)threadIdx.x < ng)
                gptr_w<int16_t>(a.exps)[p * (size_t)ng + 4 * chunk + threadIdx.x] = (int16_t)kExpNone;
        } else {
            const int r = kMidRows * chunk + (int)threadIdx.x;
            if (r < NR) gptr_w<float>(a.out)[p * NR + r] = 0.0f;
        }
    }
}

template <int MODE, int RS, bool SV>
__device__ __forceinline__ void mid_body(const MidArgs& a) {
    extern __shared__ __align__(16) uint8_t lds[];
    // this workgroup's block of an expert's tokens: from the tile list, or
    // (no list) block ti of entry 0
    const int ti = (int)blockIdx.x / a.chunks, chunk = (int)blockIdx.x - ti * a.chunks;
    int u = 0, b = ti;
    if (a.tiles) {
        const int count = gptr<int>(a.W.meta)[2], tv = uni(gptr<int>(a.tiles)[ti]);
        if (ti >= uni(count)) return;
        u = tv >> 16, b = tv & 0xffff;
    }
    const ExpertEntry x = load_entry(a.W.et, u);
    const int tb = kMidToks * b, nt = min(kMidToks, x.ntok - tb);
    if (nt <= 0) return;
    if (x.blob == 0) {
        mid_missing<MODE>(a, x, chunk, tb, nt);
        return;
    }
    const int wave = uni((int)threadIdx.x >> 6);
    const int n0 = MODE == 0 ? kActChunk * chunk + 32 * wave : kMidRows * chunk + 64 * wave;
    if (nt <= 16)
        mid_tokens<MODE, RS, SV, 1>(a, x, tb, nt, n0, lds);
    else
        mid_tokens<MODE, RS, SV, 2>(a, x, tb, nt, n0, lds);
}

}  // namespace

// Group 32 with whole 8-byte scale pieces per stage (cols a multiple of 128);
// other groups and widths read their scales one by one.
extern "C" __global__ void __launch_bounds__(256, 2) lp_mid_gateup(const MidArgs a) { mid_body<0, 0, true>(a); }
extern "C" __global__ void __launch_bounds__(256, 2) lp_mid_down(const MidArgs a) { mid_body<1, 0, true>(a); }

#define LP_MID(mode)                                      \
    switch (ilog2_pow2(a.L.group >> 5)) {                 \
        case 0: mid_body<mode, 0, false>(a); break;       \
        case 1: mid_body<mode, 1, false>(a); break;       \
        default: mid_body<mode, 2, false>(a); break;      \
    }
extern "C" __global__ void __launch_bounds__(256, 2) lp_mid_gateup_rs(const MidArgs a) { LP_MID(0) }
extern "C" __global__ void __launch_bounds__(256, 2) lp_mid_down_rs(const MidArgs a) { LP_MID(1) }
