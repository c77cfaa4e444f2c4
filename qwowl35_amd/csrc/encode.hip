// Weight producers: fp32 matrix -> GF4 / GF2 / q8_0 / Q4_K / Q5_K / Q6_K / F16 tensor bytes, on the GPU.
//
// GF4 is the reference packer pack_gf4_prepared(rows, scale_search=False)
// (tools/qw35_cook_common.py:83-119), including the optional AWQ column
// multiply that pack_ffn_gf4 applies before packing (:182-199, the multiply
// at :198).  Every step is an IEEE fp32 / binary16 operation with the same
// rounding as the numpy statement, so the words are bit-identical:
//   gmax  = first element of the 8-group with the largest |x|, with its sign
//   b     = (bits(fp16_rne(gmax)) + 0x80) >> 8          (e5m2 byte, :48-51)
//   s     = fp16(b << 8)                                (:54-56)
//   q_raw = clip(rint(fl(x / s) * -4 + 4), 0, 7), 0 where s == 0   (:67-80)
//   word  = b | sum_i (q_raw_i ^ 4) << (8 + 3 i)        (:113-118)
// q8_0, Q4_K, Q5_K and Q6_K have no encoder in the reference (it reads them through
// the external gguf-py); these are this library's own min/max encoders, the GPU
// statement of the ones the tests use, producing valid GGUF blocks.
//
// Inputs must be finite: NaN ordering in numpy's argmax and its float->int
// casts are platform behaviour, not part of the format.
#include "qw35_device.h"
#include "qw35_kernels.h"

namespace qw35 {
namespace {

__device__ __forceinline__ uint32_t f32_to_f16_bits(float v) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

// i % m; a 64-bit remainder is some 50 instructions, so it is taken only where
// i needs it (12288x4096 with a column scale, us: GF4 44.9 -> 42.3, Q4_K 64.0
// -> 60.3, GF2 52.8 -> 47.3).
__device__ __forceinline__ uint32_t mod_u64(uint64_t i, uint32_t m) {
    return (i >> 32) == 0 ? (uint32_t)i % m : (uint32_t)(i % m);
}

// Grid-stride loops keep the grid at a fixed size for any tensor.
constexpr int kEncodeThreads = 256;
constexpr int kEncodeBlocks = 2048;

// One thread per GF4 word (8 consecutive columns of a row).
__global__ __launch_bounds__(kEncodeThreads) void gf4_pack_kernel(const float* __restrict__ src,
                                                                  const float* __restrict__ col_scale,
                                                                  uint32_t* __restrict__ dst, uint64_t n_words,
                                                                  uint32_t words_per_row) {
    for (uint64_t i = (uint64_t)blockIdx.x * kEncodeThreads + threadIdx.x; i < n_words;
         i += (uint64_t)gridDim.x * kEncodeThreads) {
        const float4_t lo = *reinterpret_cast<const float4_t*>(src + 8 * i);
        const float4_t hi = *reinterpret_cast<const float4_t*>(src + 8 * i + 4);
        float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        if (col_scale) {
            const uint32_t c0 = 8u * mod_u64(i, words_per_row);
            const float4_t s0 = *reinterpret_cast<const float4_t*>(col_scale + c0);
            const float4_t s1 = *reinterpret_cast<const float4_t*>(col_scale + c0 + 4);
            const float s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __fmul_rn(v[j], s[j]);
        }
        int best = 0;
        float best_abs = fabsf(v[0]);
#pragma unroll
        for (int j = 1; j < 8; ++j) {
            if (fabsf(v[j]) > best_abs) {  // strict: the first maximum wins
                best_abs = fabsf(v[j]);
                best = j;
            }
        }
        float gmax = v[0];
#pragma unroll
        for (int j = 1; j < 8; ++j)
            if (j == best) gmax = v[j];
        const uint32_t b = ((f32_to_f16_bits(gmax) + 0x80u) >> 8) & 0xFFu;
        const float s = f16_bits_to_f32(b << 8);
        uint32_t word = b;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float ratio = (s != 0.0f) ? __fdiv_rn(v[j], s) : 0.0f;
            const float t = __fadd_rn(__fmul_rn(ratio, -4.0f), 4.0f);
            const float q = fminf(fmaxf(rintf(t), 0.0f), 7.0f);
            word |= (((uint32_t)q) ^ 4u) << (8 + 3 * j);
        }
        dst[i] = word;
    }
}

// Super-block encoders (GF2, Q4_K, Q5_K, Q6_K; q8_0 likewise): one wave per
// 256-column super-block, four consecutive columns per lane, so a super-block
// is one coalesced 1 KB load, its group maxima are lane reductions and its
// packed words one or two narrow stores; kSuperUnroll super-blocks' loads are
// in flight per wave.  The encoders are bound by their fp32 reads and, for the
// k-quants, VALU issue (the sub-blocks' arithmetic, the rounding of the codes).
// A thread per super-block (1 KB apart, three passes over its columns) took
// 1061 us for Q4_K 12288x4096 with a column scale (0.22 TB/s); this form takes
// 52.5 (4.4 TB/s; GF2 45, Q5_K 54, Q6_K 53).
constexpr int kSuperUnroll = 4;
constexpr int kEncodeWaves = kEncodeThreads / 64;

// The lane's four columns of super-blocks i0 .. i0 + kSuperUnroll - 1
// (clamped to the last one), times the column scale.
__device__ __forceinline__ void load_super(const float* __restrict__ src, const float* __restrict__ col_scale,
                                           uint64_t i0, uint64_t n_blocks, uint32_t blocks_per_row, int lane,
                                           float (&v)[kSuperUnroll][4]) {
    float4_t x[kSuperUnroll], s[kSuperUnroll];
#pragma unroll
    for (int u = 0; u < kSuperUnroll; ++u) {
        const uint64_t i = i0 + u < n_blocks ? i0 + u : n_blocks - 1;
        x[u] = *reinterpret_cast<const float4_t*>(src + 256 * i + 4 * lane);
        s[u] = float4_t{1.0f, 1.0f, 1.0f, 1.0f};
        if (col_scale)
            s[u] = *reinterpret_cast<const float4_t*>(col_scale + 256u * mod_u64(i, blocks_per_row) + 4 * lane);
    }
#pragma unroll
    for (int u = 0; u < kSuperUnroll; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) v[u][q] = __fmul_rn(x[u][q], s[u][q]);  // (a product needs no canonicalising max)
}

template <int CTRL>
__device__ __forceinline__ float dpp_fmax(float v) {
    return fmaxf(v, dpp_f32<CTRL>(v));
}
template <int CTRL>
__device__ __forceinline__ float dpp_fmin(float v) {
    return fminf(v, dpp_f32<CTRL>(v));
}

// 1 / d for rint_div4, or NaN where only the divide is sure to round right: a
// quotient of n_max / d above 40 in magnitude or a divisor outside rcp's
// accurate range.  n_max: the largest |n| that is divided by d.  d != 0.
__device__ __forceinline__ float sure_rcp(float d, float n_max) {
    const float inv = __builtin_amdgcn_rcpf(d);
    const bool sure = n_max * fabsf(inv) < 40.0f && fabsf(d) > 0x1p-100f && fabsf(d) < 0x1p+100f;
    return sure ? inv : __builtin_nanf("");
}

// r[q] = rint(fl(n[q] / d) * mul + add) in the IEEE steps that the formats
// state, without an IEEE divide where it cannot matter.  t = n * inv has a
// relative error of at most 2^-22 against the rounded quotient (rcp within one
// ulp, two roundings, the quotient's own), the affine form three more roundings
// of 2^-24: below 2^-15 for |t| < 64, so both round to the same integer unless
// t lies within 2^-14 of a tie.  Only a wave that holds such a lane (or a NaN
// inv) divides, by divisor(): 3% of them with 256 codes (a band of 0.001
// sent 40% there).  (Q4_K 12288x4096 with a column scale: 87.5 -> 64.0 us with
// this and the shared sub-block arithmetic of k_quantize_kernel; the narrower
// band 65.6 -> 60.6, Q5_K 67.5 -> 63.0, GF2 47.7 -> 45.2)
template <bool AFFINE, typename D>
__device__ __forceinline__ void rint_div4(const float (&n)[4], float inv, D&& divisor, float (&r)[4]) {
    float off[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float t = n[q] * inv;
        if (AFFINE) t = __builtin_fmaf(t, 1.5f, 1.5f);
        r[q] = rintf(t);
        off[q] = fabsf(t - r[q]);
    }
    // (a NaN inv makes all four NaN, and fmaxf of NaNs is NaN)
    const float far = fmaxf(fmaxf(off[0], off[1]), fmaxf(off[2], off[3]));
    if (__any(!(far < 0.5f - 0x1p-14f))) {
        const float d = divisor();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float t = __fdiv_rn(n[q], d);
            r[q] = rintf(AFFINE ? __fadd_rn(__fmul_rn(t, 1.5f), 1.5f) : t);
        }
    }
}

// Four whole numbers in [0, 255] -> one per byte.
__device__ __forceinline__ uint32_t pack_u8(const float (&r)[4]) {
    uint32_t code = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) code = __builtin_amdgcn_cvt_pk_u8_f32(r[q], q, code);
    return code;
}

// GF2 super-blocks (256 columns = 16 groups of 16; this library's encoder, the
// statement of oracle gf2_quantize):
//   b = e5m2(max |x|) (fp16 RNE, low byte rounded half-up), s = fp16(b << 8)
//   t = x / s (0 where s == 0), q = clip(rint(t * 1.5 + 1.5), 0, 3)
// written as the reference's super-block: 16 code words (code i of word w in
// bits 2i, 2i+1 for column 16w + i) then the 16 scale bytes
// (qw35-server/src/metal/qw35_gf2.metal:1-17).  A group is one quad of lanes.
__global__ __launch_bounds__(kEncodeThreads) void gf2_pack_kernel(const float* __restrict__ src,
                                                                  const float* __restrict__ col_scale,
                                                                  uint8_t* __restrict__ dst, uint64_t n_blocks,
                                                                  uint32_t blocks_per_row) {
    const int lane = threadIdx.x & 63;
    const uint64_t wave = (uint64_t)blockIdx.x * kEncodeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint64_t i0 = wave * kSuperUnroll; i0 < n_blocks; i0 += (uint64_t)gridDim.x * kEncodeWaves * kSuperUnroll) {
        float v[kSuperUnroll][4];
        load_super(src, col_scale, i0, n_blocks, blocks_per_row, lane, v);
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            if (i0 + u >= n_blocks) break;
            float amax = fmaxf(fmaxf(fabsf(v[u][0]), fabsf(v[u][1])), fmaxf(fabsf(v[u][2]), fabsf(v[u][3])));
            amax = dpp_fmax<kDppQuadXor1>(amax);
            amax = fmaxf(dpp_fmax<kDppQuadXor2>(amax), 0.0f);  // (a group of NaN: zero, also below)
            const uint32_t b = ((f32_to_f16_bits(amax) + 0x80u) >> 8) & 0xFFu;
            const float s = f16_bits_to_f32(b << 8);
            float r[4];
            const float div = s != 0.0f ? s : 1.0f;
            rint_div4<true>(v[u], sure_rcp(div, amax), [&] { return div; }, r);
            uint32_t word = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q)  // s == 0: t = 0, code rint(1.5) = 2
                word |= (s != 0.0f ? (uint32_t)fminf(fmaxf(r[q], 0.0f), 3.0f) : 2u) << (2 * q);
            word <<= 8 * (lane & 3);
            word |= dpp_u32<kDppQuadXor1>(word);
            word |= dpp_u32<kDppQuadXor2>(word);
            if ((lane & 3) == 0) {
                uint8_t* blk = dst + 80 * (i0 + u);
                reinterpret_cast<uint32_t*>(blk)[lane >> 2] = word;
                blk[64 + (lane >> 2)] = (uint8_t)b;
            }
        }
    }
}

// q8_0 blocks (32 columns, 8 lanes each): d = max|x| / 127, q = round_half_away(x * (1/d)).
// Four columns per lane as above, kSuperUnroll groups of eight blocks per wave
// and round; a row is any number of blocks, so blocks are counted over the
// matrix.  Bound by the fp32 reads; a thread per block (128 bytes apart, 17
// two-byte stores) took 82.7 us for 12288x4096 with a column scale, this form
// 52.0 (4.9 TB/s); 4096x4096 26.8 -> 17.2.
__global__ __launch_bounds__(kEncodeThreads) void q8_0_quantize_kernel(const float* __restrict__ src,
                                                                       const float* __restrict__ col_scale,
                                                                       uint8_t* __restrict__ dst, uint64_t n_blocks,
                                                                       uint32_t blocks_per_row) {
    // 34-byte blocks: 2-byte aligned
    struct __attribute__((packed, aligned(2))) Word {
        uint32_t v;
    };
    const int lane = threadIdx.x & 63;
    const uint64_t wave = (uint64_t)blockIdx.x * kEncodeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t per_round = (uint64_t)gridDim.x * kEncodeWaves * 8 * kSuperUnroll;
    for (uint64_t i0 = wave * 8 * kSuperUnroll; i0 < n_blocks; i0 += per_round) {
        float4_t x[kSuperUnroll], s[kSuperUnroll];
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            uint64_t i = i0 + 8 * u + (lane >> 3);
            i = i < n_blocks ? i : n_blocks - 1;
            x[u] = *reinterpret_cast<const float4_t*>(src + 32 * i + 4 * (lane & 7));
            if (col_scale)
                s[u] = *reinterpret_cast<const float4_t*>(col_scale + 32u * mod_u64(i, blocks_per_row) + 4 * (lane & 7));
        }
        // lane l keeps the maximum of its block of group l % 4, so the two
        // divides run once for the four groups
        static_assert(kSuperUnroll == 4, "one lane of a quad per group");
        float v[kSuperUnroll][4];
        float amax_u = 0.0f;
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) v[u][q] = col_scale ? __fmul_rn(x[u][q], s[u][q]) : x[u][q];
            float amax = fmaxf(fmaxf(fabsf(v[u][0]), fabsf(v[u][1])), fmaxf(fabsf(v[u][2]), fabsf(v[u][3])));
            amax = dpp_fmax<kDppRowHalfMirror>(dpp_fmax<kDppQuadXor2>(dpp_fmax<kDppQuadXor1>(amax)));
            amax_u = (lane & 3) == u ? amax : amax_u;
        }
        const float d_u = __fdiv_rn(fmaxf(amax_u, 0.0f), 127.0f);
        const float inv_u = (d_u != 0.0f) ? __fdiv_rn(1.0f, d_u) : 0.0f;
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            const int from = (lane & ~3) | u;
            const float d = __shfl(d_u, from), inv = __shfl(inv_u, from);
            uint32_t code = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float sc = __fmul_rn(v[u][q], inv);
                const float r = fminf(fmaxf(truncf(__fadd_rn(sc, copysignf(0.5f, sc))), -127.0f), 127.0f);
                code |= ((uint32_t)(int)r & 0xFFu) << (8 * q);
            }
            const uint64_t i = i0 + 8 * u + (lane >> 3);
            if (i < n_blocks) {
                uint8_t* blk = dst + 34 * i;
                reinterpret_cast<Word*>(blk + 2 + 4 * (lane & 7))->v = code;
                if ((lane & 7) == 0) *reinterpret_cast<uint16_t*>(blk) = (uint16_t)f32_to_f16_bits(d);
            }
        }
    }
}

// Q4_K (Q5_K) super-blocks (256 columns, 8 sub-blocks of 32: 8 lanes each),
// with L = 15 (31) code levels:
//   lo_j = min(min(x), 0), hi_j = max(x), scale_j = (hi_j - lo_j) / L, min_j = -lo_j
//   d = fp16(max_j scale_j / 63), dmin = fp16(max_j min_j / 63)
//   sc_j = clip(rint(scale_j / d), 0, 63), m_j = clip(rint(min_j / dmin), 0, 63)
//   q = clip(rint((x + dmin*m_j) / (d*sc_j)), 0, L)
// with the 12-byte 6-bit scale packing of get_scale_min_k4
// (qw35-server/src/metal/qw35_matvec.metal:2-12) and the nibble layout
// qs[32c + l] = q[64c + l] | q[64c + 32 + l] << 4 (low nibbles only for Q5_K,
// whose qs starts at byte 48; bit 4 of q for element 32j + l is bit j of qh[l],
// qh at byte 16; qw35_types.metal:9-15).
template <bool Q5>
__global__ __launch_bounds__(kEncodeThreads) void k_quantize_kernel(const float* __restrict__ src,
                                                                    const float* __restrict__ col_scale,
                                                                    uint8_t* __restrict__ dst, uint64_t n_blocks,
                                                                    uint32_t blocks_per_row) {
    constexpr float kLevels = Q5 ? 31.0f : 15.0f;
    constexpr int kBlockBytes = Q5 ? 176 : 144;
    constexpr int kQs = Q5 ? 48 : 16;
    const int lane = threadIdx.x & 63;
    const int j = lane >> 3;  // the lane's sub-block
    const uint64_t wave = (uint64_t)blockIdx.x * kEncodeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint64_t i0 = wave * kSuperUnroll; i0 < n_blocks; i0 += (uint64_t)gridDim.x * kEncodeWaves * kSuperUnroll) {
        float v[kSuperUnroll][4];
        load_super(src, col_scale, i0, n_blocks, blocks_per_row, lane, v);
        // lo and hi of each sub-block over its 8 lanes; lane l then keeps those
        // of super-block l % 4, so the sub-block arithmetic (five divides) runs
        // once for the four super-blocks
        static_assert(kSuperUnroll == 4, "one lane of a quad per super-block");
        float lo_u = 0.0f, hi_u = 0.0f;
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            float lo = fminf(fminf(v[u][0], v[u][1]), fminf(v[u][2], v[u][3]));
            float hi = fmaxf(fmaxf(v[u][0], v[u][1]), fmaxf(v[u][2], v[u][3]));
            lo = dpp_fmin<kDppRowHalfMirror>(dpp_fmin<kDppQuadXor2>(dpp_fmin<kDppQuadXor1>(lo)));
            hi = dpp_fmax<kDppRowHalfMirror>(dpp_fmax<kDppQuadXor2>(dpp_fmax<kDppQuadXor1>(hi)));
            lo_u = (lane & 3) == u ? lo : lo_u;
            hi_u = (lane & 3) == u ? hi : hi_u;
        }
        lo_u = fminf(lo_u, 0.0f);
        hi_u = fmaxf(hi_u, -__builtin_inff());  // (a sub-block of NaN: the maximum of no elements)
        const float scale = __fdiv_rn(__fsub_rn(hi_u, lo_u), kLevels);
        const float mins = -lo_u;
        float smax = scale, mmax = mins;
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) {
            smax = fmaxf(smax, __shfl_xor(smax, o));
            mmax = fmaxf(mmax, __shfl_xor(mmax, o));
        }
        const uint32_t d_bits_u = f32_to_f16_bits(__fdiv_rn(smax, 63.0f));
        const uint32_t dmin_bits_u = f32_to_f16_bits(__fdiv_rn(mmax, 63.0f));
        const float df = f16_bits_to_f32(d_bits_u);
        const float dminf = f16_bits_to_f32(dmin_bits_u);
        const float a = (df != 0.0f) ? rintf(__fdiv_rn(scale, df)) : 0.0f;
        const float m = (dminf != 0.0f) ? rintf(__fdiv_rn(mins, dminf)) : 0.0f;
        const uint32_t sc_u = (uint32_t)fminf(fmaxf(a, 0.0f), 63.0f);
        const uint32_t mq_u = (uint32_t)fminf(fmaxf(m, 0.0f), 63.0f);
        const float step_u = __fmul_rn(df, (float)sc_u);
        const float offs_u = __fmul_rn(dminf, (float)mq_u);
        const float div_u = step_u != 0.0f ? step_u : 1.0f;
        const float inv_u = sure_rcp(div_u, fmaxf(fabsf(__fadd_rn(lo_u, offs_u)), fabsf(__fadd_rn(hi_u, offs_u))));
        const unsigned long long zero = __ballot(step_u == 0.0f);
        // headers: lane u of the first quad gathers those of super-block u
        // (assembled per super-block, with its reciprocal and the largest
        // quotient per lane: Q4_K 12288x4096 60.8 us, now 52.5; Q5_K 62.5 / 54.2).
        // Sub-block j < 4 gives scale bytes j, j + 4 and j + 8, of its own
        // scale and min and those of sub-block j + 4 (32 lanes on).
        const uint32_t both = sc_u | (mq_u << 8);
        const uint32_t upper = (uint32_t)__shfl_xor((int)both, 32);
        const uint32_t s1 = upper & 63u, m1 = upper >> 8;
        uint32_t w[3] = {(sc_u | ((s1 >> 4) << 6)) << (8 * (j & 3)), (mq_u | ((m1 >> 4) << 6)) << (8 * (j & 3)),
                         ((s1 & 15u) | ((m1 & 15u) << 4)) << (8 * (j & 3))};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            w[q] |= (uint32_t)__shfl_xor((int)w[q], 8);
            w[q] |= (uint32_t)__shfl_xor((int)w[q], 16);
        }
        if (lane < kSuperUnroll && i0 + lane < n_blocks)  // 144- or 176-byte blocks: 16-byte aligned
            *reinterpret_cast<uint4_t*>(dst + kBlockBytes * (i0 + lane)) =
                uint4_t{d_bits_u | (dmin_bits_u << 16), w[0], w[1], w[2]};
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            if (i0 + u >= n_blocks) break;
            const int from = (lane & ~3) | u;  // this sub-block's lane of super-block u
            const float inv = __shfl(inv_u, from), offs = __shfl(offs_u, from);
            float n[4], r[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) n[q] = __fadd_rn(v[u][q], offs);
            rint_div4<false>(n, inv, [&] { return __shfl(div_u, from); }, r);
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = fminf(fmaxf(r[q], 0.0f), kLevels);
            const uint32_t code = (zero >> from) & 1 ? 0u : pack_u8(r);  // the lane's four codes
            uint8_t* blk = dst + kBlockBytes * (i0 + u);
            // nibbles: sub-blocks 2c and 2c + 1 are 8 lanes apart
            const uint32_t other = (uint32_t)__shfl_xor((int)code, 8);
            if ((lane & 8) == 0)
                reinterpret_cast<uint32_t*>(blk + kQs)[8 * (lane >> 4) + (lane & 7)] =
                    (code & 0x0F0F0F0Fu) | ((other & 0x0F0F0F0Fu) << 4);
            if constexpr (Q5) {  // qh: bit j of byte l, over the eight sub-blocks
                uint32_t qh = ((code >> 4) & 0x01010101u) << j;
#pragma unroll
                for (int o = 8; o < 64; o <<= 1) qh |= (uint32_t)__shfl_xor((int)qh, o);
                if (lane < 8) reinterpret_cast<uint32_t*>(blk + 16)[lane] = qh;
            }
        }
    }
}

// Q6_K super-blocks (256 columns, 16 sub-blocks of 16: one quad of lanes each),
// the statement of oracle q6_k_quantize:
//   sub_s = max|x| / 31, d = fp16(max_s sub_s / 127), sc_s = clip(rint(sub_s / d), 0, 127)
//   q = clip(rint(x / (d * sc_s)), -32, 31) + 32
// stored as ggml lays Q6_K out (qw35_types.metal:17-22): element
// 128h + 32g + l has its low nibble in ql[64h + 32(g&1) + l] (high nibble for
// g >= 2) and its top two bits at bit 2g of qh[32h + l].  Super-blocks are
// 210 bytes (2-byte aligned), so a word leaves as two 16-bit stores.  With the
// sub-block arithmetic per super-block instead of once for four, and the wider
// band of rint_div4, 12288x4096 with a column scale took 72.6 us, now 53.1.
__global__ __launch_bounds__(kEncodeThreads) void q6_k_quantize_kernel(const float* __restrict__ src,
                                                                       const float* __restrict__ col_scale,
                                                                       uint8_t* __restrict__ dst, uint64_t n_blocks,
                                                                       uint32_t blocks_per_row) {
    const int lane = threadIdx.x & 63;
    const uint64_t wave = (uint64_t)blockIdx.x * kEncodeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto store4 = [](uint8_t* p, uint32_t w) {
        reinterpret_cast<uint16_t*>(p)[0] = (uint16_t)w;
        reinterpret_cast<uint16_t*>(p)[1] = (uint16_t)(w >> 16);
    };
    for (uint64_t i0 = wave * kSuperUnroll; i0 < n_blocks; i0 += (uint64_t)gridDim.x * kEncodeWaves * kSuperUnroll) {
        float v[kSuperUnroll][4];
        load_super(src, col_scale, i0, n_blocks, blocks_per_row, lane, v);
        // lane l keeps the sub-block maximum of super-block l % 4, so the
        // sub-block arithmetic (three divides) runs once for the four
        static_assert(kSuperUnroll == 4, "one lane of a quad per super-block");
        float amax_u = 0.0f;
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            float amax = fmaxf(fmaxf(fabsf(v[u][0]), fabsf(v[u][1])), fmaxf(fabsf(v[u][2]), fabsf(v[u][3])));
            amax = dpp_fmax<kDppQuadXor2>(dpp_fmax<kDppQuadXor1>(amax));
            amax_u = (lane & 3) == u ? amax : amax_u;
        }
        amax_u = fmaxf(amax_u, 0.0f);
        const float sub = __fdiv_rn(amax_u, 31.0f);
        float smax = sub;
#pragma unroll
        for (int o = 4; o < 64; o <<= 1) smax = fmaxf(smax, __shfl_xor(smax, o));
        const uint32_t d_bits_u = f32_to_f16_bits(__fdiv_rn(smax, 127.0f));
        const float df = f16_bits_to_f32(d_bits_u);
        const float a = (df != 0.0f) ? rintf(__fdiv_rn(sub, df)) : 0.0f;
        const float scq = fminf(fmaxf(a, 0.0f), 127.0f);
        const float step_u = __fmul_rn(df, scq);
        const float div_u = step_u != 0.0f ? step_u : 1.0f;
        const float inv_u = sure_rcp(div_u, amax_u);
        // scale and fp16 scale of the super-block; bit 8: all codes are zero
        const uint32_t sd_u = (uint32_t)(int)scq | (step_u == 0.0f ? 256u : 0u) | (d_bits_u << 16);
#pragma unroll
        for (int u = 0; u < kSuperUnroll; ++u) {
            if (i0 + u >= n_blocks) break;
            const int from = (lane & ~3) | u;  // this sub-block's lane of super-block u
            const float inv = __shfl(inv_u, from);
            const uint32_t sd = (uint32_t)__shfl((int)sd_u, from);
            float r[4];
            rint_div4<false>(v[u], inv, [&] { return __shfl(div_u, from); }, r);
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = fminf(fmaxf(r[q], -32.0f), 31.0f) + 32.0f;
            const uint32_t code = (sd & 256u) ? 0x20202020u : pack_u8(r);  // the lane's four codes
            uint8_t* blk = dst + 210 * (i0 + u);
            // lane = 32h + 8g + l / 4: groups g and g + 2 share the bytes of ql, all four those of qh
            const int h = lane >> 5, g = (lane >> 3) & 3, l = 4 * (lane & 7);
            const uint32_t other = (uint32_t)__shfl_xor((int)code, 16);
            uint32_t qh = ((code >> 4) & 0x03030303u) << (2 * g);
            qh |= (uint32_t)__shfl_xor((int)qh, 8);
            qh |= (uint32_t)__shfl_xor((int)qh, 16);
            if (g < 2) store4(blk + 64 * h + 32 * g + l, (code & 0x0F0F0F0Fu) | ((other & 0x0F0F0F0Fu) << 4));
            if (g == 2) store4(blk + 128 + 32 * h + l, qh);
            if ((lane & 3) == 0) blk[192 + (lane >> 2)] = (uint8_t)sd;
            if (lane == 1) *reinterpret_cast<uint16_t*>(blk + 208) = (uint16_t)(sd >> 16);
        }
    }
}

// F16 (GGUF type 1): fp16 round-to-nearest-even of (col_scale *) x, 8 per thread.
__global__ __launch_bounds__(kEncodeThreads) void f16_quantize_kernel(const float* __restrict__ src,
                                                                      const float* __restrict__ col_scale,
                                                                      uint16_t* __restrict__ dst, uint64_t n_groups,
                                                                      uint32_t groups_per_row) {
    for (uint64_t i = (uint64_t)blockIdx.x * kEncodeThreads + threadIdx.x; i < n_groups;
         i += (uint64_t)gridDim.x * kEncodeThreads) {
        float v[8];
        const float4_t a = *reinterpret_cast<const float4_t*>(src + 8 * i);
        const float4_t b = *reinterpret_cast<const float4_t*>(src + 8 * i + 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = a[q];
            v[4 + q] = b[q];
        }
        if (col_scale) {
            const float* cs = col_scale + 8u * mod_u64(i, groups_per_row);
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = __fmul_rn(v[q], cs[q]);
        }
        *reinterpret_cast<uint4_t*>(dst + 8 * i) =
            uint4_t{as_u32(h2(v[0], v[1])), as_u32(h2(v[2], v[3])), as_u32(h2(v[4], v[5])), as_u32(h2(v[6], v[7]))};
    }
}

// Blocks for n super-blocks, one wave per kSuperUnroll of them at a time.
unsigned grid_for_super(uint64_t n) {
    const uint64_t g = (n + kEncodeWaves * kSuperUnroll - 1) / (kEncodeWaves * kSuperUnroll);
    return (unsigned)(g < (uint64_t)kEncodeBlocks ? g : (uint64_t)kEncodeBlocks);
}

unsigned grid_for(uint64_t n) {
    const uint64_t g = (n + kEncodeThreads - 1) / kEncodeThreads;
    return (unsigned)(g < (uint64_t)kEncodeBlocks ? g : (uint64_t)kEncodeBlocks);
}

}  // namespace

hipError_t launch_quantize(uint32_t type_id, const float* src, int rows, int k, const float* col_scale, void* dst,
                           hipStream_t stream) {
    const uint64_t r = (uint64_t)rows;
    switch (type_id) {
        case kTypeGF4: {
            const uint64_t n = r * (uint64_t)(k / 8);
            hipLaunchKernelGGL(gf4_pack_kernel, dim3(grid_for(n)), dim3(kEncodeThreads), 0, stream, src, col_scale,
                               static_cast<uint32_t*>(dst), n, (uint32_t)(k / 8));
            break;
        }
        case kTypeQ8_0: {
            const uint64_t n = r * (uint64_t)(k / 32);
            hipLaunchKernelGGL(q8_0_quantize_kernel, dim3(grid_for_super((n + 7) / 8)), dim3(kEncodeThreads), 0, stream, src,
                               col_scale, static_cast<uint8_t*>(dst), n, (uint32_t)(k / 32));
            break;
        }
        case kTypeF16: {
            const uint64_t n = r * (uint64_t)(k / 8);
            hipLaunchKernelGGL(f16_quantize_kernel, dim3(grid_for(n)), dim3(kEncodeThreads), 0, stream, src,
                               col_scale, static_cast<uint16_t*>(dst), n, (uint32_t)(k / 8));
            break;
        }
        case kTypeQ6_K: {
            const uint64_t n = r * (uint64_t)(k / 256);
            hipLaunchKernelGGL(q6_k_quantize_kernel, dim3(grid_for_super(n)), dim3(kEncodeThreads), 0, stream, src,
                               col_scale, static_cast<uint8_t*>(dst), n, (uint32_t)(k / 256));
            break;
        }
        case kTypeGF2: {
            const uint64_t n = r * (uint64_t)(k / 256);
            hipLaunchKernelGGL(gf2_pack_kernel, dim3(grid_for_super(n)), dim3(kEncodeThreads), 0, stream, src, col_scale,
                               static_cast<uint8_t*>(dst), n, (uint32_t)(k / 256));
            break;
        }
        case kTypeQ5_K: {
            const uint64_t n = r * (uint64_t)(k / 256);
            hipLaunchKernelGGL(k_quantize_kernel<true>, dim3(grid_for_super(n)), dim3(kEncodeThreads), 0, stream, src,
                               col_scale, static_cast<uint8_t*>(dst), n, (uint32_t)(k / 256));
            break;
        }
        default: {
            const uint64_t n = r * (uint64_t)(k / 256);
            hipLaunchKernelGGL(k_quantize_kernel<false>, dim3(grid_for_super(n)), dim3(kEncodeThreads), 0, stream, src,
                               col_scale, static_cast<uint8_t*>(dst), n, (uint32_t)(k / 256));
            break;
        }
    }
    return hipGetLastError();
}

}  // namespace qw35

// Streaming-read probe: the measured HBM read ceiling the GEMVs are compared
// with.  Every 16-byte word of `buf` is loaded once (non-temporal, four loads in
// flight per thread) and folded into one XOR per workgroup, written to
// sink[blockIdx.x] so that no load can be elided.
namespace qw35 {
namespace {

constexpr int kReadThreads = 512;

__global__ __launch_bounds__(kReadThreads) void stream_read_kernel(const uint4_t* __restrict__ buf, uint64_t words,
                                                                   uint32_t* __restrict__ sink) {
    uint32_t acc = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kReadThreads;
    uint64_t i = (uint64_t)blockIdx.x * kReadThreads + threadIdx.x;
    for (; i + 3 * stride < words; i += 4 * stride) {
        const uint4_t a = load_stream16(buf + i);
        const uint4_t b = load_stream16(buf + i + stride);
        const uint4_t c = load_stream16(buf + i + 2 * stride);
        const uint4_t d = load_stream16(buf + i + 3 * stride);
        acc ^= (a.x ^ a.y ^ a.z ^ a.w) ^ (b.x ^ b.y ^ b.z ^ b.w) ^ (c.x ^ c.y ^ c.z ^ c.w) ^ (d.x ^ d.y ^ d.z ^ d.w);
    }
    for (; i < words; i += stride) {
        const uint4_t a = load_stream16(buf + i);
        acc ^= a.x ^ a.y ^ a.z ^ a.w;
    }
    __shared__ uint32_t red[kReadThreads / 64];
    for (int o = 1; o < 64; o <<= 1) acc ^= (uint32_t)__shfl_xor((int)acc, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t v = 0;
        for (int w = 0; w < kReadThreads / 64; ++w) v ^= red[w];
        sink[blockIdx.x] = v;
    }
}

}  // namespace

// About 768 words (12 KiB) per workgroup, at most 16384 workgroups: the fastest
// of the launch shapes measured on MI355X for 25 MB (5.1 us) and 1 GiB (6.9 TB/s).
unsigned stream_read_blocks(uint64_t bytes) {
    uint64_t blocks = bytes / 16 / 768;
    if (blocks > 16384) blocks = 16384;
    return blocks ? (unsigned)blocks : 1u;
}

hipError_t launch_stream_read(const void* buf, uint64_t bytes, uint32_t* sink, hipStream_t stream) {
    hipLaunchKernelGGL(stream_read_kernel, dim3(stream_read_blocks(bytes)), dim3(kReadThreads), 0, stream,
                       static_cast<const uint4_t*>(buf), bytes / 16, sink);
    return hipGetLastError();
}

}  // namespace qw35
