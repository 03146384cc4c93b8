// The lhs of the kernels for a few rows (gemv_kquant_small.hip, gemv_gptq_small.hip): 256 columns of every row, narrowed to fp16 by the wavefront that multiplies them.
#pragma once
#include "gemm_lhs.h"
#include "lds_stream.h"
#include "qmm_internal.h"

namespace qmm {

typedef _Float16 ks_half4 __attribute__((ext_vector_type(4)));
typedef float ks_float4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef int ks_int4 __attribute__((ext_vector_type(4)));

// Lhs rows that one workgroup takes at most: a lane holds sums of four operand rows, and an fp32 row is two of them.  More rows go to several workgroups, each of which streams the weights itself.
template <typename AT>
constexpr int small_rows() { return sizeof(AT) == 4 ? 8 : 16; }
static_assert(small_rows<float>() == 8 && small_rows<uint16_t>() == 16, "small_most_rows");
// Places for workgroups on the part, `tiles` that share weights counted as one; these stay on one XCD, so it is what fits each of the eight.
inline int64_t small_places(int per_cu, int tiles) { return tiles == 1 ? (int64_t)compute_units() * per_cu : (int64_t)compute_units() * per_cu / 8 / tiles * 8; }

constexpr int kSmallPlane = 528;  // an lhs row of 256 columns on its way between lanes: 512 bytes + 16 (bank spread)

// hidden_load from a wave-uniform base and a byte offset per lane.
__device__ __forceinline__ void hidden_load(u32x4& d, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(d) : "v"(lane_offset), "s"(uniform_base) : "memory");
}
__device__ __forceinline__ void hidden_load(u32x2& d, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(d) : "v"(lane_offset), "s"(uniform_base) : "memory");
}
// 16 bytes per lane, global (uniform base + lane offset) -> LDS at lds_base + 16 * lane.  ONCE: non-temporal.
template <bool ONCE = true>
__device__ __forceinline__ void small_stream16(uint32_t lane_offset, const void* uniform_base, uint32_t lds_base) {
    uint32_t keep;
    const uint64_t b = (uint64_t)(uintptr_t)uniform_base;
    const uint64_t sb = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
                        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    if constexpr (ONCE)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep)
                     : "v"(lane_offset), "s"(sb), "s"(lds_base)
                     : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep)
                     : "v"(lane_offset), "s"(sb), "s"(lds_base)
                     : "memory");
}
__device__ __forceinline__ half2v to_half2(float a, float b) { return __builtin_convertvector((float2v{a, b}), half2v); }  // to nearest, one instruction
__device__ __forceinline__ uint32_t to_half2_bits(float a, float b) { return __builtin_bit_cast(uint32_t, to_half2(a, b)); }

// The order in which four (GPTQ: eight) neighbouring columns lie in a plane: 0,1,2,3; 0,2,1,3; 0,4,1,5,2,6,3,7.
enum { kSmallOrderPlain = 0, kSmallOrderK = 1, kSmallOrderGptq = 2 };

// The lhs is scaled so that what fp16 leaves out of any value, up to 2^-25, is small against its row's largest: with a scale of the row's own 2^-34 of it where weights have minima (TOP = 9: a sum of 32 values is an fp16
// number too), else 2^-39 (TOP = 14), as in the kernels for more rows; with one scale for all rows 2^-31 and 2^-36 of a row's that is only an eighth of the largest.  Which of the two it is depends on all rows of a
// workgroup, so the last bits of a row are those of a call with the same rows beside it.
// fp32 rows (hi part and residual): one power of two for all rows, which brings the largest value to [2^TOP, 2^(TOP + 1)), where every row's largest is at least an eighth of it; the result is that scale, or 0: one for each
// row.  One search over the wavefront for all of them; one for each row always, and the products, took 8 rows 4096 x 4096 from 8.0 to 8.5 (Q4_K) and 7.8 to 9.3 us (GPTQ).
template <int TOP, typename RAW, int ROWS>
__device__ __forceinline__ float small_common_scale(const RAW (&xr)[ROWS]) {
    float mx[ROWS], top = 0.0f;
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        mx[j] = fmaxf(fmaxf(fmaxf(fabsf(__uint_as_float(xr[j].x)), fabsf(__uint_as_float(xr[j].y))), fabsf(__uint_as_float(xr[j].z))), fabsf(__uint_as_float(xr[j].w)));
        top = fmaxf(top, mx[j]);
    }
    const int e = (int)(wave_max_nonneg_bits(top) >> 23) - 127;
    if (e < TOP - 126 || e > 126) return 0.0f;
    const float floor = __uint_as_float((uint32_t)max(127 + e - 3, 0) << 23);
    bool common = true;
#pragma unroll
    for (int j = 0; j < ROWS; j++) common = common & (__builtin_amdgcn_ballot_w64(mx[j] >= floor) != 0);
    return common ? __uint_as_float((uint32_t)(127 + TOP - e) << 23) : 0.0f;
}

// Rows r0 .. r0 + PASS - 1 to fp16 planes of kSmallPlane bytes in `area` (fp32 rows, PL = 2: hi part, then residual).  xr[j]: columns 4 lane .. 4 lane + 3 of row j.
// common: what small_common_scale says (fp32 rows).  bf16 rows stay as they are where every value is then an fp16 number (none but zeros below 2^-17, whose last bit is 2^-24) and none is too large.  Otherwise a power of two
// per row brings its largest value to [2^TOP, 2^(TOP + 1)), and the inverses go to `scales`.  The result is the inverse of the scale of all rows, or 0.
template <int PL, int PASS, int ORDER, int TOP, typename RAW, int ROWS>
__device__ __forceinline__ float small_narrow(const RAW (&xr)[ROWS], int r0, float common, uint8_t* area, float* scales, int lane) {
    float x[PASS][4], sc[PASS];
    bool each = common == 0.0f;
    if constexpr (PL == 1) {
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        u16x2 most = {0, 0}, least = {0xffff, 0xffff};
#pragma unroll
        for (int j = 0; j < PASS; j++) {
            const u16x2 v0 = __builtin_bit_cast(u16x2, (uint32_t)xr[r0 + j].x & 0x7fff7fffu), v1 = __builtin_bit_cast(u16x2, (uint32_t)xr[r0 + j].y & 0x7fff7fffu), one = {1, 1};
            most = __builtin_elementwise_max(most, __builtin_elementwise_max(v0, v1));
            least = __builtin_elementwise_min(least, __builtin_elementwise_min((u16x2)(v0 - one), (u16x2)(v1 - one)));  // (zeros: the largest number)
        }
        const uint16_t m0 = most.x, m1 = most.y, l0 = least.x, l1 = least.y;
        each = __builtin_amdgcn_ballot_w64(max(m0, m1) >= (127 + TOP + 1) << 7 || min(l0, l1) < ((127 - 17) << 7) - 1) != 0;
    }
#pragma unroll
    for (int j = 0; j < PASS; j++) {
        const RAW raw = xr[r0 + j];
        if constexpr (PL == 2) {
            x[j][0] = __uint_as_float(raw.x), x[j][1] = __uint_as_float(raw.y), x[j][2] = __uint_as_float(raw.z), x[j][3] = __uint_as_float(raw.w);
        } else {
            x[j][0] = __uint_as_float(raw.x << 16), x[j][1] = __uint_as_float(raw.x & 0xffff0000u);
            x[j][2] = __uint_as_float(raw.y << 16), x[j][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
        sc[j] = common;
    }
    __builtin_amdgcn_wave_barrier();
    if (each) {
#pragma unroll
        for (int j = 0; j < PASS; j++) {
            float mx = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; i++)  // (GPTQ: of the finite values: an infinity stays one, and the others are held as in any row)
                mx = fmaxf(mx, ORDER != kSmallOrderGptq || fabsf(x[j][i]) <= 3.402823466e38f ? fabsf(x[j][i]) : 0.0f);
            // (the least scale is that whose inverse is 2^-126: the least fp32 value, 2^-149, becomes 2^-23 and is held exactly; a row with an infinity stays unscaled)
            int e = max((int)(wave_max_nonneg_bits(mx) >> 23) - 127, TOP - 126);
            if (e > 127) e = TOP;
            sc[j] = __uint_as_float((uint32_t)(127 + TOP - e) << 23);
            if (lane == 0) scales[j] = __uint_as_float((uint32_t)(127 - TOP + e) << 23);
            if constexpr (PL == 1) {
#pragma unroll
                for (int i = 0; i < 4; i++) x[j][i] *= sc[j];
            }
        }
    }
    // GPTQ: the lane of an even four gives its columns 2, 3 for the next lane's 0, 1 (columns 4, 5 of the eight): (0,4), (1,5) here, (2,6), (3,7) there
    const bool second = lane & 1;
    const uint32_t pick0 = second ? 0x01000504u : 0x05040100u, pick1 = second ? 0x03020706u : 0x07060302u;
    auto put = [&](uint8_t* at, uint32_t a, uint32_t b) __attribute__((always_inline)) {
        if constexpr (ORDER == kSmallOrderGptq) {
            const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)(second ? a : b), 0xB1, 0xf, 0xf, true), own = second ? b : a;
            a = __builtin_amdgcn_perm(other, own, pick0), b = __builtin_amdgcn_perm(other, own, pick1);
        }
        *(uint2*)at = make_uint2(a, b);
    };
#pragma unroll
    for (int j = 0; j < PASS; j++) {
        constexpr int i1 = ORDER == kSmallOrderK ? 2 : 1, i2 = ORDER == kSmallOrderK ? 1 : 2;
        const float xs[4] = {x[j][0], x[j][i1], x[j][i2], x[j][3]};
        uint8_t* const at = area + (j * PL) * kSmallPlane + 8 * lane;
        if constexpr (PL == 1) {
            put(at, to_half2_bits(xs[0], xs[1]), to_half2_bits(xs[2], xs[3]));
        } else {
            // (products with a power of two: the rounding to fp16 is the only one, in one instruction with the product)
            _Float16 h[4], r[4];
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = (_Float16)__builtin_fmaf(xs[i], sc[j], 0.0f);
            // residual x - hi: exact in fp32
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = (_Float16)__builtin_fmaf(xs[i], sc[j], -(float)h[i]);
            if (ORDER == kSmallOrderGptq && each) {  // (weights without minima: an infinity has no residual, so that it gives infinities and not NaN; rows with one have no common scale)
#pragma unroll
                for (int i = 0; i < 4; i++) r[i] = fabsf((float)h[i]) <= 65504.0f ? r[i] : (_Float16)0.0f;
            }
            put(at, __builtin_bit_cast(uint32_t, half2v{h[0], h[1]}), __builtin_bit_cast(uint32_t, half2v{h[2], h[3]}));
            put(at + kSmallPlane, __builtin_bit_cast(uint32_t, half2v{r[0], r[1]}), __builtin_bit_cast(uint32_t, half2v{r[2], r[3]}));
        }
    }
    // (the inverse of a power of two: its exponent, negated)
    return each ? 0.0f : PL == 1 ? 1.0f : __uint_as_float((254u << 23) - __float_as_uint(common));
}

constexpr int kSmallCodes = 272;  // an lhs row of 256 columns as Q8_0: codes, block by block in the order of small_quantize, then the eight block scales

// Rows r0 .. r0 + PASS - 1 (at most four) as Q8_0 to `area`, kSmallCodes bytes each.  The 32 codes of a block in eight dwords: columns 4 i .. 4 i + 3 and 16 + 4 i .. + 3 lie in dwords 2 i and 2 i + 1.
// Eight lanes hold a block of every row; the divisions of a block's rule are made once for four rows, by the lane whose number is the row's.
template <int PASS, typename RAW, int ROWS>
__device__ __forceinline__ void small_quantize(const RAW (&xr)[ROWS], int r0, uint8_t* area, int lane) {
    static_assert(PASS <= 4, "a lane of four for each row");
    float x[PASS][4], amax[PASS];
#pragma unroll
    for (int j = 0; j < PASS; j++) {
        const RAW raw = xr[r0 + j];
        if constexpr (sizeof(RAW) == 16) {
            x[j][0] = __uint_as_float(raw.x), x[j][1] = __uint_as_float(raw.y), x[j][2] = __uint_as_float(raw.z), x[j][3] = __uint_as_float(raw.w);
        } else {
            x[j][0] = __uint_as_float(raw.x << 16), x[j][1] = __uint_as_float(raw.x & 0xffff0000u);
            x[j][2] = __uint_as_float(raw.y << 16), x[j][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
        float mx = fmaxf(fmaxf(fmaxf(fabsf(x[j][0]), fabsf(x[j][1])), fabsf(x[j][2])), fabsf(x[j][3]));
        mx = fmaxf(mx, dpp_move<0xB1>(mx));   // lane ^ 1
        mx = fmaxf(mx, dpp_move<0x4E>(mx));   // lane ^ 2
        amax[j] = fmaxf(mx, dpp_move<0x141>(mx));  // the other four of the eight (half mirror)
    }
    const int mine = lane & 3;
    float top = amax[0];
#pragma unroll
    for (int j = 1; j < PASS; j++) top = mine == j ? amax[j] : top;
    uint16_t dh;
    const float id = q8_0_block_rule(top, dh);
    __builtin_amdgcn_wave_barrier();
    if ((lane & 4) == 0 && mine < PASS) *(uint16_t*)(area + mine * kSmallCodes + 256 + 2 * (lane >> 3)) = dh;
#pragma unroll
    for (int j = 0; j < PASS; j++) {
        const float inv = j == 0 ? dpp_move<0x00>(id) : j == 1 ? dpp_move<0x55>(id) : j == 2 ? dpp_move<0xAA>(id) : dpp_move<0xFF>(id);  // that of lane j of the four
        uint32_t c[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // q8_0_code: rounded with halves away from zero.  Adding the number below 0.5, not 0.5, makes that exact: 0.5 - 2^-25 stays below one, and a half still rounds up.
            const float t = x[j][i] * inv;
            c[i] = (uint32_t)(int)(t + __builtin_copysignf(0.49999997f, t));
        }
        const uint32_t codes = __builtin_amdgcn_perm(__builtin_amdgcn_perm(c[3], c[2], 0x0C0C0400u), __builtin_amdgcn_perm(c[1], c[0], 0x0C0C0400u), 0x05040100u);
        *(uint32_t*)(area + j * kSmallCodes + 32 * (lane >> 3) + 8 * (lane & 3) + (lane & 4)) = codes;
    }
}

}  // namespace qmm
