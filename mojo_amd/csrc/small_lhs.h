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

constexpr int kSmallPlane = 528;  // an lhs row of 256 columns on its way between lanes: 512 bytes + 16 (bank spread)

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

// Rows r0 .. r0 + PASS - 1 to fp16 planes of kSmallPlane bytes in `area` (fp32 rows, PL = 2: hi part, then residual).  xr[j]: columns 4 lane .. 4 lane + 3 of row j.
// Where the values are not of ordinary size, each row is scaled by a power of two first, whose inverses go to `scales`, and the result is true.
template <int PL, int PASS, int ORDER, typename RAW, int ROWS>
__device__ __forceinline__ bool small_narrow(const RAW (&xr)[ROWS], int r0, uint8_t* area, float* scales, int lane) {
    float x[PASS][4], mx[PASS], top = 0.0f;
    bool floor_ok = true;
#pragma unroll
    for (int j = 0; j < PASS; j++) {
        const RAW raw = xr[r0 + j];
        if constexpr (PL == 2) {
            x[j][0] = __uint_as_float(raw.x), x[j][1] = __uint_as_float(raw.y), x[j][2] = __uint_as_float(raw.z), x[j][3] = __uint_as_float(raw.w);
        } else {
            x[j][0] = __uint_as_float(raw.x << 16), x[j][1] = __uint_as_float(raw.x & 0xffff0000u);
            x[j][2] = __uint_as_float(raw.y << 16), x[j][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
        mx[j] = fmaxf(fmaxf(fmaxf(fabsf(x[j][0]), fabsf(x[j][1])), fabsf(x[j][2])), fabsf(x[j][3]));
        top = fmaxf(top, mx[j]);
        floor_ok = floor_ok & (__builtin_amdgcn_ballot_w64(mx[j] >= 0.125f) != 0);
    }
    // Every row's largest value between 2^-3 and 2^10 (activations of ordinary size): the values go to fp16 as they are, what is below fp16's
    // normal range (2^-14) is small against the largest, and a sum of 32 is an fp16 number.  Otherwise a power of two per row brings its largest value to [2^9, 2^10) first.
    const bool scaled = !floor_ok || __builtin_amdgcn_ballot_w64(top >= 1024.0f) != 0;
    __builtin_amdgcn_wave_barrier();
    if (scaled) {
#pragma unroll
        for (int j = 0; j < PASS; j++) {
            if constexpr (ORDER == kSmallOrderGptq) {  // (of the finite values: an infinity stays one, and the others are held as in any row)
                mx[j] = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) mx[j] = fmaxf(mx[j], fabsf(x[j][i]) <= 3.402823466e38f ? fabsf(x[j][i]) : 0.0f);
            }
            // (2^-117: the least fp32 value, 2^-149, becomes 2^-23 and is held exactly; a row with an infinity stays unscaled)
            int e = max((int)(wave_max_nonneg_bits(mx[j]) >> 23) - 127, -117);
            if (e > 127) e = 9;
            const float sc = __uint_as_float((uint32_t)(127 + 9 - e) << 23);
            if (lane == 0) scales[j] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
#pragma unroll
            for (int i = 0; i < 4; i++) x[j][i] *= sc;
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
        const half2v ha = to_half2(xs[0], xs[1]), hb = to_half2(xs[2], xs[3]);
        uint8_t* const at = area + (j * PL) * kSmallPlane + 8 * lane;
        put(at, __builtin_bit_cast(uint32_t, ha), __builtin_bit_cast(uint32_t, hb));
        if constexpr (PL == 2) {  // residual x - hi: exact in fp32
            // (GPTQ, whose weights have no minima: an infinity has no residual, so that it gives infinities and not NaN)
            auto residual = [&](_Float16 h, float v) __attribute__((always_inline)) {
                return ORDER != kSmallOrderGptq || fabsf((float)h) <= 65504.0f ? fmaf((float)h, -1.0f, v) : 0.0f;
            };
            const half2v ra = to_half2(residual(ha.x, xs[0]), residual(ha.y, xs[1]));
            const half2v rb = to_half2(residual(hb.x, xs[2]), residual(hb.y, xs[3]));
            put(at + kSmallPlane, __builtin_bit_cast(uint32_t, ra), __builtin_bit_cast(uint32_t, rb));
        }
    }
    return scaled;
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
