// What the GEMMs that unpack the weights in their matrix-core loop share (gemm_direct.hip, gemm_shared.hip): the operand order of the lhs and
// where its preparation leaves it, and, per encoding, how a wavefront turns the packed weights of 32 FN columns into matrix-core operands.
#pragma once
#include <algorithm>
#include <type_traits>

#include "gemm_lhs.h"
#include "qmm_internal.h"

namespace qmm {

// Sizes of what the preparation launch leaves behind.  Every row tile of 32 rows: k / 16 operands of 1 KB, rounded up to whole units of 16 (fp32 lhs: pairs of
// them, hi then residual), and room for one more unit behind the last (the loop reads ahead); sums: one operand per 256 columns; inverse row scales.
struct DirectSpace {
    _Float16* a16;
    _Float16* sums;  // of 32 columns, hi and lo parts (Q4_0: the block scales)
    float* sums32;   // the same in fp32: four per lane and 256 columns (Q4_K, Q5_K)
    float* inv;
    int64_t bytes;
};

// The matrices of one launch (they share the lhs): their results, and where each ends in the grid, in eights of column tiles.
struct DirectMats {
    const uint8_t* w[kDirectMaxMats];
    float* out[kDirectMaxMats];
    int n[kDirectMaxMats], end[kDirectMaxMats];
    int count;
};

struct WeightTensors {
    const uint8_t* w;        // K-quant blocks, or GPTQ qweight
    const uint16_t* scales;  // GPTQ
    const uint32_t* qzeros;
    int n, k, group;
};

// How a call is cut: every wavefront takes 32 fm rows x 32 fn columns.  wn = 1: the wk wavefronts of a workgroup take wk parts of K of one tile
// (gemm_direct.hip).  wn > 1: wn wavefronts side by side share the lhs, wk parts of K (gemm_shared.hip, and with fn = 0, which means one, gemm_staged.hip).  shares:
// workgroups per tile (1, or 2 that add onto zeros).  fold, gemm_staged.hip: sums over kStagedFold units are added up in others (staged_folds).  centred: gemm_staged.hip, codes of Q4_K and Q5_K around their middle.
struct DirectPlan {
    int fm, fn, wk, shares, wn;
    bool centred = false, fold = false;
};
hipError_t launch_gemm_shared(int encoding, bool hilo, const DirectPlan& pl, const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16,
                              int64_t m, int units, hipStream_t s);
// gptq_order.hip: the columns of the weights sorted by group and, unless !lhs_done, those of the lhs in p, with `zero` (up to `zeros` results each) zeroed.
hipError_t launch_gptq_order(const GptqOrder& order, int64_t n, int64_t k, int group, const void* lhs, int lhs_dtype, int64_t m, const DirectSpace& p, const DirectMats& zero,
                             int64_t zeros, bool& lhs_done, hipStream_t s);
hipError_t launch_gemm_staged(int encoding, bool hilo, const DirectPlan& pl, const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16,
                              int64_t m, int units, hipStream_t s);

// What gemm_staged.hip has: fp32 rows, small groups and codes around their middle, which all sum a unit of K by itself, leave no registers for 128 rows a wavefront.
constexpr bool staged_built(int encoding, int flush, int fm, bool hilo, bool centred) { return fm <= 3 || !(hilo || centred || (encoding == QMM_GPTQ && flush == 2)); }
// The last row tile of 32 fm rows as one of 32: where that is all it has, and not the only one (sections: workgroups of a row tile on an XCD; the grid's z has 16 bits).
inline bool staged_short_last(int fm, int64_t m, int64_t sections) { return m > 32 * fm && (m - 1) % (32 * fm) < 32 && 2 * sections < 65536; }
// What folds its sums there: GPTQ in groups of 128 and more, where there are registers for a second set.
constexpr int kStagedFold = 4;  // units
constexpr bool staged_folds(int encoding, int flush, int fm, bool hilo) { return encoding == QMM_GPTQ && flush == 8 && fm <= (hilo ? 2 : 3); }

namespace {

// Where a workgroup of the direct or the shared kernel is: ids congruent mod 8 run on one XCD; there the row tiles of a column tile follow each other, so that its L2 fetches the
// weights once.  The shape of the grid, 8 x row tiles x (shares of column sections), spares the divisions; where it does not hold them, one number counts through (tiles_m > 0).
struct DirectGrid {
    dim3 grid;
    int tiles_m;
};
inline DirectGrid direct_grid(int tiles_m, int places) {
    if (tiles_m < 65536 && places < 65536) return {dim3(8, (unsigned)tiles_m, (unsigned)places), 0};
    return {dim3((unsigned)(8 * tiles_m * places)), tiles_m};
}
struct DirectPlace {
    int tile_m, share, section, eighth;
};
__device__ __forceinline__ DirectPlace direct_place(int tiles_m, int shares) {
    int tile_m = (int)blockIdx.y, place = (int)blockIdx.z, eighth = (int)blockIdx.x;
    if (tiles_m) {
        const int i = eighth >> 3;
        eighth &= 7;
        place = i / tiles_m, tile_m = i - place * tiles_m;
    }
    return {tile_m, place & (shares - 1), place >> (shares - 1), eighth};
}

typedef uint32_t gd_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t gd_u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ half2v as_h2(uint32_t x) { return __builtin_bit_cast(half2v, x); }
__device__ __forceinline__ uint32_t as_u32(half2v x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t pk_add(uint32_t x, uint32_t y) { return as_u32(as_h2(x) + as_h2(y)); }
// byte j of v under the byte `top` in both halves: with top 0x18 the fp16 pair 2^-9 + byte 2^-19, with 0x64 1024 + byte, with 0x68 2048 + 2 byte, with 0x78 32768 + 32 byte
template <int J>
__device__ __forceinline__ uint32_t byte_pair(uint32_t top4, uint32_t v) { return __builtin_amdgcn_perm(top4, v, 0x04000400u | (J << 16) | J); }

// A constant in a vector register that the compiler takes for a variable: (x & mask) | top is one instruction then (v_and_or_b32 has room for one scalar operand and no literal; given two
// constants the compiler makes two instructions of it).  14 -> 10 of them a step for GPTQ, 16 -> 12 for Q4_0.
__device__ __forceinline__ uint32_t code_top(uint32_t top) {
    asm("" : "+v"(top));
    return top;
}

// A row is scaled by a power of two so that its largest value lies in [2^kRowTop, 2^(kRowTop + 1)), as high as fp16 goes: an fp32 value is then
// held to 22 bits down to 2^-17 of the row's largest and to 2^-39 of that below (2^-12 and 2^-34 with a top of 9).  Where sums of 32 values
// are held in fp16 too (Q4_K, Q5_K), 2^9 leaves them room.
constexpr int kRowTop = 14, kRowTopWithSums = 9;

// The operand order of the lhs: step t = 2 blk + a of 16 columns holds, for half wavefront g, the columns
//   32 blk + 16 g + 8 a + slot order   (kOrderK: slots 0,2,1,3,4,6,5,7; kOrderGptq: 0,4,1,5,2,6,3,7)
constexpr int kOrderK = 0, kOrderGptq = 1;  // (Q4_0: 32 blk + 16 a + 8 g + the slots of kOrderK)

// Eight columns of a row as they lie in memory.
template <typename AT>
struct LhsPiece {
    gd_u4 raw[sizeof(AT) / 2];
};
template <typename AT>
__device__ __forceinline__ LhsPiece<AT> load_piece(const AT* p) {
    LhsPiece<AT> x;
#pragma unroll
    for (int i = 0; i < (int)sizeof(AT) / 2; i++) x.raw[i] = ((const gd_u4*)p)[i];
    return x;
}
template <typename AT>
__device__ __forceinline__ void unpack_piece(const LhsPiece<AT>& x, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if constexpr (sizeof(AT) == 4) v[i] = __uint_as_float(x.raw[i >> 2][i & 3]);
        else v[i] = __uint_as_float((i & 1) ? x.raw[0][i >> 1] & 0xffff0000u : x.raw[0][i >> 1] << 16);
    }
}
// Their largest magnitude, on the bits: two vector instructions a dword, where a comparison that leaves out what is not finite takes five.  (bf16: the low and the high halves apart, until largest_of.)
template <typename AT>
__device__ __forceinline__ uint32_t largest_bits(uint32_t top, const LhsPiece<AT>& x) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < (int)sizeof(AT) / 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (sizeof(AT) == 4) top = max(top, x.raw[i][j] & 0x7fffffffu);
            else top = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, top), __builtin_bit_cast(u16x2, x.raw[i][j] & 0x7fff7fffu)));
        }
    return top;
}
template <typename AT>
__device__ __forceinline__ float largest_of(uint32_t top) { return __uint_as_float(sizeof(AT) == 4 ? top : max(top & 0xffff0000u, top << 16)); }
// Of the finite ones: for wavefronts in which largest_of is none.
template <typename AT>
__device__ __forceinline__ float largest_finite(float mx, const LhsPiece<AT>& x) {
    float v[8];
    unpack_piece(x, v);
#pragma unroll
    for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]) <= 3.402823466e38f ? fabsf(v[i]) : 0.0f);
    return mx;
}
__device__ __forceinline__ bool any_not_finite(float mx) { return __any(__float_as_uint(mx) >= 0x7f800000u); }
// What a row is multiplied by, and its inverse, from the bits of its largest magnitude.
__device__ __forceinline__ float row_scale(uint32_t largest_bits, int row_top, float& inv) {
    int e = (int)((largest_bits >> 23) & 0xffu) - 127;
    e = max(e, row_top - 126);  // (the smallest inverse scale that is a normal number, 2^-126: the least fp32 value, 2^-149, becomes 2^-23 and is held exactly)
    inv = __uint_as_float((uint32_t)(127 - row_top + e) << 23);
    return __uint_as_float((uint32_t)(127 + row_top - e) << 23);
}
// Two values as fp16, one instruction.
__device__ __forceinline__ uint32_t narrow2(float x, float y) {
    typedef float float2v __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v{x, y}), half2v));
}
// Where the eight values of lane (row of the tile, half g of a step's 16 columns) lie among the operands of a row tile, in bytes; per: terms of a value (bf16 1, fp32 2).  A row tile takes 64 K per
// bytes: more than 32 bits from K = 2^25 on.
constexpr int64_t operand_offset(int step, int row, int g, int per) { return (int64_t)step * (1024 * per) + (row + 32 * g) * 16; }
// Piece pc (eight columns) of a row, scaled by s (v is left so), as its part of the operands.
template <typename AT, int ORDER>
__device__ __forceinline__ void store_piece(_Float16* a16, int steps, int row, int pc, float s, float (&v)[8]) {
    constexpr bool kF32 = sizeof(AT) == 4;
    constexpr int perm[2][8] = {{0, 2, 1, 3, 4, 6, 5, 7}, {0, 4, 1, 5, 2, 6, 3, 7}};
    const int blk = pc >> 2, g = (pc >> 1) & 1, step = 2 * blk + (pc & 1);
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] *= s;
    HalfPack hi;
#pragma unroll
    for (int i = 0; i < 4; i++) hi.u[i] = narrow2(v[perm[ORDER][2 * i]], v[perm[ORDER][2 * i + 1]]);
    uint8_t* const at = (uint8_t*)a16 + (int64_t)(row >> 5) * operand_offset(steps, 0, 0, kF32 ? 2 : 1) + operand_offset(step, row & 31, g, kF32 ? 2 : 1);
    *(half8*)at = hi.h;
    if constexpr (kF32) {
        HalfPack lo;
        float residual[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float h = (float)hi.h[i], x = v[perm[ORDER][i]];
            residual[i] = fabsf(h) <= 65504.0f ? x - h : 0.0f;  // (an infinity has no residual: inf - inf)
        }
#pragma unroll
        for (int i = 0; i < 4; i++) lo.u[i] = narrow2(residual[2 * i], residual[2 * i + 1]);
        *(half8*)(at + 1024) = lo.h;
    }
}
// The e-th of `count` workgroups zeroes its part of the results (m rows).
__device__ __forceinline__ void zero_out(const DirectMats& z, int m, int e, int count) {
    const int threads = (int)blockDim.x;
    for (int j = 0; j < z.count; j++) {
        float* __restrict__ const out = z.out[j];
        const int64_t values = (int64_t)m * z.n[j];
        for (int64_t i = ((int64_t)e * threads + threadIdx.x) * 4; i < values; i += (int64_t)count * threads * 4) {
            if (i + 3 < values) *(float4*)(out + i) = make_float4(0.f, 0.f, 0.f, 0.f);
            else
                for (int64_t q = i; q < values; q++) out[q] = 0.0f;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
// the weights of one wavefront: what it holds of a unit of K, how a step's operands come out of it
// ---------------------------------------------------------------------------------------------------------------------------
// The packed rows of a K-quant: 32 FN columns x one block.  A lane that loaded its own column's codes would touch a cache line of its
// own with every load (64 lines an instruction, which took longer than everything else here), so the wavefront loads the blocks as they
// lie in memory, 16 bytes per lane, a whole unit ahead, and hands them out through a part of LDS that is its own (no barrier).
template <int BPB, int FN>
struct StagedRows {
    static constexpr int kPieces = (BPB + 15) / 16, kRow = kPieces * 16;  // the last piece ends with the block (Q6_K: bytes 194 .. 209)
    static constexpr int kTotal = 32 * FN * kPieces, kLoads = (kTotal + 63) / 64, kBytes = 32 * FN * kRow;
    const uint8_t* w;
    uint8_t* lds;
    uint32_t off[kLoads];
    gd_u4 raw[kLoads];
    struct __attribute__((packed, aligned(2))) Bytes16 {
        gd_u4 v;
    };
    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* stage) {
        w = t.w;
        lds = stage;
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const int i = min(j * 64 + lane, kTotal - 1), row = i / kPieces, piece = i - row * kPieces;
            off[j] = (uint32_t)min(n0 + row, t.n - 1) * (uint32_t)(t.k / 256 * BPB) + min(16 * piece, BPB - 16);
        }
    }
    __device__ __forceinline__ void load(int unit) {
        const uint8_t* b = w + (int64_t)unit * BPB;
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            if constexpr (BPB % 16 == 0) raw[j] = *(const gd_u4*)(b + off[j]);
            else raw[j] = ((const Bytes16*)(b + off[j]))->v;
        }
    }
    __device__ __forceinline__ void to_lds(int lane) {
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            if (j * 64 + 63 < kTotal || j * 64 + lane < kTotal) *(gd_u4*)(lds + j * 1024 + lane * 16) = raw[j];
    }
};

// Q4_K, Q5_K.  Lane (column nl of a group, half g) takes bytes 16 g .. 16 g + 15 of each of the four 32-byte code runs of a block: run c is
// sub-block 2 c in its low nibbles and 2 c + 1 in its high ones.  A nibble masked in place reads as the fp16 subnormal q 2^-24 (low) or
// q 2^-20 (high); times 32 sc or 2 sc it is sc q 2^-19, exact (sc q at most 1953), and a normal number from sc q = 32 on: the matrix cores
// keep fewer bits of a sum whose operands are subnormal (fp32 rows, 2.5e-7 relative error against 6e-7 with sc q 2^-24).  Q5_K: whole bytes with the fifth bit in them, spread by
// permutes (the low nibbles as subnormals, the high ones under 64), the same operands with 14 .. 15 vector instructions a step, 18 with nibbles and bits masked in place: 14336 x 4096
// 200 bf16 rows 46.3 -> 43.7 us, 11008 x 4096 33 rows 21.5 -> 21.0.  (The same for Q6_K: no faster.)
//
// CENTER: the operand is sc (q - kMid), exact as well (one fused multiply-add), and what that leaves out, kMid d sc - dmin mn per sub-block, multiplies the
// sums of the lhs.  Codes that are all positive make sums 2.4 times as large as what the minima leave of them, and the error of a sum of the lhs counts
// fifteenfold.  Relative error without and with it, direct kernel (decode kernel): Q4_K 4096 x 4096 17 bf16 rows 1.9e-7, 0.9e-7 (0.9e-7), fp32 3.1e-7,
// 1.7e-7 (2.6e-7); Q5_K 2.2e-7, 1.0e-7 (1.0e-7), 3.2e-7, 1.7e-7 (2.4e-7).
// - direct kernel: always, the sums in fp32 (four matrix-core instructions of their own, onto the running sums); bf16 rows take 0 .. 5 % longer
//   (weights from memory; 14336 x 4096 17 rows 19.1 -> 19.9 us), fp32 rows, whose residual would need sums of its own otherwise, 2 .. 6 % less.
// - shared kernel, whose matrix cores are busier: both the offsets and the sums as two fp16 terms (two instructions a unit; the offsets exact to 22 bits of the
//   larger product).  fp32 rows 3.4e-7 -> 1.85e-7 in the same time.  bf16 rows 2.3e-7 -> 1.1e-7, but 3 .. 4 % slower, its vector units being the limit: only Q5_K up
//   to 64 rows, where the small-batch kernel has 1.6e-7; beyond, the GEMMs that it replaces have 2.6e-7 and more.
template <int ENC, int FN, bool CENTER>
struct KQuantWeights {
    static constexpr int kMid = ENC == QMM_Q5_K ? 16 : 8;
    static constexpr int kSteps = 16, kFlush = 16, kPlanes = 1;
    static constexpr bool kMin = true, kPairs = false;
    static constexpr int kCodes = ENC == QMM_Q5_K ? 48 : 16;
    using Rows = StagedRows<ENC == QMM_Q5_K ? Q5_K_BPB : Q4_K_BPB, FN>;
    static constexpr int kStage = Rows::kBytes;
    Rows rows;
    const uint8_t* mine;  // the lane's column in LDS
    int goff, lane_;
    gd_u4 q[FN][2], fifth[ENC == QMM_Q5_K ? FN : 1];
    uint32_t scs[FN][2], mns[FN][2], dm[FN];
    uint32_t top = code_top(0x54545454u);  // (Q5_K)

    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* stage) {
        rows.init(t, n0, lane, stage);
        goff = 16 * (lane >> 5);
        lane_ = lane;
        mine = stage + (lane & 31) * Rows::kRow;
    }
    __device__ __forceinline__ void load(int unit) { rows.load(unit); }
    __device__ __forceinline__ void read_codes(int c) {
#pragma unroll
        for (int f = 0; f < FN; f++) q[f][c & 1] = *(const gd_u4*)(mine + f * 32 * Rows::kRow + goff + (kCodes + 32 * c));
    }
    // the loaded unit becomes the current one
    __device__ __forceinline__ void open() {
        rows.to_lds(lane_);
        read_head();
    }
    __device__ __forceinline__ void read_head() {
        read_codes(0);
#pragma unroll
        for (int f = 0; f < FN; f++) {
            if constexpr (ENC == QMM_Q5_K) fifth[f] = *(const gd_u4*)(mine + f * 32 * Rows::kRow + goff + 16);
            const gd_u4 hdr = *(const gd_u4*)(mine + f * 32 * Rows::kRow);
            const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
            dm[f] = hdr.x;
            scs[f][0] = s0 & 0x3f3f3f3fu;
            scs[f][1] = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
            mns[f][0] = s1 & 0x3f3f3f3fu;
            mns[f][1] = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
        }
    }
    // operands of step T (plane 0 only)
    template <int T>
    __device__ __forceinline__ void step(int f, half8 (&b)[1]) const {
        constexpr int c = T >> 2, h = (T >> 1) & 1, a = T & 1, blk = 2 * c + h;
        if constexpr (ENC == QMM_Q5_K && h == 1) {  // the high nibbles under 64 in fp16, the fifth bit above them: (64 + q - (64 + mid)) sc 2^-19
            const uint32_t sp = pk_add(byte_pair<(blk & 3)>(0x18181818u, scs[f][blk >> 2]), 0x98009800u);  // 2^-9 + sc 2^-19 - 2^-9
            const uint32_t less = pk_mul(sp, CENTER ? 0xD500D500u : 0xD400D400u);  // -80, -64
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t lo = q[f][c & 1][2 * a + i] & 0xF0F0F0F0u, hi = ((fifth[f][2 * a + i] >> blk) & 0x01010101u) | top;
                v[2 * i] = __builtin_amdgcn_perm(hi, lo, 0x06020400u);
                v[2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030501u);
            }
            b[0] = pack4(pk_fma(v[0], sp, less), pk_fma(v[1], sp, less), pk_fma(v[2], sp, less), pk_fma(v[3], sp, less));
            return;
        }
        uint32_t sp;
        if constexpr (h == 0) sp = pk_add(byte_pair<(blk & 3)>(0x78787878u, scs[f][blk >> 2]), 0xF800F800u);  // 32768 + 32 sc - 32768
        else sp = pk_add(byte_pair<(blk & 3)>(0x68686868u, scs[f][blk >> 2]), 0xE800E800u);                   // 2048 + 2 sc - 2048
        constexpr uint32_t mask = h == 0 ? 0x000F000Fu : 0x00F000F0u;
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t x = q[f][c & 1][2 * a + i];
            if constexpr (ENC == QMM_Q5_K) {  // (bytes joined with their fifth bit, then spread)
                const uint32_t e = fifth[f][2 * a + i], u = (x & 0x0F0F0F0Fu) | ((blk <= 4 ? e << (4 - blk) : e >> (blk - 4)) & 0x10101010u);
                v[2 * i] = __builtin_amdgcn_perm(u, u, 0x0c020c00u);
                v[2 * i + 1] = __builtin_amdgcn_perm(u, u, 0x0c030c01u);
            } else {
                v[2 * i] = x & mask;
                v[2 * i + 1] = (x >> 8) & mask;
            }
        }
        if constexpr (CENTER) {
            const uint32_t mid = pk_mul(sp, 0x80008000u | (uint32_t)kMid * (h == 0 ? 0x00010001u : 0x00100010u));  // -kMid 2^-24 or 2^-20
            b[0] = pack4(pk_fma(v[0], sp, mid), pk_fma(v[1], sp, mid), pk_fma(v[2], sp, mid), pk_fma(v[3], sp, mid));
        } else {
            b[0] = pack4(pk_mul(v[0], sp), pk_mul(v[1], sp), pk_mul(v[2], sp), pk_mul(v[3], sp));
        }
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr ((T & 3) == 0 && T < 12) read_codes((T >> 2) + 1);
    }
    template <int T>
    __device__ __forceinline__ void after_step(int) {}
    __device__ __forceinline__ float scale(int f) const { return h2f((uint16_t)(dm[f] & 0xffffu)) * 524288.0f; }
    __device__ __forceinline__ float min_scale(int f) const { return -h2f((uint16_t)(dm[f] >> 16)); }
    __device__ __forceinline__ float4 offsets(int f) const {  // kMid d sc - dmin mn of sub-blocks g, 2 + g, 4 + g, 6 + g
        const float d = (float)kMid * h2f((uint16_t)(dm[f] & 0xffffu)), dmin = min_scale(f);
        const uint32_t by = goff >> 1;  // 8 g
        const uint32_t s0 = scs[f][0] >> by, s1 = scs[f][1] >> by, m0 = mns[f][0] >> by, m1 = mns[f][1] >> by;
        auto of = [&](uint32_t s, uint32_t mn) __attribute__((always_inline)) { return fmaf(d, (float)(s & 0xffu), dmin * (float)(mn & 0xffu)); };
        return make_float4(of(s0, m0), of(s0 >> 16, m0 >> 16), of(s1, m1), of(s1 >> 16, m1 >> 16));
    }
    // The same as two fp16 terms each, in units of the returned power of two, of all eight sub-blocks (the shared kernel): open them, add sub-block by
    // sub-block, and they multiply sums that are held as hi (g = 0) and lo parts (g = 1).
    float od, om;
    uint32_t ohi[4], olo[4];
    __device__ __forceinline__ float open_offsets() {
        const float d = (float)kMid * h2f((uint16_t)(dm[0] & 0xffffu)), dmin = min_scale(0);
        const int e = __builtin_amdgcn_frexp_expf(64.0f * fmaxf(fabsf(d), fabsf(dmin)));  // both products below 2^e
        od = ldexpf(d, 14 - e);
        om = ldexpf(dmin, 14 - e);
        return ldexpf(1.0f, e - 14);
    }
    __device__ __forceinline__ float scale_per_unit() const { return od * (524288.0f / (float)kMid); }
    // (each half wavefront works out four sub-blocks)
    template <int PAIR>
    __device__ __forceinline__ void add_offsets() {
        if constexpr (PAIR < 2) {
            const uint32_t sc = goff ? scs[0][1] : scs[0][0], mn = goff ? mns[0][1] : mns[0][0];
            float v[2];
#pragma unroll
            for (int i = 0; i < 2; i++) v[i] = fmaf(od, (float)((sc >> (16 * PAIR + 8 * i)) & 0xffu), om * (float)((mn >> (16 * PAIR + 8 * i)) & 0xffu));
            const half2v hi = {(_Float16)v[0], (_Float16)v[1]};
            const half2v lo = {(_Float16)(v[0] - (float)hi.x), (_Float16)(v[1] - (float)hi.y)};
            ohi[PAIR] = as_u32(hi);
            olo[PAIR] = as_u32(lo);
        } else {
            // (both operands the same register: the result's first half is the low lanes' value in every lane, the second that of the high lanes)
            const auto h = __builtin_amdgcn_permlane32_swap(ohi[PAIR - 2], ohi[PAIR - 2], false, false);
            const auto l = __builtin_amdgcn_permlane32_swap(olo[PAIR - 2], olo[PAIR - 2], false, false);
            ohi[PAIR - 2] = h[0], ohi[PAIR] = h[1];
            olo[PAIR - 2] = l[0], olo[PAIR] = l[1];
        }
    }
    __device__ __forceinline__ half8 offsets_hi() const { return pack4(ohi[0], ohi[1], ohi[2], ohi[3]); }
    __device__ __forceinline__ half8 offsets_lo() const { return pack4(olo[0], olo[1], olo[2], olo[3]); }
    __device__ __forceinline__ half8 min_operand(int f) const {  // the eight mins, for the hi sums (g = 0) and the lo sums (g = 1)
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            v[i] = pk_add(__builtin_amdgcn_perm(0x64646464u, mns[f][i >> 1], (i & 1) ? 0x04030402u : 0x04010400u), 0xE400E400u);
        return pack4(v[0], v[1], v[2], v[3]);
    }
};

struct NoOffsets {  // the encodings without minima
    __device__ __forceinline__ float min_scale(int) const { return 0.0f; }
    __device__ __forceinline__ half8 min_operand(int) const { return half8{}; }
    __device__ __forceinline__ float4 offsets(int) const { return float4{}; }
    __device__ __forceinline__ float open_offsets() { return 0.0f; }
    __device__ __forceinline__ float scale_per_unit() const { return 0.0f; }
    template <int PAIR>
    __device__ __forceinline__ void add_offsets() {}
    __device__ __forceinline__ half8 offsets_hi() const { return half8{}; }
    __device__ __forceinline__ half8 offsets_lo() const { return half8{}; }
};

// Q6_K.  Half block h: code bytes ql[0..31] (quarters 0 low, 2 high nibbles) and ql[32..63] (quarters 1, 3), two more bits of all four
// quarters in qh[0..31]; a lane takes bytes 16 g .. 16 g + 15 of each.  (u - 32) 2^-24 or 2^-20 as above, then the two integer operands
// 16 (sc >> 4) q and (sc & 15) q, times 2^-19.  FLUSH: steps after which the matrix cores' sums go to the running ones.  Every instruction rounds its
// sum; with 8, which the direct kernel takes, the relative error of bf16 rows is 0.95e-7 and not 1.2e-7 (small-batch kernel: 0.95e-7), of fp32 rows 1.6e-7
// and not 2.1e-7 (1.6e-7), for up to 6 % of the time.  The shared kernel takes 8 up to 64 rows, with sums of a unit of their own (1.1e-7, 1.7e-7; 2 .. 3 % of the
// time), and 16 beyond (1.26e-7, 2.1e-7), where the plane GEMM that it replaces has 4e-7 and more.
template <int FN, int FLUSH>
struct Q6Weights : NoOffsets {
    static constexpr int kSteps = 16, kFlush = FLUSH, kPlanes = 2;
    static constexpr bool kMin = false, kPairs = false;
    using Rows = StagedRows<Q6_K_BPB, FN>;
    static constexpr int kStage = Rows::kBytes;
    Rows rows;
    const uint8_t* mine;
    int g, lane_;
    gd_u4 ql[FN][2], qh[FN];
    uint32_t sc[FN][2], d[FN];

    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* stage) {
        rows.init(t, n0, lane, stage);
        g = lane >> 5;
        lane_ = lane;
        mine = stage + (lane & 31) * Rows::kRow;
    }
    __device__ __forceinline__ void load(int unit) { rows.load(unit); }
    __device__ __forceinline__ void read_half(int h) {
#pragma unroll
        for (int f = 0; f < FN; f++) {
            const uint8_t* p = mine + f * 32 * Rows::kRow + 16 * g;
            ql[f][0] = *(const gd_u4*)(p + 64 * h);
            ql[f][1] = *(const gd_u4*)(p + (64 * h + 32));
            qh[f] = *(const gd_u4*)(p + (128 + 32 * h));
        }
    }
    __device__ __forceinline__ void open() {
        rows.to_lds(lane_);
        read_half(0);
#pragma unroll
        for (int f = 0; f < FN; f++) {
            // the lane's scales: index 2 (4 h + quarter) + g, as bytes 4 h + quarter of two dwords
            const gd_u4 s = *(const gd_u4*)(mine + f * 32 * Rows::kRow + 192);
            const uint32_t sel = g ? 0x07050301u : 0x06040200u;
            sc[f][0] = __builtin_amdgcn_perm(s.y, s.x, sel);
            sc[f][1] = __builtin_amdgcn_perm(s.w, s.z, sel);
            d[f] = *(const uint16_t*)(mine + f * 32 * Rows::kRow + 222);
        }
    }
    template <int T>
    __device__ __forceinline__ void step(int f, half8 (&b)[2]) const {
        constexpr int h = T >> 3, quarter = (T >> 1) & 3, a = T & 1;
        constexpr bool high = quarter >= 2;
        const uint32_t sb = (uint32_t)((int32_t)(sc[f][h] << (24 - 8 * quarter)) >> 24);  // sign-extended
        // sc = 16 hi + lo; low nibbles: 32 times 16 hi and lo, high nibbles (codes 16-fold): twice
        const _Float16 s1 = (_Float16)(float)((int)sb >> 4), s0 = (_Float16)(float)(sb & 15u);
        const _Float16 m1 = s1 * (_Float16)(high ? 32.0f : 512.0f), m0 = s0 * (_Float16)(high ? 2.0f : 32.0f);
        const uint32_t p1 = as_u32(half2v{m1, m1}), p0 = as_u32(half2v{m0, m0});
        constexpr uint32_t mask = high ? 0x00F000F0u : 0x000F000Fu, hm = high ? 0x03000300u : 0x00300030u;
        constexpr int bit = high ? 8 : 4;
        constexpr uint32_t minus32 = high ? 0x82008200u : 0x80208020u;  // -32 in the unit of the codes
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t x = ql[f][quarter & 1][2 * a + i], e = qh[f][2 * a + i];
            constexpr int from = 2 * quarter;
            const uint32_t e0 = bit >= from ? e << (bit - from) : e >> (from - bit);
            const uint32_t e1 = bit >= from + 8 ? e << (bit - from - 8) : e >> (from + 8 - bit);
            v[2 * i] = pk_add((x & mask) | (e0 & hm), minus32);
            v[2 * i + 1] = pk_add(((x >> 8) & mask) | (e1 & hm), minus32);
        }
        b[0] = pack4(pk_mul(v[0], p1), pk_mul(v[1], p1), pk_mul(v[2], p1), pk_mul(v[3], p1));
        b[1] = pack4(pk_mul(v[0], p0), pk_mul(v[1], p0), pk_mul(v[2], p0), pk_mul(v[3], p0));
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr (T == 7) read_half(1);  // (step 7 is unpacked)
    }
    template <int T>
    __device__ __forceinline__ void after_step(int) {}
    __device__ __forceinline__ float scale(int f) const { return h2f((uint16_t)d[f]) * 524288.0f; }
};

// GPTQ, plain groups.  Word row 32 unit + 4 blk + 2 g + a is a lane's share of step 2 blk + a.  With FN = 2 a lane owns two neighbouring columns
// (8-byte loads).  FLUSH: steps per scale block, 8 (groups that are multiples of 128) or 2 (any group: blocks of 32).  A K that is no multiple of
// 256 ends in a partial unit: its lhs columns beyond K are zeros, its words and scales the last ones of the tensors.
template <int FN, int FLUSH>
struct GptqWeights : NoOffsets {
    static constexpr int kSteps = 16, kFlush = FLUSH, kPlanes = 1;
    static constexpr bool kMin = false, kPairs = FN == 2;
    static constexpr int kBlocks = 16 / FLUSH, kStage = 0;
    const uint32_t* qw;
    const uint16_t* scales;
    const uint32_t* qzeros;
    int n, group, col, g, rows, groups;
    uint32_t q[16][FN], s_next[kBlocks], z_next[kBlocks], s_raw[kBlocks], z_raw[kBlocks];
    uint32_t top0 = code_top(0x64006400u), top1 = code_top(0x54005400u);

    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t*) {
        qw = (const uint32_t*)t.w;
        scales = t.scales;
        qzeros = t.qzeros;
        n = t.n;
        group = t.group;
        rows = t.k >> 3;
        groups = t.k / group;
        g = lane >> 5;
        col = min(n0 + FN * (lane & 31), n - FN);
    }
    __device__ __forceinline__ void load_words(int unit, int t) {
        const int row = min(32 * unit + 4 * (t >> 1), rows - 4) + (t & 1);  // (K / 8 is a multiple of 4)
        const uint32_t* p = qw + (int64_t)row * n + (uint32_t)(2 * g * n + col);
#pragma unroll
        for (int f = 0; f < FN; f++) q[t][f] = p[f];
    }
    __device__ __forceinline__ void load_head(int unit) {
#pragma unroll
        for (int i = 0; i < kBlocks; i++) {
            const int64_t gi = min((unit * 256 + i * 16 * FLUSH) / group, groups - 1);
            const uint16_t* sp = scales + gi * n + col;
            s_next[i] = sp[0];
            if constexpr (FN == 2) s_next[i] |= (uint32_t)sp[1] << 16;
            z_next[i] = qzeros[gi * (n >> 3) + (col >> 3)];
        }
    }
    __device__ __forceinline__ void load(int unit) {  // (the words of later units step by step, as those of this one are used up)
        load_head(unit);
    }
    __device__ __forceinline__ void load_first(int unit) {
        load_head(unit);
#pragma unroll
        for (int t = 0; t < 16; t++) load_words(unit, t);
    }
    __device__ __forceinline__ void open() {
#pragma unroll
        for (int i = 0; i < kBlocks; i++) {
            s_raw[i] = s_next[i];
            z_raw[i] = z_next[i];
        }
    }
    template <int T>
    __device__ __forceinline__ void before_step() {}
    template <int T>
    __device__ __forceinline__ void step(int f, half8 (&b)[1]) const {
        const uint32_t z = ((z_raw[T / FLUSH] >> (4 * ((col + f) & 7))) & 0xFu) + 1u;
        // nibbles under 0x6400 read as 1024 + q, in their place one nibble up under 0x5400 as 64 + q; the difference to 1024 (64) + zero is
        // exact.  (As fp16 subnormals, codes this small lost bits in the matrix-core sums: 3e-5 relative, against 3e-7.)
        const uint32_t m0 = 0xE400E400u | (z * 0x00010001u), m1 = 0xD400D400u | (z * 0x00100010u);
        const uint32_t x = q[T][f], y = x >> 8;
        b[0] = pack4(pk_add((x & 0x000F000Fu) | top0, m0), pk_add((x & 0x00F000F0u) | top1, m1), pk_add((y & 0x000F000Fu) | top0, m0), pk_add((y & 0x00F000F0u) | top1, m1));
    }
    template <int T>
    __device__ __forceinline__ void after_step(int next_unit) { load_words(next_unit, T); }
    template <int I>
    __device__ __forceinline__ float scale_at(int f) const { return h2f((uint16_t)(f ? s_raw[I] >> 16 : s_raw[I] & 0xffffu)); }
};

// Q4_0: the exact integer block dots of the Q8_0 lhs (codes as fp16) with q - 8, block by block.  Lane half g takes bytes 8 g .. 8 g + 7 of a
// block: its low nibbles are columns 8 g + 0..7 of the block (step a = 0), the high ones 16 + 8 g + 0..7 (a = 1).  Rows
// whose K is no multiple of 256 end in a partial unit: what lies behind the row's end is read as zeros.
template <int FN>
struct Q40Weights : NoOffsets {
    static constexpr int kSteps = 16, kFlush = 2, kPlanes = 1;
    static constexpr bool kMin = false, kPairs = false;
    static constexpr int kUnit = 8 * Q4_0_BPB, kPieces = kUnit / 16;
    static constexpr int kTotal = 32 * FN * kPieces, kLoads = (kTotal + 63) / 64, kStage = 32 * FN * kUnit;
    const uint8_t* w;
    uint8_t* lds;
    const uint8_t* mine;
    int row_bytes, g, lane_;
    uint32_t off[kLoads];
    gd_u4 raw[kLoads];
    uint32_t x[FN][2][3];  // block b in x[f][b & 1]: its eight code bytes in dwords 0, 1 (odd b) or from byte 2 of dword 0 on (even b)
    uint32_t d[FN][8];     // (of lanes g = 0; zero in the others)
    uint32_t top0 = code_top(0x64006400u), top1 = code_top(0x54005400u);
    struct __attribute__((packed, aligned(2))) Bytes16 {
        gd_u4 v;
    };

    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* stage) {
        w = t.w;
        lds = stage;
        g = lane >> 5;
        lane_ = lane;
        mine = stage + (lane & 31) * kUnit;
        row_bytes = t.k / 32 * Q4_0_BPB;
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const int i = min(j * 64 + lane, kTotal - 1), row = i / kPieces, piece = i - row * kPieces;
            off[j] = (uint32_t)min(n0 + row, t.n - 1) * (uint32_t)row_bytes + 16 * piece;
        }
    }
    __device__ __forceinline__ void load(int unit) {
        const uint8_t* b = w + (int64_t)unit * kUnit;
        const int left = row_bytes - unit * kUnit;  // bytes of the rows from here on
        if (left >= kUnit) {
#pragma unroll
            for (int j = 0; j < kLoads; j++) raw[j] = ((const Bytes16*)(b + off[j]))->v;
        } else {
#pragma unroll
            for (int j = 0; j < kLoads; j++) {
                const int i = min(j * 64 + lane_, kTotal - 1), at = (i % kPieces) * 16;
                // the last 16 bytes of the row, moved down to the place the piece would have (rows are at least 18 bytes long)
                const int over = max(at + 16 - left, 0);
                const gd_u4 v = ((const Bytes16*)(b + off[j] - over))->v;
                uint64_t lo = v.x | (uint64_t)v.y << 32, hi = v.z | (uint64_t)v.w << 32;
                if (over >= 16) lo = hi = 0;
                else if (over >= 8) { lo = hi >> (8 * over - 64); hi = 0; }
                else if (over > 0) { lo = (lo >> (8 * over)) | (hi << (64 - 8 * over)); hi >>= 8 * over; }
                raw[j] = gd_u4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
            }
        }
    }
    __device__ __forceinline__ void read_block(int b) {
#pragma unroll
        for (int f = 0; f < FN; f++) {
            const uint32_t* p = (const uint32_t*)(mine + f * 32 * kUnit + 8 * g + (b & 1 ? 18 * b + 2 : 18 * b));
            x[f][b & 1][0] = p[0];
            x[f][b & 1][1] = p[1];
            if (!(b & 1)) x[f][b & 1][2] = p[2];
        }
    }
    __device__ __forceinline__ void open() {
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            if (j * 64 + 63 < kTotal || j * 64 + lane_ < kTotal) *(gd_u4*)(lds + j * 1024 + lane_ * 16) = raw[j];
        read_block(0);
#pragma unroll
        for (int f = 0; f < FN; f++)
#pragma unroll
            for (int b = 0; b < 8; b++) d[f][b] = g ? 0u : (uint32_t)*(const uint16_t*)(mine + f * 32 * kUnit + 18 * b);
    }
    template <int T>
    __device__ __forceinline__ void step(int f, half8 (&b)[1]) const {
        constexpr int blk = T >> 1, a = T & 1;
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t q = blk & 1 ? x[f][1][i] : __builtin_amdgcn_alignbyte(x[f][0][i + 1], x[f][0][i], 2), y = q >> 8;
            if constexpr (a == 0) {
                v[2 * i] = pk_add((q & 0x000F000Fu) | top0, 0xE408E408u);  // 1024 + q - 1032
                v[2 * i + 1] = pk_add((y & 0x000F000Fu) | top0, 0xE408E408u);
            } else {
                v[2 * i] = pk_add((q & 0x00F000F0u) | top1, 0xD480D480u);  // 64 + q - 72
                v[2 * i + 1] = pk_add((y & 0x00F000F0u) | top1, 0xD480D480u);
            }
        }
        b[0] = pack4(v[0], v[1], v[2], v[3]);
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr ((T & 1) == 0 && T < 14) read_block((T >> 1) + 1);
    }
    template <int T>
    __device__ __forceinline__ void after_step(int) {}
    template <int B>
    __device__ __forceinline__ half8 scale_operand(int f) const {
        const uint32_t v = d[f][B] << (16 * (B & 1));
        return pack4(B >> 1 == 0 ? v : 0u, B >> 1 == 1 ? v : 0u, B >> 1 == 2 ? v : 0u, B >> 1 == 3 ? v : 0u);
    }
    __device__ __forceinline__ float scale(int) const { return 0.0f; }
};

// Scale blocks of 32 columns: the sums of a unit of K (eight blocks) are kept apart from the running ones, which otherwise are a chain of K / 32 rounded
// sums.  Relative error of GPTQ in groups of 32, bf16 rows: 11008 x 4096 with 300 rows 2.0e-7 -> 0.9e-7 (column kernel: 0.95e-7), 5120 x 5120
// with 700 rows 2.3e-7 -> 1.0e-7; Q4_0, where the wavefronts share the lhs, 5120 x 5120 with 700 rows 2.3e-7 -> 1.1e-7; for less than 1 % of the time.
// (fp32 rows: two products a value, no more than 2.2e-7 where the column kernel had 3.3e-7.)
constexpr bool unit_sums(int enc, int flush, bool hilo) { return (enc == QMM_Q6_K && flush == 8) || ((enc == QMM_GPTQ || enc == QMM_Q4_0) && flush == 2 && !hilo); }

template <int ENC, int FN, int FLUSH, bool CENTER>
using WeightsOf = std::conditional_t<ENC == QMM_GPTQ, GptqWeights<FN, FLUSH>, std::conditional_t<ENC == QMM_Q6_K, Q6Weights<FN, FLUSH>,
                  std::conditional_t<ENC == QMM_Q4_0, Q40Weights<FN>, KQuantWeights<ENC == QMM_Q5_K ? QMM_Q5_K : QMM_Q4_K, FN, CENTER>>>>;

// compile-time loop: f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

}  // namespace

}  // namespace qmm
