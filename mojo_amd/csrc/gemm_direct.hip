// From a few lhs rows up to a few hundred: a GEMM whose wavefronts work alone.
//
// What bounds this range is neither the weights (0.5 .. 0.8 bytes each, read once) nor the matrix cores but everything between
// launches and barriers: a conversion pass over the weights, tiles too large to fill 256 compute units, partial results that go
// through memory.  Here a wavefront owns 32 FN columns x 32 FM rows of the output over a share of K and needs no other wavefront until
// it is done: packed weights come from memory straight into its registers, are unpacked there into matrix-core operands (exact small
// integers in fp16), and the lhs operands come from L2 in operand order (1 KB contiguous per instruction), made by one small launch in
// front.  The WK wavefronts of a workgroup take WK shares of K of the same tile and add their results through LDS; where that still
// leaves compute units idle, two workgroups share a tile and add their halves atomically onto zeros (two terms: the order is
// immaterial).  No LDS traffic and no barrier inside the loop; the lhs costs 1 KB of L2 reads per FN matrix-core instructions, which is
// 1.1 PFLOP/s with FN = 2 (35 TB/s of L2 reads measured, 60 bytes per clock and compute unit).
//
// Arithmetic (exact products, fp32 sums), per scale block of a column:
//   acc += d * sum(u * a16) [+ -dmin * sum(mn * s)],  u: integer weights (sc * q, or q - zero), a16: the row scaled by a power of two and
//   narrowed to fp16 (fp32 rows: hi + residual, both products into one accumulator), s: sub-block sums of the scaled row as hi + lo.
//   Q6_K: sc * q may need 13 bits, so sc = 16 hi + lo gives two integer operands per weight (see gemm_planes.hip).
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "gemm_lhs.h"
#include "qmm_internal.h"

namespace qmm {

namespace {

typedef uint32_t gd_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t gd_u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ half2v as_h2(uint32_t x) { return __builtin_bit_cast(half2v, x); }
__device__ __forceinline__ uint32_t as_u32(half2v x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t pk_add(uint32_t x, uint32_t y) { return as_u32(as_h2(x) + as_h2(y)); }
// byte j of v under the byte `top` in both halves: with top 0x64 the fp16 pair 1024 + byte, with 0x68 2048 + 2 byte, with 0x78 32768 + 32 byte
template <int J>
__device__ __forceinline__ uint32_t byte_pair(uint32_t top4, uint32_t v) { return __builtin_amdgcn_perm(top4, v, 0x04000400u | (J << 16) | J); }

// The operand order of the lhs: step t = 2 blk + a of 16 columns holds, for half wavefront g, the columns
//   32 blk + 16 g + 8 a + slot order   (kOrderK: slots 0,2,1,3,4,6,5,7; kOrderGptq: 0,4,1,5,2,6,3,7)
constexpr int kOrderK = 0, kOrderGptq = 1;  // (Q4_0: 32 blk + 16 a + 8 g + the slots of kOrderK)

// Sizes of what the preparation launch leaves behind.  Every row tile of 32 rows: k / 16 operands of 1 KB, rounded up to whole units of 16 (fp32 lhs: pairs of
// them, hi then residual), and room for one more unit behind the last (the loop reads ahead); sums: one operand per 256 columns; inverse row scales.
struct DirectSpace {
    _Float16* a16;
    _Float16* sums;
    float* inv;
    int64_t bytes;
};
DirectSpace direct_space(void* ws, bool f32, bool with_sums, int64_t m, int64_t k) {
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t tiles = (m + 31) / 32;
    DirectSpace p;
    char* base = (char*)ws;
    int64_t off = 0;
    p.a16 = (_Float16*)base;
    off += tiles * ((k + 255) / 256) * 16384 * (f32 ? 2 : 1) + 32768;
    p.sums = (_Float16*)(base + off);
    off += with_sums ? tiles * ((k + 255) / 256) * 1024 : 0;
    p.inv = (float*)(base + off);
    off += up(tiles * 32 * 4);
    p.bytes = off;
    return p;
}

// The matrices of one launch (they share the lhs): their results, and where each ends in the grid, in eights of column tiles.
struct DirectMats {
    const uint8_t* w[kDirectMaxMats];
    float* out[kDirectMaxMats];
    int n[kDirectMaxMats], end[kDirectMaxMats];
    int count;
};

// ---------------------------------------------------------------------------------------------------------------------------
// preparation: one workgroup per lhs row (the first m workgroups), then zeroing of `out` for two workgroups per tile
// ---------------------------------------------------------------------------------------------------------------------------
template <typename AT>
__device__ __forceinline__ void load8(const AT* p, float (&v)[8]) {
    if constexpr (sizeof(AT) == 4) {
        const float4 x = *(const float4*)p, y = *(const float4*)(p + 4);
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
    } else {
        const uint4 x = *(const uint4*)p;
        const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
}
// the e-th of `count` workgroups zeroes its part of the results (m rows)
__device__ __forceinline__ void zero_out(const DirectMats& z, int m, int e, int count) {
    for (int j = 0; j < z.count; j++) {
        float* __restrict__ const out = z.out[j];
        const int64_t values = (int64_t)m * z.n[j];
        for (int64_t i = ((int64_t)e * 256 + threadIdx.x) * 4; i < values; i += (int64_t)count * 1024) {
            if (i + 3 < values) *(float4*)(out + i) = make_float4(0.f, 0.f, 0.f, 0.f);
            else
                for (int64_t q = i; q < values; q++) out[q] = 0.0f;
        }
    }
}

// Rows of one group of eight go to workgroups of one XCD (ids congruent mod 8): a 128-byte line of an operand holds eight rows.
template <typename AT, int ORDER>
__global__ __launch_bounds__(256) void direct_prep_kernel(const AT* __restrict__ a, int m, int k, DirectSpace p, int with_sums, DirectMats zero) {
    constexpr bool kF32 = sizeof(AT) == 4;
    __shared__ uint32_t wmax[4];
    const int tid = threadIdx.x, rows = (m + 63) / 64 * 64;
    if ((int)blockIdx.x >= rows) {
        zero_out(zero, m, (int)blockIdx.x - rows, (int)gridDim.x - rows);
        return;
    }
    const int b = blockIdx.x, row = (b & ~63) + (b & 7) * 8 + ((b >> 3) & 7);
    if (row >= m) return;
    const AT* ar = a + (int64_t)row * k;
    const int pieces = k >> 3;  // of eight columns, one per thread and turn
    const int steps = (k + 255) / 256 * 16;
    constexpr int kHeld = 4;    // rows of up to 8192 columns stay in registers between the search for the maximum and the narrowing
    float held[kHeld][8];
    const bool hold = pieces <= kHeld * 256;
    auto load = [&](int pc, float (&v)[8]) __attribute__((always_inline)) { load8(ar + pc * 8, v); };
    float mx = 0.0f;
    auto top = [&](const float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
    };
    if (hold) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + i * 256 < pieces) load(tid + i * 256, held[i]);
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + i * 256 < pieces) top(held[i]);
    } else {
        for (int pc = tid; pc < pieces; pc += 256) {
            float v[8];
            load(pc, v);
            top(v);
        }
    }
    const uint32_t mb = wave_max_nonneg_bits(mx);
    if ((tid & 63) == 0) wmax[tid >> 6] = mb;
    __syncthreads();
    const uint32_t mxb = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    int e = (int)((mxb >> 23) & 0xffu) - 127;
    if (e < -100 || e > 127) e = 9;  // zero, denormal or non-finite row: leave unscaled
    const float s = __uint_as_float((uint32_t)(127 + 9 - e) << 23);
    if (tid == 0) p.inv[row] = __uint_as_float((uint32_t)(127 - 9 + e) << 23);
    const int tile = row >> 5, lane = row & 31;
    auto emit = [&](int pc, float (&v)[8]) __attribute__((always_inline)) {
        constexpr int perm[2][8] = {{0, 2, 1, 3, 4, 6, 5, 7}, {0, 4, 1, 5, 2, 6, 3, 7}};
        const int blk = pc >> 2, g = (pc >> 1) & 1, step = 2 * blk + (pc & 1);
        float h[8], sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] *= s;
#pragma unroll
        for (int i = 0; i < 8; i++) h[i] = h2f(f2h(v[i]));
        gd_u4 hi;
#pragma unroll
        for (int i = 0; i < 4; i++) hi[i] = pack_half2(h[perm[ORDER][2 * i]], h[perm[ORDER][2 * i + 1]]);
        _Float16* at = p.a16 + ((int64_t)tile * steps + step) * (kF32 ? 1024 : 512) + (lane + 32 * g) * 8;
        *(gd_u4*)at = hi;
        if constexpr (kF32) {
            gd_u4 lo;
#pragma unroll
            for (int i = 0; i < 4; i++)
                lo[i] = pack_half2(v[perm[ORDER][2 * i]] - h[perm[ORDER][2 * i]], v[perm[ORDER][2 * i + 1]] - h[perm[ORDER][2 * i + 1]]);
            *(gd_u4*)(at + 512) = lo;
        }
        if (with_sums) {
#pragma unroll
            for (int i = 0; i < 8; i += 2) sum += v[i] + v[i + 1];
            sum += dpp_move<0xB1>(sum);
            sum += dpp_move<0x4E>(sum);  // the four threads of a 32-wide sub-block
            if ((pc & 3) == 0) {
                const float sh = h2f(f2h(sum));
                _Float16* sp = p.sums + ((int64_t)tile * (k >> 8) + (blk >> 3)) * 512 + lane * 8 + (blk & 7);
                sp[0] = (_Float16)sh;
                sp[256] = (_Float16)(sum - sh);
            }
        }
    };
    for (int pc = pieces + tid; pc < 2 * steps; pc += 256) {  // zeros up to a whole unit
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        emit(pc, v);
    }
    if (hold) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + i * 256 < pieces) emit(tid + i * 256, held[i]);
    } else {
        for (int pc = tid; pc < pieces; pc += 256) {
            float v[8];
            load(pc, v);
            emit(pc, v);
        }
    }
}

// The same for Q4_0: rows quantised to Q8_0, codes as fp16, no row scale; the fp16 block scales of a row as the first eight slots of the
// unit's operand in `sums` (lanes g = 0; zeros in g = 1).  Four neighbouring threads hold a block.
template <typename AT>
__global__ __launch_bounds__(256) void direct_prep_q8_kernel(const AT* __restrict__ a, int m, int k, DirectSpace p, DirectMats zero) {
    const int tid = threadIdx.x, rows = (m + 63) / 64 * 64;
    if ((int)blockIdx.x >= rows) {
        zero_out(zero, m, (int)blockIdx.x - rows, (int)gridDim.x - rows);
        return;
    }
    const int b = blockIdx.x, row = (b & ~63) + (b & 7) * 8 + ((b >> 3) & 7);
    if (row >= m) return;
    const AT* ar = a + (int64_t)row * k;
    const int pieces = k >> 3, units = (k + 255) / 256;
    const int tile = row >> 5, lane = row & 31;
    if (tid == 0) p.inv[row] = 1.0f;
    for (int pc = tid; pc < units * 32; pc += 256) {
        const int blk = pc >> 2, sub = pc & 3, g = sub & 1, step = 2 * blk + (sub >> 1);
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (pc < pieces) load8(ar + pc * 8, v);
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
        mx = fmaxf(mx, dpp_move<0xB1>(mx));
        mx = fmaxf(mx, dpp_move<0x4E>(mx));
        uint16_t dh;
        const float id = q8_0_block_rule(mx, dh);
        constexpr int perm[8] = {0, 2, 1, 3, 4, 6, 5, 7};
        gd_u4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = pack_half2((float)q8_0_code(v[perm[2 * i]], id), (float)q8_0_code(v[perm[2 * i + 1]], id));
        *(gd_u4*)(p.a16 + ((int64_t)tile * units * 16 + step) * 512 + (lane + 32 * g) * 8) = o;
        if (sub == 0) {
            uint16_t* sp = (uint16_t*)p.sums + ((int64_t)tile * units + (blk >> 3)) * 512 + lane * 8 + (blk & 7);
            sp[0] = dh;
            sp[256] = 0;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------
// the weights of one wavefront: what it holds of a unit of K, how a step's operands come out of it
// ---------------------------------------------------------------------------------------------------------------------------
struct WeightTensors {
    const uint8_t* w;        // K-quant blocks, or GPTQ qweight
    const uint16_t* scales;  // GPTQ
    const uint32_t* qzeros;
    int n, k, group;
};

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
// keep fewer bits of a sum whose operands are subnormal (fp32 rows, 2.5e-7 relative error against 6e-7 with sc q 2^-24).
template <int ENC, int FN>
struct KQuantWeights {
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
        uint32_t sp;
        if constexpr (h == 0) sp = pk_add(byte_pair<(blk & 3)>(0x78787878u, scs[f][blk >> 2]), 0xF800F800u);  // 32768 + 32 sc - 32768
        else sp = pk_add(byte_pair<(blk & 3)>(0x68686868u, scs[f][blk >> 2]), 0xE800E800u);                   // 2048 + 2 sc - 2048
        constexpr uint32_t mask = h == 0 ? 0x000F000Fu : 0x00F000F0u;
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t x = q[f][c & 1][2 * a + i], y = x >> 8;
            v[2 * i] = x & mask;
            v[2 * i + 1] = y & mask;
            if constexpr (ENC == QMM_Q5_K) {
                constexpr int bit = h == 0 ? 4 : 8;  // where the fifth bit goes, from bit blk of its byte
                constexpr uint32_t fm = h == 0 ? 0x00100010u : 0x01000100u;
                const uint32_t e = fifth[f][2 * a + i];
                v[2 * i] |= (bit >= blk ? e << (bit - blk) : e >> (blk - bit)) & fm;
                v[2 * i + 1] |= (bit >= blk + 8 ? e << (bit - blk - 8) : e >> (blk + 8 - bit)) & fm;
            }
        }
        b[0] = pack4(pk_mul(v[0], sp), pk_mul(v[1], sp), pk_mul(v[2], sp), pk_mul(v[3], sp));
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr ((T & 3) == 0 && T < 12) read_codes((T >> 2) + 1);
    }
    template <int T>
    __device__ __forceinline__ void after_step(int) {}
    __device__ __forceinline__ float scale(int f) const { return h2f((uint16_t)(dm[f] & 0xffffu)) * 524288.0f; }
    __device__ __forceinline__ float min_scale(int f) const { return -h2f((uint16_t)(dm[f] >> 16)); }
    __device__ __forceinline__ half8 min_operand(int f) const {  // the eight mins, for the hi sums (g = 0) and the lo sums (g = 1)
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            v[i] = pk_add(__builtin_amdgcn_perm(0x64646464u, mns[f][i >> 1], (i & 1) ? 0x04030402u : 0x04010400u), 0xE400E400u);
        return pack4(v[0], v[1], v[2], v[3]);
    }
};

// Q6_K.  Half block h: code bytes ql[0..31] (quarters 0 low, 2 high nibbles) and ql[32..63] (quarters 1, 3), two more bits of all four
// quarters in qh[0..31]; a lane takes bytes 16 g .. 16 g + 15 of each.  (u - 32) 2^-24 or 2^-20 as above, then the two integer operands
// 16 (sc >> 4) q and (sc & 15) q, times 2^-19.
template <int FN>
struct Q6Weights {
    static constexpr int kSteps = 16, kFlush = 16, kPlanes = 2;
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
    __device__ __forceinline__ float min_scale(int) const { return 0.0f; }
    __device__ __forceinline__ half8 min_operand(int) const { return half8{}; }
};

// GPTQ, plain groups.  Word row 32 unit + 4 blk + 2 g + a is a lane's share of step 2 blk + a.  With FN = 2 a lane owns two neighbouring columns
// (8-byte loads).  FLUSH: steps per scale block, 8 (groups that are multiples of 128) or 2 (any group: blocks of 32).  A K that is no multiple of
// 256 ends in a partial unit: its lhs columns beyond K are zeros, its words and scales the last ones of the tensors.
template <int FN, int FLUSH>
struct GptqWeights {
    static constexpr int kSteps = 16, kFlush = FLUSH, kPlanes = 1;
    static constexpr bool kMin = false, kPairs = FN == 2;
    static constexpr int kBlocks = 16 / FLUSH, kStage = 0;
    const uint32_t* qw;
    const uint16_t* scales;
    const uint32_t* qzeros;
    int n, group, col, g, rows, groups;
    uint32_t q[16][FN], s_next[kBlocks], z_next[kBlocks], s_raw[kBlocks], z_raw[kBlocks];

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
        b[0] = pack4(pk_add((x & 0x000F000Fu) | 0x64006400u, m0), pk_add((x & 0x00F000F0u) | 0x54005400u, m1),
                     pk_add((y & 0x000F000Fu) | 0x64006400u, m0), pk_add((y & 0x00F000F0u) | 0x54005400u, m1));
    }
    template <int T>
    __device__ __forceinline__ void after_step(int next_unit) { load_words(next_unit, T); }
    template <int I>
    __device__ __forceinline__ float scale_at(int f) const { return h2f((uint16_t)(f ? s_raw[I] >> 16 : s_raw[I] & 0xffffu)); }
    __device__ __forceinline__ float min_scale(int) const { return 0.0f; }
    __device__ __forceinline__ half8 min_operand(int) const { return half8{}; }
};

// Q4_0: the exact integer block dots of the Q8_0 lhs (codes as fp16) with q - 8, block by block.  Lane half g takes bytes 8 g .. 8 g + 7 of a
// block: its low nibbles are columns 8 g + 0..7 of the block (step a = 0), the high ones 16 + 8 g + 0..7 (a = 1).  Rows
// whose K is no multiple of 256 end in a partial unit: what lies behind the row's end is read as zeros.
template <int FN>
struct Q40Weights {
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
                v[2 * i] = pk_add((q & 0x000F000Fu) | 0x64006400u, 0xE408E408u);  // 1024 + q - 1032
                v[2 * i + 1] = pk_add((y & 0x000F000Fu) | 0x64006400u, 0xE408E408u);
            } else {
                v[2 * i] = pk_add((q & 0x00F000F0u) | 0x54005400u, 0xD480D480u);  // 64 + q - 72
                v[2 * i + 1] = pk_add((y & 0x00F000F0u) | 0x54005400u, 0xD480D480u);
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
    __device__ __forceinline__ float min_scale(int) const { return 0.0f; }
    __device__ __forceinline__ half8 min_operand(int) const { return half8{}; }
};

template <int ENC, int FN, int FLUSH>
using WeightsOf = std::conditional_t<ENC == QMM_GPTQ, GptqWeights<FN, FLUSH>, std::conditional_t<ENC == QMM_Q6_K, Q6Weights<FN>,
                  std::conditional_t<ENC == QMM_Q4_0, Q40Weights<FN>, KQuantWeights<ENC == QMM_Q5_K ? QMM_Q5_K : QMM_Q4_K, FN>>>>;

constexpr int direct_ahead(int flush, int fm, int fn, bool hilo) {
    if (fm * fn == 2) return hilo ? 4 : 8;
    return flush == 2 && hilo ? 8 : 16;
}

template <typename W>
constexpr int direct_slot(int frags) { return W::kStage > frags * 4096 ? W::kStage : frags * 4096; }

// compile-time loop: f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

}  // namespace

// Workgroup id -> tile: ids congruent mod 8 run on one XCD; there the row tiles of a column tile follow each other, so that its L2 fetches the
// weights once.  shares: workgroups per tile (1, or 2 that add onto zeros).
template <int ENC, int FLUSH, int FM, int FN, int WK, bool HILO>
__global__ __launch_bounds__(64 * WK, 2) void gemm_direct_kernel(WeightTensors wt, DirectMats mats, DirectSpace p, uint16_t* __restrict__ out16, int m, int units,
                                                                int tiles_m, int shares) {
    using W = WeightsOf<ENC, FN, FLUSH>;
    constexpr int kSlot = direct_slot<W>(FM * FN);
    extern __shared__ __attribute__((aligned(16))) float red[];  // a slot per wavefront: its packed rows, at the end its results [FM * FN][4][64] float4
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int i = (int)(blockIdx.x >> 3), tile_m = i % tiles_m, rest = i / tiles_m, share = rest % shares;
    int section = rest / shares, first = 0;
    wt.w = mats.w[0], wt.n = mats.n[0];
    float* __restrict__ out = mats.out[0];
#pragma unroll
    for (int j = 1; j < kDirectMaxMats; j++)
        if (j < mats.count && section >= mats.end[j - 1]) wt.w = mats.w[j], wt.n = mats.n[j], out = mats.out[j], first = mats.end[j - 1];
    const int tile_n = (section - first) * 8 + (int)(blockIdx.x & 7);
    if (tile_n * 32 * FN >= wt.n) return;
    const int n0 = tile_n * 32 * FN, m0 = tile_m * 32 * FM;
    // this wavefront's units of K
    const int parts = WK * shares, part = share * WK + wave;
    const int u0 = (int)((unsigned)units * (unsigned)part / (unsigned)parts), u1 = (int)((unsigned)units * (unsigned)(part + 1) / (unsigned)parts);

    constexpr int kParts = FM * FN * 4, kMine = (kParts + WK - 1) / WK;  // parts of the tile (four rows per half wavefront), of which this wavefront stores kMine
    float inv[kMine][4];
#pragma unroll
    for (int e = 0; e < kMine; e++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int part_e = min(e * WK + wave, kParts - 1), row = m0 + 32 * ((part_e >> 2) / FN) + 8 * (part_e & 3) + 4 * (lane >> 5) + r;
            inv[e][r] = p.inv[min(row, m - 1)];
        }
    float16v T[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int b = 0; b < FN; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) T[a][b][r] = 0.0f;

    if (u0 < u1) {
        // Lhs operands are loaded kAhead steps ahead.  Loads return in the order they were issued, so an lhs operand (from L2) waits for
        // the weights (from memory) requested before it: a whole unit ahead where the registers allow it.
        constexpr int kPer = HILO ? 2 : 1, kAhead = direct_ahead(FLUSH, FM, FN, HILO);
        const float16v zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        W w;
        w.init(wt, n0, lane, (uint8_t*)red + wave * kSlot);
        if constexpr (ENC == QMM_GPTQ) w.load_first(u0);
        else w.load(u0);
        const int64_t row_bytes = (int64_t)units * W::kSteps * 1024 * kPer;  // of a row tile
        const uint8_t* ap[FM];
#pragma unroll
        for (int a = 0; a < FM; a++) {
            const int tile = min(tile_m * FM + a, (m - 1) >> 5);
            ap[a] = (const uint8_t*)p.a16 + tile * row_bytes + (int64_t)u0 * W::kSteps * 1024 * kPer;
        }
        const uint32_t l16 = lane * 16;
        half8 af[FM][kAhead][kPer];
        auto load_lhs = [&](int step, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int a = 0; a < FM; a++)
#pragma unroll
                for (int q = 0; q < kPer; q++) af[a][slot][q] = *(const half8*)(ap[a] + (step * kPer + q) * 1024 + l16);
        };
#pragma unroll
        for (int t = 0; t < kAhead; t++) load_lhs(t, t);
        for (int u = u0; u < u1; u++) {
            const bool more = u + 1 < u1;
            w.open();
            if (more) w.load(u + 1);
            float16v P[FM][FN];
            half8 sf[FM];
            if constexpr (W::kMin || ENC == QMM_Q4_0) {
#pragma unroll
                for (int a = 0; a < FM; a++) {
                    const int tile = min(tile_m * FM + a, (m - 1) >> 5);
                    sf[a] = *(const half8*)((const uint8_t*)p.sums + ((int64_t)tile * units + u) * 1024 + l16);
                }
            }
            half8 b[2][FN][W::kPlanes];
#pragma unroll
            for (int f = 0; f < FN; f++) w.template step<0>(f, b[0][f]);
            __builtin_amdgcn_sched_barrier(0);
            // One step: its matrix-core instructions, the unpacking of the next step's weights between them, loads for later.  (The fences keep
            // the compiler from moving the loads next to their use to save registers.)
            unrolled<W::kSteps>([&](auto tt) __attribute__((always_inline)) {
                constexpr int t = decltype(tt)::value, slot = t % kAhead, cur = t & 1;
                constexpr int kMfma = FM * FN * kPer * W::kPlanes;
#pragma unroll
                for (int pl = 0; pl < W::kPlanes; pl++)
#pragma unroll
                    for (int q = 0; q < kPer; q++)
#pragma unroll
                        for (int a = 0; a < FM; a++)
#pragma unroll
                            for (int f = 0; f < FN; f++) {
                                if (t % W::kFlush == 0 && pl == 0 && q == 0) P[a][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a][slot][q], b[cur][f][pl], zero16, 0, 0, 0);
                                else P[a][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a][slot][q], b[cur][f][pl], P[a][f], 0, 0, 0);
                            }
                if constexpr (t + 1 < W::kSteps) {
                    w.template before_step<t>();
#pragma unroll
                    for (int f = 0; f < FN; f++) w.template step<t + 1>(f, b[cur ^ 1][f]);
                }
                if (more || t + kAhead < W::kSteps) load_lhs(t + kAhead, slot);
                if (more) {
                    if constexpr (t > 0) w.template after_step<t - 1>(u + 1);
                    if constexpr (t + 1 == W::kSteps) w.template after_step<t>(u + 1);
                }
                unrolled<kMfma>([&](auto) __attribute__((always_inline)) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, (W::kPlanes == 2 ? 28 : 11) * FN / kMfma + 1, 0);
                });
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (t % W::kFlush == W::kFlush - 1) {
#pragma unroll
                    for (int f = 0; f < FN; f++) {
                        if constexpr (ENC == QMM_Q4_0) {
                            // the scales of a block as a matrix: the lhs scale in slot t / 2 times the weight scale in the same slot
                            const half8 dw = w.template scale_operand<t / 2>(f);
#pragma unroll
                            for (int a = 0; a < FM; a++) {
                                const float16v S = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[a], dw, zero16, 0, 0, 0);
#pragma unroll
                                for (int r = 0; r < 16; r++) T[a][f][r] = fmaf(P[a][f][r], S[r], T[a][f][r]);
                                asm volatile("" : "+v"(T[a][f]));
                            }
                            continue;
                        }
                        float d = 0.0f;
                        if constexpr (ENC == QMM_GPTQ) d = w.template scale_at<t / W::kFlush>(f);
                        else d = w.scale(f);
#pragma unroll
                        for (int a = 0; a < FM; a++) {
#pragma unroll
                            for (int r = 0; r < 16; r++) T[a][f][r] = fmaf(d, P[a][f][r], T[a][f][r]);
                            // (left to itself the compiler puts these off and keeps the P of every scale block)
                            asm volatile("" : "+v"(T[a][f]));
                        }
                        if constexpr (W::kMin) {
                            const half8 mo = w.min_operand(f);
                            const float dmin = w.min_scale(f);
#pragma unroll
                            for (int a = 0; a < FM; a++) {
                                const float16v M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[a], mo, zero16, 0, 0, 0);
#pragma unroll
                                for (int r = 0; r < 16; r++) T[a][f][r] = fmaf(dmin, M[r], T[a][f][r]);
                            }
                        }
                    }
                }
            });
#pragma unroll
            for (int a = 0; a < FM; a++) ap[a] += W::kSteps * 1024 * kPer;
        }
    }

    // the WK shares of K, added in order; then every wavefront stores its part of the tile
    float4* rp = (float4*)red;
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int f = 0; f < FN; f++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                rp[wave * (kSlot / 16) + (a * FN + f) * 256 + j * 64 + lane] = make_float4(T[a][f][4 * j], T[a][f][4 * j + 1], T[a][f][4 * j + 2], T[a][f][4 * j + 3]);
    __syncthreads();
    const int nl = lane & 31, g = lane >> 5;
#pragma unroll
    for (int e0 = 0; e0 < kParts; e0 += WK) {
        const int e = e0 + wave;
        if (kParts % WK != 0 && e >= kParts) break;
        const int frag = e >> 2, j = e & 3, a = frag / FN, f = frag % FN;
        float4 v = rp[frag * 256 + j * 64 + lane];
#pragma unroll
        for (int q = 1; q < WK; q++) {
            const float4 x = rp[q * (kSlot / 16) + frag * 256 + j * 64 + lane];
            v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
        }
        const int col = W::kPairs ? n0 + 2 * nl + f : n0 + 32 * f + nl;
        const float vv[4] = {v.x, v.y, v.z, v.w};
        if (col < wt.n) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = m0 + 32 * a + 8 * j + 4 * g + r;
                if (row < m) {
                    const float x = vv[r] * inv[e0 / WK][r];
                    const int64_t at = (int64_t)row * wt.n + col;
                    if (shares > 1) unsafeAtomicAdd(out + at, x);
                    else if (out16) out16[at] = f2bf(x);
                    else out[at] = x;
                }
            }
        }
    }
}

namespace {

struct DirectPlan {
    int fm, fn, wk, shares;
};

int64_t direct_units(int64_t k) { return (k + 255) / 256; }

// What a call takes, in microseconds: launches and the preparation of the lhs, a fixed part per round of workgroups (eight wavefronts fill
// a compute unit, four half of it), the units of K that a wavefront walks, and terms for the weights, the lhs and the results.  Fitted to 143
// problems per encoding and lhs type (N 512 .. 28672, K 1024 .. 14336, 4 .. 512 rows) in every plan: 4 .. 8 % mean error, and the plan
// it picks is within 1 % of the best one on average (3 % for GPTQ with a bf16 lhs).
struct DirectCost {
    float base, round, weights, lhs, out;  // us, us, us per MB of packed weights, us per million lhs values, us per million results and share
    float unit[6];                         // us per unit of K: the plans of kDirectPlans
};
constexpr DirectPlan kDirectPlans[6] = {{1, 1, 8, 0}, {2, 1, 8, 0}, {1, 2, 8, 0}, {1, 1, 4, 0}, {2, 1, 4, 0}, {1, 2, 4, 0}};
constexpr DirectCost kDirectCost[6][2] = {
    // bf16 lhs; fp32 lhs
    {{3.98f, 1.61f, 0.18f, 3.99f, 2.25f, {2.43f, 3.65f, 4.78f, 1.86f, 2.70f, 3.76f}}, {3.99f, 1.60f, 0.18f, 3.98f, 2.32f, {2.43f, 3.63f, 4.77f, 1.86f, 2.70f, 3.75f}}},  // Q4_0
    {{3.94f, 1.39f, 0.15f, 4.32f, 2.03f, {2.08f, 2.81f, 3.01f, 1.43f, 1.99f, 2.13f}}, {3.42f, 1.40f, 0.18f, 7.65f, 3.27f, {3.19f, 4.39f, 3.95f, 2.13f, 3.06f, 2.62f}}},  // Q4_K
    {{3.90f, 1.46f, 0.14f, 4.31f, 2.37f, {2.38f, 3.02f, 3.76f, 1.66f, 2.14f, 2.59f}}, {3.36f, 1.52f, 0.16f, 7.53f, 3.65f, {3.46f, 4.46f, 4.43f, 2.29f, 3.08f, 2.91f}}},  // Q5_K
    {{3.71f, 1.15f, 0.18f, 4.46f, 3.39f, {3.08f, 3.97f, 7.05f, 2.19f, 2.75f, 5.49f}}, {3.00f, 1.77f, 0.22f, 7.86f, 4.87f, {4.39f, 5.70f, 7.66f, 3.01f, 3.67f, 5.98f}}},  // Q6_K
    {{4.74f, 0.70f, 0.14f, 3.76f, 2.23f, {1.98f, 3.12f, 3.22f, 1.48f, 2.43f, 2.28f}}, {3.48f, 1.55f, 0.16f, 6.98f, 3.33f, {3.20f, 4.42f, 4.00f, 2.35f, 3.20f, 2.87f}}},  // GPTQ, groups of 128
    {{4.99f, 0.29f, 0.14f, 3.82f, 3.07f, {2.87f, 4.18f, 4.52f, 2.05f, 3.04f, 3.16f}}, {3.78f, 1.19f, 0.14f, 6.67f, 3.76f, {3.83f, 5.23f, 5.14f, 2.79f, 3.72f, 3.56f}}},  // GPTQ, other groups
};
double direct_us(const DirectCost& c, int plan, int shares, int encoding, int64_t m, int64_t n, int64_t k) {
    const DirectPlan& p = kDirectPlans[plan];
    const int64_t wgs = ((m + 32 * p.fm - 1) / (32 * p.fm)) * ((n + 32 * p.fn - 1) / (32 * p.fn)) * shares;
    const int64_t slots = p.wk == 8 ? 256 : 512, rounds = (wgs + slots - 1) / slots, walk = (direct_units(k) + p.wk * shares - 1) / (p.wk * shares);
    const double bytes = encoding == QMM_Q6_K ? 0.82 : encoding == QMM_Q5_K ? 0.69 : 0.56;
    return c.base + rounds * (c.round + walk * c.unit[plan]) + c.weights * (bytes * n * k * 1e-6) + c.lhs * (m * k * 1e-6) + c.out * (m * n * 1e-6) * shares;
}
// whole_tiles: one workgroup per tile (bf16 results are stored, not added up); like: with that plan's cut of K
DirectPlan direct_plan(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, bool whole_tiles, const DirectPlan* like = nullptr) {
    const int row = encoding == QMM_Q4_0 ? 0 : encoding == QMM_Q4_K ? 1 : encoding == QMM_Q5_K ? 2 : encoding == QMM_Q6_K ? 3 : group % 128 == 0 ? 4 : 5;
    const DirectCost& c = kDirectCost[row][lhs_dtype == QMM_F32 ? 1 : 0];
    DirectPlan best{1, 1, 8, 1};
    double best_us = 1e30;
    for (int i = 0; i < 6; i++)
        for (int shares = 1; shares <= (whole_tiles ? 1 : 2); shares++) {
            if (like && (kDirectPlans[i].wk != like->wk || shares != like->shares)) continue;
            const double t = direct_us(c, i, shares, encoding, m, n, k);
            if (t < best_us) {
                best_us = t;
                best = kDirectPlans[i];
                best.shares = shares;
            }
        }
    return best;
}

template <int ENC, int FLUSH, int FM, int FN, int WK, bool HILO>
hipError_t run_direct(const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units, int shares, hipStream_t s) {
    const int tiles_m = (int)((m + 32 * FM - 1) / (32 * FM));
    int eights = 0;
    for (int j = 0; j < mats.count; j++) mats.end[j] = eights += (mats.n[j] + 256 * FN - 1) / (256 * FN);
    constexpr int lds = WK * direct_slot<WeightsOf<ENC, FN, FLUSH>>(FM * FN);
    hipError_t e = allow_full_lds<gemm_direct_kernel<ENC, FLUSH, FM, FN, WK, HILO>>();
    if (e != hipSuccess) return e;
    gemm_direct_kernel<ENC, FLUSH, FM, FN, WK, HILO><<<dim3((unsigned)(8 * eights * tiles_m * shares)), dim3(64 * WK), lds, s>>>(wt, mats, p, out16, (int)m,
                                                                                                                              units, tiles_m, shares);
    return hipGetLastError();
}

template <int ENC, int FLUSH, bool HILO>
hipError_t run_direct_plan(const DirectPlan& pl, const WeightTensors& wt, const DirectMats& mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units,
                           hipStream_t s) {
#define QMM_GD(FM, FN, WK) \
    if (pl.fm == FM && pl.fn == FN && pl.wk == WK) return run_direct<ENC, FLUSH, FM, FN, WK, HILO>(wt, mats, p, out16, m, units, pl.shares, s)
    QMM_GD(1, 1, 8);
    QMM_GD(2, 1, 8);
    QMM_GD(1, 2, 8);
    QMM_GD(1, 2, 4);
    QMM_GD(1, 1, 4);
    QMM_GD(2, 1, 4);
#undef QMM_GD
    return hipErrorInvalidValue;
}

}  // namespace

bool gemm_direct_wanted(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    if (kernel_disabled("direct") || k % (encoding == QMM_GPTQ || encoding == QMM_Q4_0 ? 32 : 256) || n * k >= ((int64_t)1 << 32)) return false;
    if (encoding == QMM_GPTQ && (n % 8 || group % 32)) return false;
    // Served from `from` rows on, where this kernel's time crosses that of the small-batch kernels (passes of four to sixteen rows over
    // the weights; at their best on long weight matrices and on the row lengths their wavefronts divide evenly, 512, 2048 or 4096 values;
    // this kernel has no such preference), and up to where it crosses that of the GEMMs that unpack a tile or all weights once and then
    // share them (r = outputs, w = weights, in Mi; beyond about 1100 rows the lhs no longer stays in an L2).  Both lines were fitted to
    // timings of 4700 calls, 512 x 512 .. 28672 x 4096 with K of 512 .. 14336 and 1 .. 2048 rows: within 2 % on average of always taking
    // the faster of the two.  E.g. 5120 x 5120, 17 bf16 rows: Q4_0 22 -> 16 us, Q4_K 19.6 -> 14.4, Q5_K 34 -> 15.7, Q6_K 54 -> 17.9.
    const bool f32 = lhs_dtype == QMM_F32, wide = n >= 6000;
    const double w = (double)n * k / (1 << 20), r = (double)m * n / (1 << 20);
    int64_t from = 17;
    double most = 2.75;      // bf16 outputs at which the other kernels' matrix products, which convert once for all rows, take over
    int64_t anyway = 0;      // rows up to which the number of outputs does not matter
    switch (encoding) {
        case QMM_Q4_0:
            from = wide && k <= 1024 ? 3 : k <= 2048 ? 5 : 17;
            most = 3.5, anyway = 450;
            break;
        case QMM_Q4_K:
            // (with few long rows the small-batch kernel cuts K to fill the part)
            from = n >= 2048 && (k <= 1024 || (k < 1536 && w <= 8)) ? 2
                   : !f32 && k > 4096 && n <= 4096 && gemv_q4_k_mm_plain_workspace_bytes(lhs_dtype, m, n, k) == 0 ? 5 : 9;
            if (k > 4096) most = 1.3;
            break;
        case QMM_Q5_K:
            from = wide && k <= 2048 ? 2 : n >= 2048 && (k % 512 || w <= (f32 ? 16 : 24)) ? 3 : w <= 32 ? 5 : f32 ? 9 : 17;
            break;
        case QMM_Q6_K:
            if (f32) from = k % 2048 == 0 ? 9 : wide ? 3 : n >= 2048 ? 4 : 6;
            else from = k % 2048 == 0 && !(wide && k <= 2048) ? (w <= 30 ? 5 : 17) : wide ? 2 : n >= 2048 ? 3 : 6;
            most = 3.5, anyway = 450;
            break;
        case QMM_GPTQ:
            // Groups that are no multiple of 128: the alternative is the decode kernel, eight rows a pass.
            if (group % 128) return m >= (k >= 7936 && n <= 4096 ? 1 : k >= 2048 ? 2 : w >= 1 ? 3 : 5);
            from = !f32 || k < 2048 ? 17 : k <= 8192 ? 8 : 9;
            if (k > 4096) most = 1.3;
            break;
        default: return false;
    }
    if (m < from) return false;
    if (r <= (f32 && encoding != QMM_Q4_0 ? 1.6 : 1)) return true;
    // fp32 rows are split in two fp16 terms here and in the other kernels, so both multiply twice
    if (f32) return m <= (w <= 24 || (encoding != QMM_Q4_0 && encoding != QMM_GPTQ) ? 720 : 450) || (k <= 1024 ? r <= 6 : m < 1100 && r <= 3.5);
    return m <= anyway || (m <= 1100 && r <= most);
}

int64_t gemm_direct_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t k) {
    return direct_space(nullptr, lhs_dtype == QMM_F32 && encoding != QMM_Q4_0, encoding == QMM_Q4_K || encoding == QMM_Q5_K || encoding == QMM_Q4_0, m, k).bytes;
}

// Several matrices: one preparation, and one launch for all those whose own plans cut K the same way (the order of the sums is that of a
// call of its own; the tile is the one that suits them together).  q | k | v of 4096 | 1024 | 1024 x 4096 with 16 rows: one launch for three.
hipError_t launch_gemm_direct(int encoding, const void* lhs, int lhs_dtype, int count, const void* const* ws, const int64_t* ns, float* const* outs,
                              const uint16_t* scales, const uint32_t* qzeros, int group, int64_t m, int64_t k, uint16_t* out16, void* workspace,
                              hipStream_t s) {
    const bool q40 = encoding == QMM_Q4_0, f32 = lhs_dtype == QMM_F32, sums = encoding == QMM_Q4_K || encoding == QMM_Q5_K || q40;
    if (count < 1 || count > kDirectMaxMats) return hipErrorInvalidValue;
    const DirectSpace p = direct_space(workspace, f32 && !q40, sums, m, k);
    DirectPlan plans[kDirectMaxMats];
    DirectMats zero{};
    int64_t zeros = 0;
    for (int j = 0; j < count; j++) {
        plans[j] = direct_plan(encoding, lhs_dtype, m, ns[j], k, group, out16 != nullptr);
        if (plans[j].shares > 1) zero.out[zero.count] = outs[j], zero.n[zero.count++] = (int)ns[j], zeros = std::max(zeros, m * ns[j]);
    }
    const unsigned grid = (unsigned)((m + 63) / 64 * 64 + std::min<int64_t>(1024, (zeros + 4095) / 4096));
    if (q40) {
        if (f32) direct_prep_q8_kernel<float><<<dim3(grid), dim3(256), 0, s>>>((const float*)lhs, (int)m, (int)k, p, zero);
        else direct_prep_q8_kernel<uint16_t><<<dim3(grid), dim3(256), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, zero);
    } else if (encoding == QMM_GPTQ) {
        if (f32) direct_prep_kernel<float, kOrderGptq><<<dim3(grid), dim3(256), 0, s>>>((const float*)lhs, (int)m, (int)k, p, sums, zero);
        else direct_prep_kernel<uint16_t, kOrderGptq><<<dim3(grid), dim3(256), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, sums, zero);
    } else {
        if (f32) direct_prep_kernel<float, kOrderK><<<dim3(grid), dim3(256), 0, s>>>((const float*)lhs, (int)m, (int)k, p, sums, zero);
        else direct_prep_kernel<uint16_t, kOrderK><<<dim3(grid), dim3(256), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, sums, zero);
    }
    hipError_t e = hipGetLastError();
    const WeightTensors wt{nullptr, scales, qzeros, 0, (int)k, group};
    const int units = (int)direct_units(k);
    bool done[kDirectMaxMats] = {};
    for (int j = 0; j < count && e == hipSuccess; j++) {
        if (done[j]) continue;
        DirectPlan pl = plans[j];
        DirectMats mats{};
        int64_t n = 0;
        for (int i = j; i < count; i++) {
            if (done[i] || plans[i].wk != pl.wk || plans[i].shares != pl.shares) continue;
            mats.w[mats.count] = (const uint8_t*)ws[i], mats.out[mats.count] = outs[i], mats.n[mats.count++] = (int)ns[i];
            n += ns[i];
            done[i] = true;
        }
        if (mats.count > 1) pl = direct_plan(encoding, lhs_dtype, m, n, k, group, false, &pl);
#define QMM_GD_ENC(ENC, FLUSH) \
    e = f32 ? run_direct_plan<ENC, FLUSH, true>(pl, wt, mats, p, out16, m, units, s) : run_direct_plan<ENC, FLUSH, false>(pl, wt, mats, p, out16, m, units, s)
        if (q40) e = run_direct_plan<QMM_Q4_0, 2, false>(pl, wt, mats, p, out16, m, units, s);
        else if (encoding == QMM_Q4_K) QMM_GD_ENC(QMM_Q4_K, 16);
        else if (encoding == QMM_Q5_K) QMM_GD_ENC(QMM_Q5_K, 16);
        else if (encoding == QMM_Q6_K) QMM_GD_ENC(QMM_Q6_K, 16);
        else if (group % 128 == 0) QMM_GD_ENC(QMM_GPTQ, 8);
        else QMM_GD_ENC(QMM_GPTQ, 2);
#undef QMM_GD_ENC
    }
    return e;
}

}  // namespace qmm
