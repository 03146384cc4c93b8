// The direct GEMM (gemm_direct.hip) for products from some tens of rows on: lhs and packed weights go to LDS by themselves.
//
// gemm_shared.hip has the same division of labour (wavefronts side by side share the lhs, each unpacks the weights of its 32 columns between the matrix-core
// instructions), but brings everything through registers, which leaves room for 64 rows a wavefront: 8.5 vector instructions a matrix-core instruction, where
// a wavefront of those hides four (32 cycles against 12 + 4 each), and 2.3 us a unit of 256 columns for 64 x 256 results.  Here loads go from
// memory to LDS directly (load16_to_lds) and hold no registers while they are on their way, so that a wavefront takes up to 128 rows: 5 vector instructions
// a matrix-core instruction, 2.4 .. 2.9 us a unit for 128 x 256 results.  What bounds a unit now: the matrix cores (2.2 us of it, at the 1.7 GHz that the power leaves them) and the loads to
// LDS, 16 cycles of a compute unit a KB (reads from LDS take 4), which overlap less than they might; then a barrier every four or eight steps.  By the counters (profiles/staged_gemm__counters.txt) the matrix cores of the compute units in use are busy 0.41 .. 0.61 of a launch of
// 40 us and more (0.26 of one of 20), a wavefront waits 0.26 .. 0.39 of its time, 0.02 .. 0.03 for LDS, which is active 0.19 .. 0.32 of it.  What bounds a call of a few units: 14 us
// around them (the preparation 2.6, the boundary between the launches 2.4, the way to the first unit 3, the results 3 .. 4).
//
// us, without this kernel / with it, weights from memory (profiles/staged_gemm__plans.txt): Q4_K 14336 x 4096 200 bf16 rows 53 / 44, 320 85 / 60, 4096 x 4096 200 rows 25 / 22,
// 4096 x 14336 2048 rows 301 / 261; Q5_K 32000 x 4096 200 rows 167 / 82; GPTQ 14336 x 4096 160 rows 52 / 33; Q6_K 4096 x 14336 500 rows 143 / 121; Q4_K 14336 x 4096 1300 fp32 rows
// 525 / 347.  Over 1215 problems from 33 rows on, geometric means by encoding: 0.87 .. 0.95 (bf16 rows) and 0.90 .. 0.96 (fp32 rows) of what it was within the rows that the direct and
// shared kernels served, 0.80 .. 0.85 and 0.65 .. 0.71 beyond.
//
// Tried without gain: 64 x 64 results a wavefront with one wavefront a SIMD (nothing hides its waits: 2.1 us for 64 x 256); wavefronts that load only weights or
// only lhs, with the weights two units ahead; chunks of the lhs half as long and twice as many or of two steps with up to six buffers (14336 x 4096 200 rows 38.2 / 39.9 us, 4096 x 14336 54.5 / 65.4);
// one buffer for the packed weights of Q6_K and chunks twice as long (4096 x 14336 500 rows 113.8 / 113.2).
#include "gemm_direct.h"
#include "lds_stream.h"

namespace qmm {

namespace {

// The weights of one wavefront: 32 columns, two buffers of a unit of K in LDS that only it writes (issue, a load at a time) and reads (open, before_step).
// Q4_K, Q5_K: rows as they lie in memory.
template <int ENC, bool CENTER>
struct StagedK : KQuantWeights<ENC, 1, CENTER> {
    using Base = KQuantWeights<ENC, 1, CENTER>;
    using Rows = typename Base::Rows;
    static constexpr int kLoads = Rows::kLoads;
    uint32_t stage_lds;
    const uint8_t* stage;
    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* at) {
        Base::init(t, n0, lane, at);
        stage_lds = lds_address(at);
        stage = this->mine;
    }
    template <int J>
    __device__ __forceinline__ void issue(int unit, int buf) {
        if (J * 64 + 63 < Rows::kTotal || J * 64 + this->lane_ < Rows::kTotal)
            load16_to_lds(this->rows.off[J], this->rows.w + (int64_t)unit * Rows::kRow, stage_lds + buf * Base::kStage + J * 1024);
    }
    __device__ __forceinline__ void open(int, int buf) {
        this->mine = stage + buf * Base::kStage;
        this->read_head();
    }
};

// GPTQ, plain groups, K a multiple of 256 (the packed words of a unit: 32 rows).  FLUSH as for GptqWeights.
template <int FLUSH>
struct StagedGptq : NoOffsets {
    static constexpr int kSteps = 16, kFlush = FLUSH, kPlanes = 1;
    static constexpr bool kMin = false;
    static constexpr int kBlocks = 16 / FLUSH, kHead = 20, kHeads = (kBlocks * kHead + 63) / 64;  // scale blocks a unit, 16 dwords of scales and 4 of zeros each
    static constexpr int kStage = 4096 + kHeads * 256, kLoads = 4 + kHeads;
    const uint8_t* qw;
    const uint8_t* stage;
    const uint8_t* cur;
    uint32_t stage_lds, off[4];  // off: of the lane's 16 bytes in the rows 8 j .. 8 j + 7 of a unit
    int n, lane_, zshift;
    float per_group;  // 32 / group
    const uint8_t* head[kHeads];
    uint32_t head_stride[kHeads];
    int head_block[kHeads];  // its first column of a unit, in 32s
    uint32_t words[2][2];    // of a block of 32 columns
    uint32_t top0 = code_top(0x64006400u), top1 = code_top(0x54005400u);
    uint32_t s_raw[kBlocks], z_raw[kBlocks];

    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* at) {
        qw = t.w;
        stage = at;
        stage_lds = lds_address(at);
        n = t.n;
        lane_ = lane;
        zshift = 4 * (lane & 7);
        per_group = 32.0f / (float)t.group;
        // LDS row p holds word row 4 blk + 2 g + a with p = 4 blk + 2 a + g: the two half wavefronts read other banks
        const int p = lane >> 3, row = (p & 4) + 2 * (p & 1) + ((p >> 1) & 1);
#pragma unroll
        for (int j = 0; j < 4; j++) off[j] = (uint32_t)(row + 8 * j) * (uint32_t)n * 4u + (uint32_t)min(n0 + 4 * (lane & 7), n - 4) * 4u;
#pragma unroll
        for (int j = 0; j < kHeads; j++) {
            const int i = j * 64 + lane, blk = min(i / kHead, kBlocks - 1), part = i % kHead;
            head_block[j] = blk * (FLUSH / 2);
            head[j] = part < 16 ? (const uint8_t*)t.scales + min(n0 + 2 * part, n - 2) * 2 : (const uint8_t*)t.qzeros + min((n0 >> 3) + part - 16, (n >> 3) - 1) * 4;
            head_stride[j] = part < 16 ? (uint32_t)n * 2u : (uint32_t)(n >> 3) * 4u;
        }
    }
    template <int J>
    __device__ __forceinline__ void issue(int unit, int buf) {
        const uint32_t to = stage_lds + buf * kStage;
        if constexpr (J < 4) {
            load16_to_lds(off[J], qw + (int64_t)(32 * unit) * n * 4, to + J * 1024);
        } else {
            // (a group is a whole number of 32s and K below 2^27: half of one keeps the product off the integers by more than its rounding)
            const int group = (int)(((float)(8 * unit + head_block[J - 4]) + 0.5f) * per_group);
            load4_to_lds(head[J - 4] + (uint64_t)(uint32_t)group * head_stride[J - 4], to + 4096 + (J - 4) * 256);
        }
    }
    __device__ __forceinline__ void read_words(int blk) {
#pragma unroll
        for (int a = 0; a < 2; a++) words[blk & 1][a] = *(const uint32_t*)(cur + (4 * blk + 2 * a) * 128 + lane_ * 4);
    }
    __device__ __forceinline__ void open(int, int buf) {
        cur = stage + buf * kStage;
        read_words(0);
#pragma unroll
        for (int i = 0; i < kBlocks; i++) {
            s_raw[i] = *(const uint16_t*)(cur + 4096 + i * 80 + 2 * (lane_ & 31));
            z_raw[i] = *(const uint32_t*)(cur + 4096 + i * 80 + 64 + 4 * ((lane_ & 31) >> 3));
        }
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr ((T & 1) == 0 && T < 14) read_words((T >> 1) + 1);
    }
    template <int T>
    __device__ __forceinline__ void step(int, half8 (&b)[1]) const {
        const uint32_t z = ((z_raw[T / FLUSH] >> zshift) & 0xFu) + 1u;
        const uint32_t m0 = 0xE400E400u | (z * 0x00010001u), m1 = 0xD400D400u | (z * 0x00100010u);
        const uint32_t x = words[(T >> 1) & 1][T & 1], y = x >> 8;
        b[0] = pack4(pk_add((x & 0x000F000Fu) | top0, m0), pk_add((x & 0x00F000F0u) | top1, m1), pk_add((y & 0x000F000Fu) | top0, m0), pk_add((y & 0x00F000F0u) | top1, m1));
    }
    template <int I>
    __device__ __forceinline__ float scale_at() const { return h2f((uint16_t)s_raw[I]); }
};

// Q6_K in a tensor that begins at a multiple of four: blocks of 210 bytes lie at even addresses, loads to LDS want multiples of four: a row's 212 bytes from the last such address on, 208 of them in pieces
// of 16, the last four apart.  The fields begin `skew` (0 or 2) bytes later, other in every row and unit.  With an even number of blocks the last one of the matrix
// begins at 2 mod 4 and ends with those four bytes; an odd number of them, whose last would be read two bytes beyond its end, is not this kernel's (staged_plan).
template <int FLUSH>
struct StagedQ6 : Q6Weights<1, FLUSH> {
    using Base = Q6Weights<1, FLUSH>;
    static constexpr int kPieces = 13, kTotal = 32 * kPieces, kWide = (kTotal + 63) / 64, kLoads = kWide + 1, kTail = kTotal * 16, kStage = kTail + 128;
    const uint8_t* w;
    const uint8_t* stage;
    const uint8_t* cur;
    uint32_t stage_lds, off[kWide], off_tail;
    const uint8_t* tail;
    uint32_t odd, skew, mine_odd;  // odd: bit 1 + j: the row of piece j begins at 2 mod 4 in even units; mine_odd: the lane's own row, bit 1
    __device__ __forceinline__ void init(const WeightTensors& t, int n0, int lane, uint8_t* at) {
        this->g = lane >> 5;
        this->lane_ = lane;
        w = t.w;
        stage = at;
        stage_lds = lds_address(at);
        const uint32_t row_bytes = (uint32_t)(t.k / 256 * Q6_K_BPB);
        auto row_at = [&](int row) __attribute__((always_inline)) { return (uint32_t)min(n0 + row, t.n - 1) * row_bytes; };
        odd = 0;
#pragma unroll
        for (int j = 0; j < kWide; j++) {
            const int i = min(j * 64 + lane, kTotal - 1), row = i / kPieces;
            off[j] = row_at(row) + 16 * (i - row * kPieces);
            odd |= (row_at(row) & 2u) << j;
        }
        off_tail = row_at(lane & 31) + 208;
        mine_odd = row_at(lane & 31) & 2u;
    }
    template <int J>
    __device__ __forceinline__ void issue(int unit, int buf) {
        const uint8_t* b = w + (int64_t)unit * Q6_K_BPB;
        const uint32_t o = (unit & 1) ? ~odd : odd, to = stage_lds + buf * kStage;
        if constexpr (J < kWide) {
            if (J * 64 + 63 < kTotal || J * 64 + this->lane_ < kTotal) load16_to_lds(off[J] + 2 - ((o >> J) & 2u), b - 2, to + J * 1024);
        } else if (this->lane_ < 32) {
            load4_to_lds(b - 2 + (off_tail + 2 - ((mine_odd ^ (unit << 1)) & 2u)), to + kTail);
        }
    }
    // 16 bytes at offset `at` of the block
    __device__ __forceinline__ gd_u4 field(int at) const {
        const gd_u4 v = *(const gd_u4*)(cur + at);
        const uint32_t e = *(const uint32_t*)(at == 192 ? tail : cur + at + 16);
        return gd_u4{__builtin_amdgcn_alignbyte(v.y, v.x, skew), __builtin_amdgcn_alignbyte(v.z, v.y, skew), __builtin_amdgcn_alignbyte(v.w, v.z, skew),
                     __builtin_amdgcn_alignbyte(e, v.w, skew)};
    }
    __device__ __forceinline__ void read_half(int h) {
        this->ql[0][0] = field(64 * h + 16 * this->g);
        this->ql[0][1] = field(64 * h + 32 + 16 * this->g);
        this->qh[0] = field(128 + 32 * h + 16 * this->g);
    }
    __device__ __forceinline__ void open(int unit, int buf) {
        const uint8_t* b = stage + buf * kStage;
        cur = b + (this->lane_ & 31) * 208;
        tail = b + kTail + 4 * (this->lane_ & 31);
        skew = (mine_odd ^ (unit << 1)) & 2u;
        read_half(0);
        const gd_u4 s = field(192);
        const uint32_t sel = this->g ? 0x07050301u : 0x06040200u;
        this->sc[0][0] = __builtin_amdgcn_perm(s.y, s.x, sel);
        this->sc[0][1] = __builtin_amdgcn_perm(s.w, s.z, sel);
        this->d[0] = (*(const uint32_t*)tail >> (8 * skew)) & 0xffffu;
    }
    template <int T>
    __device__ __forceinline__ void before_step() {
        if constexpr (T == 7) read_half(1);
    }
};

template <int ENC, int FLUSH, bool CENTER>
using StagedOf = std::conditional_t<ENC == QMM_GPTQ, StagedGptq<FLUSH>, std::conditional_t<ENC == QMM_Q6_K, StagedQ6<FLUSH>, StagedK<ENC == QMM_Q5_K ? QMM_Q5_K : QMM_Q4_K, CENTER>>>;

// A tile's results from LDS to memory, whole rows of COLS columns (one row of 64 or two of 32 an instruction), eight instructions at
// a time.  Left in the order the matrix cores leave them in, with a choice of the kind of result at each value, the stores of 64 x 64 values took a
// wavefront 6 us (a branch and a wait at each); this way 2.4.
constexpr int result_row(int cols) { return cols + 8; }  // floats: the rows of the two half wavefronts (r and r + 4) lie in other banks
// fragment (a, f) of a wavefront's tile; column of lane i: f_cols f + lane_cols i
template <int ROW, int F_COLS, int LANE_COLS>
__device__ __forceinline__ void result_to_lds(float* tile, const float16v& t, int a, int f, int lane) {
    float* const p = tile + 4 * (lane >> 5) * ROW + LANE_COLS * (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; r++) p[(32 * a + 8 * (r >> 2) + (r & 3)) * ROW + F_COLS * f] = t[r];
}
// tile: the first of PARTS copies, `apart` floats from each other, added in order; inv: the inverse row scales; rows of the tile that are there: `rows`, at most
// ROWS; this wavefront is number `me` of WORKERS; (m0, n0): the tile's place
template <int ROWS, int COLS, int PARTS, int WORKERS>
__device__ __forceinline__ void store_results(const float* tile, int apart, const float* inv, int rows, int me, int lane, int m0, int n0, int n, bool add,
                                              uint16_t* __restrict__ out16, float* __restrict__ out) {
    constexpr int kRow = result_row(COLS), kEach = 64 / COLS, kTurns = std::min(8, ROWS / (kEach * WORKERS));
    static_assert(kTurns >= 1 && ROWS % (kTurns * kEach) == 0, "no turn reaches beyond the tile");
    const int col = n0 + (lane & (COLS - 1)), first = lane / COLS;
    if (col >= n) return;
    const float* const mine = tile + (lane & (COLS - 1));
    auto each = [&](auto&& store) __attribute__((always_inline)) {
        for (int r0 = me * (kTurns * kEach) + first; r0 < rows; r0 += WORKERS * (kTurns * kEach)) {
            float x[kTurns];
#pragma unroll
            for (int j = 0; j < kTurns; j++) {
                const int row = r0 + j * kEach;
                x[j] = mine[row * kRow];
#pragma unroll
                for (int q = 1; q < PARTS; q++) x[j] += mine[q * apart + row * kRow];
                x[j] *= inv[row];
            }
            int64_t at = (int64_t)(m0 + r0) * n + col;
#pragma unroll
            for (int j = 0; j < kTurns; j++, at += (int64_t)kEach * n)
                if (r0 + j * kEach < rows) store(at, x[j]);
        }
    };
    if (add) each([&](int64_t at, float x) __attribute__((always_inline)) { unsafeAtomicAdd(out + at, x); });
    else if (out16) each([&](int64_t at, float x) __attribute__((always_inline)) { out16[at] = f2bf(x); });
    else each([&](int64_t at, float x) __attribute__((always_inline)) { out[at] = x; });
}

// LDS: two (where that leaves room, three) chunks of the lhs for each part of K, two units of the weights and of the sums of the lhs.
template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER>
struct StagedLds {
    using W = StagedOf<ENC, FLUSH, CENTER>;
    static constexpr int kPer = HILO ? 2 : 1, kInvBytes = 64 * ((FM + 1) / 2) * 4, kResults = WN * WK * 64 * result_row(32) * 4;
    static constexpr int kWeights = 2 * WN * WK * W::kStage, kSums = W::kMin ? WK * 2 * FM * 1024 : 0;
    static constexpr int lhs(int steps, int bufs) { return WK * bufs * FM * steps * kPer * 1024; }
    static constexpr bool fits(int steps, int bufs) { return lhs(steps, bufs) + kWeights + kSums + kInvBytes <= kLdsPerCu; }
    static constexpr int kSteps = fits(8 / kPer, 2) ? 8 / kPer : fits(4 / kPer, 2) ? 4 / kPer : fits(2 / kPer, 2) ? 2 / kPer : 0;
    static_assert(kSteps >= 1, "fits a compute unit");
    static constexpr int kBufs = kSteps == 8 / kPer ? 2 : fits(kSteps, 3) ? 3 : 2;
    static constexpr int kBuf = FM * kSteps * kPer * 1024;
    static constexpr int kW = lhs(kSteps, kBufs), kS = kW + kWeights, kInv = std::max(kS + kSums, kResults), kBytes = kInv + kInvBytes;
};

// The grid: 8 x `full` row tiles x (shares of column sections), `sections` of the latter; then the last row tile, if it has up to 32 rows and is not the only one, which is not among the full ones.
struct StagedGrid {
    int full, sections, shares;
};

// How many of n loads, spread over the steps before `end` (0: asked for before the first one), are asked for before step t.
constexpr int spread_before(int n, int end, int t) { return t < 0 ? 0 : t >= end ? n : (t * n + end - 1) / end; }

// What arrives in scalar registers with a workgroup (the rest of the arguments is asked for when it runs).
struct StagedStart {
    const void *a16, *sums;
    int m, units, count;  // count: of the matrices
};

// wt: of the first matrix; row0: the first 32 rows of the tile, in 32s; place: which share of which column section
template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER, bool FOLD>
__device__ __forceinline__ void staged_tile(WeightTensors wt, const StagedStart& start, const DirectMats& mats, const DirectSpace& p, uint16_t* __restrict__ out16, int shares, int row0, int place) {
    const int m = start.m, units = start.units;
    using W = StagedOf<ENC, FLUSH, CENTER>;
    using L = StagedLds<ENC, FLUSH, FM, WN, WK, HILO, CENTER>;
    // a chunk of the lhs: kCS steps, kPieces operands of 1 KB (fp32 rows: hi and residual) for each row tile
    constexpr int kPer = L::kPer, kCS = L::kSteps, kBufs = L::kBufs, kPieces = kCS * kPer, kChunks = W::kSteps / kCS, kBuf = L::kBuf;
    constexpr int kTotal = FM * kPieces, kLoads = (kTotal + WN - 1) / WN, kSums = W::kMin ? (FM + WN - 1) / WN : 0;
    constexpr int kWeightLoads = W::kLoads + kSums;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];  // [WK][kBufs][kBuf] lhs, [WN WK][2] packed weights, [WK][2][FM] sums, inverse row scales
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wn = wave % WN, wk = wave / WN;
    float* const inv = (float*)(smem + L::kInv);
    const int share = place & (shares - 1);
    int section = place >> (shares - 1), first = 0;
    float* __restrict__ out = mats.out[0];
    if (start.count > 1) {
#pragma unroll
        for (int j = 1; j < kDirectMaxMats; j++)
            if (j < start.count && section >= mats.end[j - 1]) wt.w = mats.w[j], wt.n = mats.n[j], out = mats.out[j], first = mats.end[j - 1];
    }
    const int tile_n = (section - first) * 8 + (int)blockIdx.x;
    if (tile_n * 32 * WN >= wt.n) return;
    const int n0 = tile_n * 32 * WN + 32 * wn, m0 = row0 * 32;
    // this wavefront's units of K; the workgroup's barriers are those of its longest part
    constexpr int kLogWk = WK == 4 ? 2 : WK == 2 ? 1 : 0;
    const int log_parts = kLogWk + shares - 1, part = share * WK + wk, walk = (units + (1 << log_parts) - 1) >> log_parts;
    const int u0 = (units * part) >> log_parts, u1 = (units * (part + 1)) >> log_parts;

    // (the offsets of a unit first join its products, as in the direct and shared kernels: with two additions to T a unit instead of one, Q4_K with fp32 rows was
    // off by 2.30e-7 instead of 2.04e-7 after sums of 40 units, Q5_K with bf16 rows by 1.06e-7 instead of 0.99e-7; for codes from 0 the error is that of larger
    // terms.  Never a question of FM: matrices that share a launch share its tile, and keep the bits that calls of their own give.)
    constexpr bool kUnit = unit_sums(ENC, FLUSH, HILO) || (W::kMin && (HILO || CENTER));
    // FOLD: sums over kStagedFold units are added up in others, so that a workgroup that walks all of K is as exact as wavefronts with a part of it each (K = 4096, bf16 rows: 1.03e-7
    // relative error, folded 0.68e-7, as the direct kernel with four parts).  A fold takes two instructions a value, 1 .. 5 % of a call.
    float16v T[FM], P[FM], M, U[kUnit ? FM : 1], S[FOLD ? FM : 1];
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            T[a][r] = 0.0f, P[a][r] = 0.0f;
            if constexpr (kUnit) U[a][r] = 0.0f;
            if constexpr (FOLD) S[a][r] = 0.0f;
        }
    const float16v zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const uint32_t l16 = lane * 16;
    const uint32_t lds0 = lds_address(smem);
    W w;
    w.init(wt, n0, lane, smem + L::kW + wave * 2 * W::kStage);
    const int64_t row_bytes = (int64_t)units * W::kSteps * 1024 * kPer;
    const int last_tile = (m - 1) >> 5;
    // a wavefront loads kLoads neighbouring operands of a chunk (the last ones some that its neighbour loads too); of one row tile, unless kLoads does not divide what a tile has
    constexpr bool kOneTile = kPieces % kLoads == 0 && kTotal % kLoads == 0;
    static_assert(kOneTile || FM == 3, "the plans with 64 rows a tile take rows of any length (kStagedLongRows)");
    const int piece0 = min(wn * kLoads, kTotal - kLoads);
    auto tile_of = [&](int piece) __attribute__((always_inline)) { return min(row0 + piece / kPieces, last_tile); };
    const uint8_t* const src = (const uint8_t*)start.a16 + tile_of(piece0) * row_bytes + ((int64_t)u0 * W::kSteps * kPer + piece0 % kPieces) * 1024;
    uint32_t from[kOneTile ? 1 : kLoads];
    from[0] = l16;
    if constexpr (!kOneTile) {
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            from[j] = l16 + load_run_offset(j) + (uint32_t)max<int64_t>((tile_of(piece0 + j) - tile_of(piece0)) * row_bytes + 1024 * ((piece0 + j) % kPieces - piece0 % kPieces), 0);  // (0: of no row)
    }
    const int last_chunk = (u1 - u0) * kChunks - 1;
    auto issue_lhs = [&](int chunk, int buf) __attribute__((always_inline)) {
        load_run_to_lds<kLoads>(from, src + (int64_t)min(chunk, last_chunk) * (kPieces * 1024), lds0 + (wk * kBufs + buf) * kBuf + piece0 * 1024);
    };
    // bf16 rows: loads are asked for a few at a time; at many at once, 16 cycles of a compute unit's load path for each, the wavefronts stand still.  The chunk that a boundary makes room for in two
    // halves, the second one a step later; the weights and sums of the next unit over the first steps of this one, early enough to be older than the chunk that the last boundary waits for.
    // us, all at once / this way: GPTQ 14336 x 4096 400 rows 59.0 / 57.5, Q6_K 8192 x 8192 500 rows 128.8 / 126.3, Q4_K 4096 x 14336 2048 rows 261.7 / 257.8, 4096 x 4096 64 rows 13.2 / 12.5; but fp32 rows, which
    // have twice the matrix-core instructions to hide loads behind, GPTQ 14336 x 4096 500 rows 116.6 / 119.2, and groups of 32 8192 x 8192 300 bf16 rows 93.2 / 95.0.
    constexpr bool kFew = !HILO && !(ENC == QMM_GPTQ && FLUSH == 2), kTwice = kFew && kCS >= 4 && kLoads % 2 == 0 && kOneTile;
    constexpr int kSpread = kFew ? std::min(10, 15 - kCS * (kBufs - 1)) : 0;
    auto issue_half = [&](int half, int chunk, int buf) __attribute__((always_inline)) {
        constexpr int kHalf = kLoads / 2;
        load_run_to_lds<kHalf>(from, src + (int64_t)min(chunk, last_chunk) * (kPieces * 1024) + half * (kHalf * 1024), lds0 + (wk * kBufs + buf) * kBuf + (piece0 + half * kHalf) * 1024);
    };
    auto issue_weights = [&](auto first, auto end, int unit, int buf) __attribute__((always_inline)) {  // loads first .. end - 1 of a unit
        constexpr int kFirst = decltype(first)::value, kEnd = decltype(end)::value;
        unrolled<kEnd - kFirst>([&](auto i) __attribute__((always_inline)) {
            constexpr int j = kFirst + decltype(i)::value;
            if constexpr (j < W::kLoads) {
                w.template issue<j>(unit, buf);
            } else {
                const int a = (wn + WN * (j - W::kLoads)) % FM;
                load16_to_lds(l16, (const uint8_t*)start.sums + ((int64_t)min(row0 + a, last_tile) * units + unit) * 1024,
                              (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + L::kS + ((wk * 2 + buf) * FM + a) * 1024)));
            }
        });
    };
    half8 af[2][FM][kPer];
    uint32_t at = 0;  // where the lane's operands of the current chunk are
    auto read_lhs = [&](int step, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < FM; a++)
#pragma unroll
            for (int q = 0; q < kPer; q++) af[slot][a][q] = *(const half8*)(smem + at + ((a * kCS + step) * kPer + q) * 1024);
    };
    auto buffer = [&](int buf) __attribute__((always_inline)) { at = (uint32_t)((wk * kBufs + buf) * kBuf) + l16; };
    half8 b[2][W::kPlanes];
    float d = 0.0f;
    if (u0 < u1) {
        issue_weights(std::integral_constant<int, 0>{}, std::integral_constant<int, kWeightLoads>{}, u0, 0);
#pragma unroll
        for (int c = 0; c < kBufs; c++) issue_lhs(c, c);
    }
    if (threadIdx.x < 32 * FM) inv[threadIdx.x] = p.inv[min(m0 + (int)threadIdx.x, m - 1)];
    wait_vmcnt<(kBufs - 1) * kLoads>();
    __syncthreads();
    if (u0 < u1) {
        w.open(u0, 0);
        buffer(0);
        read_lhs(0, 0);
        w.template step<0>(0, b[0]);
    }
    int buf = 0, free_buf = 0;  // of the current chunk, of the one before
    for (int it = 0; it < walk; it++) {
        const int u = u0 + it;
        if (u >= u1) {
#pragma unroll
            for (int c = 0; c < kChunks; c++) __syncthreads();
            continue;
        }
        const int next = min(u + 1, u1 - 1);
        if constexpr (kSpread == 0) issue_weights(std::integral_constant<int, 0>{}, std::integral_constant<int, kWeightLoads>{}, next, (it + 1) & 1);
        float dmin = w.min_scale(0), dnext = 0.0f;  // (CENTER: the power of two that the offsets are in units of, made in the first five steps)
        if constexpr (ENC != QMM_GPTQ) dnext = w.scale(0);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<W::kSteps>([&](auto tt) __attribute__((always_inline)) {
            constexpr int t = decltype(tt)::value, chunk = t / kCS, cur = t & 1;
            if constexpr ((t + 1) % kCS == 0) {
                // Lhs chunk c + 1 has arrived (asked for kBufs - 1 boundaries ago, its second half a step later), at the last boundary of a unit also the weights of the next one, and
                // every wavefront has read chunk c: its buffer takes chunk c + kBufs.  Younger than what is waited for: the chunks asked for since, and the weights of the steps since.
                constexpr int kSince = t - kCS * (kBufs - 1) + (kTwice ? 1 : 0);
                static_assert(t + 1 < W::kSteps || kSince >= kSpread, "at the last boundary the weights are older than the chunk that is waited for");
                static_assert(kSince >= 0 || 16 + kSince >= kSpread, "none of the unit before are younger");
                wait_vmcnt<(kBufs - 2) * kLoads + spread_before(kWeightLoads, kSpread, t) - spread_before(kWeightLoads, kSpread, kSince)>();
                __syncthreads();
                if constexpr (kTwice) issue_half(0, it * kChunks + chunk + kBufs, buf);
                else issue_lhs(it * kChunks + chunk + kBufs, buf);
                free_buf = buf;
                buf = buf == kBufs - 1 ? 0 : buf + 1;
                buffer(buf);
            }
            if constexpr (kTwice && t % kCS == 0) {
                if (t > 0 || it > 0) issue_half(1, it * kChunks + t / kCS - 1 + kBufs, free_buf);
            }
            read_lhs((t + 1) % kCS, cur ^ 1);
            if constexpr (t + 1 == W::kSteps) w.open(u + 1 < u1 ? u + 1 : u, (it + 1) & 1);
            w.template before_step<t>();
            // one row tile every three steps, the last at steps 14 and 15
            constexpr int min_a = (t - 14 + 3 * (FM - 1)) / 3, min_at = 14 - 3 * (FM - 1);
            constexpr bool min_now = W::kMin && t >= min_at && (t - min_at) % 3 == 0, min_add = W::kMin && t > min_at && (t - min_at) % 3 == 1;
            half8 sf;
            if constexpr (min_now) sf = *(const half8*)(smem + L::kS + ((wk * 2 + (it & 1)) * FM + min_a) * 1024 + l16);
            if constexpr (CENTER && t < 5) {
                if constexpr (t == 0) dmin = w.open_offsets();
                else w.template add_offsets<t - 1>();
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (t % W::kFlush == 0) {
#pragma unroll
                for (int a = 0; a < FM; a++) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        if constexpr (!kUnit) T[a][r] = fmaf(d, P[a][r], T[a][r]);
                        else if constexpr (t == 0) T[a][r] += fmaf(d, P[a][r], U[a][r]);
                        else U[a][r] = t == W::kFlush ? d * P[a][r] : fmaf(d, P[a][r], U[a][r]);
                    }
                    if constexpr (!kUnit || t == 0) asm volatile("" : "+v"(T[a]));
                    else asm volatile("" : "+v"(U[a]));
                    if constexpr (FOLD && t == 0) {
                        if (it > 0 && it % kStagedFold == 0) {
#pragma unroll
                            for (int r = 0; r < 16; r++) S[a][r] += T[a][r], T[a][r] = 0.0f;
                        }
                    }
#pragma unroll
                    for (int pl = 0; pl < W::kPlanes; pl++)
#pragma unroll
                        for (int q = 0; q < kPer; q++) P[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[cur][a][q], b[cur][pl], q || pl ? P[a] : zero16, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (ENC == QMM_GPTQ) d = w.template scale_at<t / W::kFlush>();
                else d = dnext;
            } else {
#pragma unroll
                for (int pl = 0; pl < W::kPlanes; pl++)
#pragma unroll
                    for (int q = 0; q < kPer; q++)
#pragma unroll
                        for (int a = 0; a < FM; a++) P[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[cur][a][q], b[cur][pl], P[a], 0, 0, 0);
            }
            if constexpr (min_now) {
                if constexpr (CENTER) {
                    M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf, w.offsets_lo(), zero16, 0, 0, 0);
                    M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf, w.offsets_hi(), M, 0, 0, 0);
                } else {
                    M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf, w.min_operand(0), zero16, 0, 0, 0);
                }
            }
            if constexpr (min_add) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    if constexpr (kUnit) U[min_a][r] = dmin * M[r];
                    else T[min_a][r] = fmaf(dmin, M[r], T[min_a][r]);
                }
            }
            issue_weights(std::integral_constant<int, spread_before(kWeightLoads, kSpread, t)>{}, std::integral_constant<int, spread_before(kWeightLoads, kSpread, t + 1)>{}, next, (it + 1) & 1);
            w.template step<(t + 1) % W::kSteps>(0, b[cur ^ 1]);
            if constexpr (t % W::kFlush != 0) {
                constexpr int kMfma = FM * kPer * W::kPlanes, kValu = (W::kPlanes == 2 ? 28 : W::kMin ? 12 : 14) + (min_add ? 16 : 0);  // spread evenly
                unrolled<kMfma + (min_now ? (CENTER ? 2 : 1) : 0)>([&](auto) __attribute__((always_inline)) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, (kValu + kMfma - 1) / kMfma, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            T[a][r] = kUnit ? T[a][r] + fmaf(d, P[a][r], U[a][r]) : fmaf(d, P[a][r], T[a][r]);
            if constexpr (FOLD) T[a][r] += S[a][r];
        }
    wait_vmcnt<0>();
    __syncthreads();  // nothing is on its way into the buffers any more, which now take the results
    constexpr int kTile = 64 * result_row(32);
    float* const mine = (float*)smem + wave * kTile;
#pragma unroll
    for (int a0 = 0; a0 < FM; a0 += 2) {  // (64 rows at a time)
        if (a0) __syncthreads();
#pragma unroll
        for (int a = a0; a < FM && a < a0 + 2; a++) result_to_lds<result_row(32), 32, 1>(mine, T[a], a - a0, 0, lane);
        __syncthreads();
        store_results<64, 32, WK, WK>((const float*)smem + wn * kTile, WN * kTile, inv + 32 * a0, min(32 * std::min(2, FM - a0), m - m0 - 32 * a0), wk, lane, m0 + 32 * a0, n0, wt.n, shares > 1, out16, out);
    }
}

// A last row tile of up to 32 rows takes 0.6 .. 0.7 of a full one's time when it is not treated as one; such tiles come last in the grid and fill the last round.  us, before / with it: act-order GPTQ
// 14336 x 4096 400 bf16 rows (4 x 56 tiles of 96 rows and 56 of 16 on 256 compute units) 95 / 86, Q4_K 4096 x 14336 400 rows 80 / 73, 14336 x 4096 400 fp32 rows 129 / 105, Q5_K 11008 x 4096 260
// rows 51 / 48, Q6_K 8192 x 8192 400 rows 127 / 114.  Over 1280 problems of 70 .. 1000 rows 0.976 of the time (geometric mean), none more than 4 % slower.
template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER, bool FOLD>
__global__ __launch_bounds__(64 * WN * WK, 2) void gemm_staged_kernel(const uint8_t* w0, const void* a16, const void* sums, int rows0, int m, int units, int full, int sections, int shares, int count,
                                                                 WeightTensors wt, DirectMats mats, DirectSpace p, uint16_t* __restrict__ out16) {
    // (the first arguments arrive in scalar registers with the workgroup)
    const StagedGrid grid{full, sections, shares};
    const StagedStart start{a16, sums, m, units, count};
    wt.w = w0, wt.n = rows0, wt.k = units * 256;
    // (the shape of the grid spares the divisions)
    int row_tile = (int)blockIdx.y, place = (int)blockIdx.z;
    if (place < grid.sections) {
        // The last row tile without 32 rows that it has not: 200 rows as 128 + 96.  The same rounds of workgroups, but products of rows that nobody asked for heat the part as others do, and its clock is what
        // the power leaves (1.7 GHz here): 14336 x 4096 200 bf16 rows 43.9 -> 41.0 us.
        if constexpr (FM > 2)
            if (row_tile == grid.full - 1 && m <= (grid.full * FM - 1) * 32) return staged_tile<ENC, FLUSH, FM - 1, WN, WK, HILO, CENTER, FOLD>(wt, start, mats, p, out16, grid.shares, row_tile * FM, place);
        staged_tile<ENC, FLUSH, FM, WN, WK, HILO, CENTER, FOLD>(wt, start, mats, p, out16, grid.shares, row_tile * FM, place);
    } else {
        place = (place - grid.sections) * grid.full + row_tile;
        if (place < grid.sections) staged_tile<ENC, FLUSH, 1, WN, WK, HILO, CENTER, FOLD>(wt, start, mats, p, out16, grid.shares, grid.full * FM, place);
    }
}

template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER, bool FOLD = false>
hipError_t run_staged(const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units, int shares, hipStream_t s) {
    using L = StagedLds<ENC, FLUSH, FM, WN, WK, HILO, CENTER>;
    static_assert(L::kBytes <= kLdsPerCu, "fits a compute unit");
    using L1 = StagedLds<ENC, FLUSH, 1, WN, WK, HILO, CENTER>;
    using LR = StagedLds<ENC, FLUSH, FM - 1, WN, WK, HILO, CENTER>;  // (of the last row tile)
    constexpr int lds = std::max(std::max(L::kBytes, L1::kBytes), LR::kBytes);
    int eights = 0;
    for (int j = 0; j < mats.count; j++) mats.end[j] = eights += (mats.n[j] + 256 * WN - 1) / (256 * WN);
    hipError_t e = allow_full_lds<gemm_staged_kernel<ENC, FLUSH, FM, WN, WK, HILO, CENTER, FOLD>>();
    if (e != hipSuccess) return e;
    const bool short_last = staged_short_last(FM, m, (int64_t)eights * shares);
    const int full = (int)(short_last ? m / (32 * FM) : (m + 32 * FM - 1) / (32 * FM)), sections = eights * shares, more = short_last ? (sections + full - 1) / full : 0;
    gemm_staged_kernel<ENC, FLUSH, FM, WN, WK, HILO, CENTER, FOLD><<<dim3(8, (unsigned)full, (unsigned)(sections + more)), dim3(64 * WN * WK), lds, s>>>(
        mats.w[0], p.a16, p.sums, mats.n[0], (int)m, units, full, sections, shares, mats.count, wt, mats, p, out16);
    return hipGetLastError();
}

template <int ENC, int FLUSH, bool HILO, bool CENTER = false>
hipError_t run_staged_plan(const DirectPlan& pl, const WeightTensors& wt, const DirectMats& mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units, hipStream_t s) {
#define QMM_GS(FM, WN, WK)                       \
    if constexpr (staged_folds(ENC, FLUSH, FM, HILO)) \
        if (pl.fold && pl.fm == FM && pl.wn == WN && pl.wk == WK) return run_staged<ENC, FLUSH, FM, WN, WK, HILO, CENTER, true>(wt, mats, p, out16, m, units, pl.shares, s); \
    if constexpr (staged_built(ENC, FLUSH, FM, HILO, CENTER)) \
        if (pl.fm == FM && pl.wn == WN && pl.wk == WK) return run_staged<ENC, FLUSH, FM, WN, WK, HILO, CENTER>(wt, mats, p, out16, m, units, pl.shares, s)
    QMM_GS(2, 2, 4);
    QMM_GS(2, 4, 2);
    QMM_GS(2, 8, 1);
    QMM_GS(3, 4, 2);
    QMM_GS(3, 8, 1);
    QMM_GS(4, 4, 2);
    QMM_GS(4, 8, 1);
#undef QMM_GS
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm_staged(int encoding, bool hilo, const DirectPlan& pl, const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16,
                              int64_t m, int units, hipStream_t s) {
#define QMM_GS_RUN(...) return run_staged_plan<__VA_ARGS__>(pl, wt, mats, p, out16, m, units, s)
    switch (encoding) {
        case QMM_Q4_K:
            if (hilo) QMM_GS_RUN(QMM_Q4_K, 16, true, true);
            if (pl.centred) QMM_GS_RUN(QMM_Q4_K, 16, false, true);
            QMM_GS_RUN(QMM_Q4_K, 16, false);
        case QMM_Q5_K:
            if (hilo) QMM_GS_RUN(QMM_Q5_K, 16, true, true);
            if (pl.centred) QMM_GS_RUN(QMM_Q5_K, 16, false, true);
            QMM_GS_RUN(QMM_Q5_K, 16, false);
        case QMM_Q6_K:
            if (hilo) QMM_GS_RUN(QMM_Q6_K, 16, true);
            QMM_GS_RUN(QMM_Q6_K, 16, false);
        case QMM_GPTQ:
            if (wt.group % 128 == 0) {
                if (hilo) QMM_GS_RUN(QMM_GPTQ, 8, true);
                QMM_GS_RUN(QMM_GPTQ, 8, false);
            }
            if (hilo) QMM_GS_RUN(QMM_GPTQ, 2, true);
            QMM_GS_RUN(QMM_GPTQ, 2, false);
        default: return hipErrorInvalidValue;
    }
#undef QMM_GS_RUN
}

}  // namespace qmm
