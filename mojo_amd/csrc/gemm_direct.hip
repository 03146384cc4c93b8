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
//   acc += d * sum(u * a16) [+ sum((mid * d * sc - dmin * mn) * s)],  u: integer weights (sc * (q - mid), or q - zero), a16: the row scaled by a power of
//   two and narrowed to fp16 (fp32 rows: hi + residual, both products into one accumulator), s: sub-block sums of the scaled row in fp32.
//   Q6_K: sc * q may need 13 bits, so sc = 16 hi + lo gives two integer operands per weight (see gemm_planes.hip).
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "gemm_direct.h"

namespace qmm {

namespace {

DirectSpace direct_space(void* ws, bool f32, bool with_sums, bool with_sums32, int64_t m, int64_t k) {
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t tiles = (m + 31) / 32;
    DirectSpace p;
    char* base = (char*)ws;
    int64_t off = 0;
    p.a16 = (_Float16*)base;
    off += tiles * ((k + 255) / 256) * 16384 * (f32 ? 2 : 1) + 32768;
    p.sums = (_Float16*)(base + off);
    off += with_sums ? tiles * ((k + 255) / 256) * 1024 : 0;
    p.sums32 = (float*)(base + off);
    off += with_sums32 ? tiles * ((k + 255) / 256) * 1024 : 0;
    p.inv = (float*)(base + off);
    off += up(tiles * 32 * 4);
    p.bytes = off;
    return p;
}

// ---------------------------------------------------------------------------------------------------------------------------
// preparation: one workgroup per lhs row (the first m workgroups), then zeroing of `out` for two workgroups per tile
// ---------------------------------------------------------------------------------------------------------------------------
// With few rows the latency of a row's passes (load, maximum, narrow, store) bounds it: as many threads as leave each one or two pieces of eight
// columns (200 x 14336 bf16 rows with 256 threads a row 10.1 us, with 1024 7.2), all of which are asked for before the first is looked at; with many, that a row writes 16 bytes of a
// 128-byte line, the rest of which other workgroups of the XCD fill.  us in a trace, the pieces widened to fp32 as they arrive (a wait after each) and compared as such / kept as they are:
// 500 x 14336 bf16 rows 13.8 / 11.7 (28 MB), 200 x 14336 7.6 / 7.1; of calls, Q4_K 4096 x 14336 200 rows 47.0 / 46.4, 4096 x 28672 40 fp32 rows 57.3 / 56.3, 512 x 2048 24 fp32 rows 9.7 / 8.6.
// Two workgroups of 1024 threads to a compute unit, 64 registers: with 66 one, GPTQ 696 x 7936 327 fp32 rows 33.9 / 34.9 us, Q4_K 616 x 6400 416 rows 33.65 / 34.15.
// Rows of one group of eight go to workgroups of one XCD (ids congruent mod 8): a 128-byte line of an operand holds eight rows.
// SORTED: column p of the operands is column source[p] of the row, which lies in LDS (k values) meanwhile.
template <typename AT, int ORDER, bool SORTED = false>
__global__ __launch_bounds__(1024, 8) void direct_prep_kernel(const AT* __restrict__ a, int m, int k, DirectSpace p, int with_sums, DirectMats zero,
                                                           const int32_t* __restrict__ source) {
    extern __shared__ __attribute__((aligned(16))) uint8_t row_lds[];
    __shared__ uint32_t wmax[16];
    const int tid = threadIdx.x, threads = (int)blockDim.x, rows = (m + 63) / 64 * 64;
    if ((int)blockIdx.x >= rows) {
        zero_out(zero, m, (int)blockIdx.x - rows, (int)gridDim.x - rows);
        return;
    }
    const int b = blockIdx.x, row = (b & ~63) + (b & 7) * 8 + ((b >> 3) & 7);
    if (row >= m) return;
    const AT* ar = a + (int64_t)row * k;
    const int pieces = k >> 3;  // of eight columns, one per thread and turn
    const int steps = (k + 255) / 256 * 16;
    constexpr int kHeld = 4;    // rows of up to 32768 columns (1024 threads) stay in registers between the search for the maximum and the narrowing
    LhsPiece<AT> held[kHeld];   // (as they came: a conversion after each load would wait for it before the next is asked for)
    const int turns = (pieces + threads - 1) / threads;
    if constexpr (SORTED) {
        constexpr int kPer = 16 / sizeof(AT);
        for (int i = tid * kPer; i < k; i += threads * kPer) *(gd_u4*)((AT*)row_lds + i) = *(const gd_u4*)(ar + i);
        __syncthreads();
    }
    auto load = [&](int pc) __attribute__((always_inline)) {
        if constexpr (SORTED) {
            const int4 s0 = *(const int4*)(source + 8 * pc), s1 = *(const int4*)(source + 8 * pc + 4);
            const int from[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
            LhsPiece<AT> x;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if constexpr (sizeof(AT) == 4) x.raw[i >> 2][i & 3] = ((const uint32_t*)row_lds)[from[i]];
                else if (i & 1) x.raw[0][i >> 1] |= (uint32_t)((const uint16_t*)row_lds)[from[i]] << 16;
                else x.raw[0][i >> 1] = ((const uint16_t*)row_lds)[from[i]];
            }
            return x;
        } else {
            return load_piece(ar + pc * 8);
        }
    };
    uint32_t top = 0;
    if (turns <= kHeld) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i < turns) held[i] = load(min(tid + i * threads, pieces - 1));
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i < turns) top = largest_bits(top, held[i]);
    } else {
        for (int pc = tid; pc < pieces; pc += threads) top = largest_bits(top, load(pc));
    }
    float mx = largest_of<AT>(top);
    if (any_not_finite(mx)) {
        mx = 0.0f;
        for (int pc = tid; pc < pieces; pc += threads) mx = largest_finite(mx, load(pc));
    }
    const uint32_t mb = wave_max_nonneg_bits(mx);
    if ((tid & 63) == 0) wmax[tid >> 6] = mb;
    __syncthreads();
    const uint32_t mxb = wave_max_nonneg_bits(__uint_as_float((tid & 63) < threads >> 6 ? wmax[tid & 63] : 0u));
    float inv;
    const float s = row_scale(mxb, with_sums ? kRowTopWithSums : kRowTop, inv);
    if (tid == 0) p.inv[row] = inv;
    const int tile = row >> 5, lane = row & 31;
    auto emit = [&](int pc, float (&v)[8]) __attribute__((always_inline)) {
        store_piece<AT, ORDER>(p.a16, steps, row, pc, s, v);
        if (with_sums) {
            const int blk = pc >> 2;
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i += 2) sum += v[i] + v[i + 1];
            sum += dpp_move<0xB1>(sum);
            sum += dpp_move<0x4E>(sum);  // the four threads of a 32-wide sub-block
            if ((pc & 3) == 0) {
                const float sh = h2f(f2h(sum));
                _Float16* sp = p.sums + ((int64_t)tile * (k >> 8) + (blk >> 3)) * 512 + lane * 8 + (blk & 7);
                sp[0] = (_Float16)sh;
                sp[256] = (_Float16)(sum - sh);
                p.sums32[((int64_t)tile * (k >> 8) + (blk >> 3)) * 256 + (lane + 32 * (blk & 1)) * 4 + ((blk & 7) >> 1)] = sum;
            }
        }
    };
    for (int pc = pieces + tid; pc < 2 * steps; pc += threads) {  // zeros up to a whole unit
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        emit(pc, v);
    }
    auto emit_piece = [&](int pc, const LhsPiece<AT>& x) __attribute__((always_inline)) {
        float v[8];
        unpack_piece(x, v);
        emit(pc, v);
    };
    if (turns <= kHeld) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + i * threads < pieces) emit_piece(tid + i * threads, held[i]);
    } else {
        for (int pc = tid; pc < pieces; pc += threads) emit_piece(pc, load(pc));
    }
}

// The same for Q4_0: rows quantised to Q8_0, codes as fp16, no row scale; the fp16 block scales of a row as the first eight slots of the
// unit's operand in `sums` (lanes g = 0; zeros in g = 1).  Four neighbouring threads hold a block.
template <typename AT>
__global__ __launch_bounds__(1024) void direct_prep_q8_kernel(const AT* __restrict__ a, int m, int k, DirectSpace p, DirectMats zero) {
    const int tid = threadIdx.x, threads = (int)blockDim.x, rows = (m + 63) / 64 * 64;
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
    for (int pc = tid; pc < units * 32; pc += threads) {
        const int blk = pc >> 2, sub = pc & 3, g = sub & 1, step = 2 * blk + (sub >> 1);
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (pc < pieces) unpack_piece(load_piece(ar + pc * 8), v);
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

int prep_threads(int64_t k) { return k <= 2048 ? 256 : k <= 4096 ? 512 : 1024; }
// For a sorted row, whose values come from LDS: as many turns, with as few threads as they need.  us, act-order calls, 512 or 1024 threads in every turn / branches around what a wavefront has no piece of, with
// a wait at each / this way: 1232 x 3712 2507 bf16 rows 95.6 / 92.6 / 91.5, 2208 x 2688 1940 rows 88.0 / 83.3 / 82.2, 888 x 4352 1610 fp32 rows 66.6 / 63.2 / 62.9.
int sorted_prep_threads(int64_t k) {
    const int64_t pieces = k / 8, turns = (pieces + prep_threads(k) - 1) / prep_threads(k);
    return (int)((pieces + turns * 64 - 1) / (turns * 64) * 64);
}

constexpr int direct_ahead(int enc, int fm, int fn, bool hilo, int flush) {
    if (fm * fn == 2) return hilo ? 4 : 8;
    // (one fragment of the K-quants with fp32 rows: 16 ahead takes 5 % longer)
    return hilo && (enc != QMM_GPTQ || flush == 2) ? 8 : 16;
}

template <typename W>
constexpr int direct_slot(int frags) { return W::kStage > frags * 4096 ? W::kStage : frags * 4096; }

}  // namespace

// shares: workgroups per tile (1, or 2 that add onto zeros).  (The first arguments arrive in scalar registers with the workgroup.)
template <int ENC, int FLUSH, int FM, int FN, int WK, bool HILO>
__global__ __launch_bounds__(64 * WK, 2) void gemm_direct_kernel(const uint8_t* w0, const void* a16, const float* inv_scales, int rows0, int m, int units, int tiles_m, int shares,
                                                                 int count, WeightTensors wt, DirectMats mats, DirectSpace p, uint16_t* __restrict__ out16) {
    using W = WeightsOf<ENC, FN, FLUSH, true>;
    constexpr int kSlot = direct_slot<W>(FM * FN);
    extern __shared__ __attribute__((aligned(16))) float red[];  // a slot per wavefront: its packed rows, at the end its results [FM * FN][4][64] float4
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const DirectPlace at = direct_place(tiles_m, shares);
    const int tile_m = at.tile_m, share = at.share;
    int section = at.section, first = 0;
    wt.w = w0, wt.n = rows0;
    if constexpr (ENC != QMM_GPTQ && ENC != QMM_Q4_0) wt.k = units * 256;
    float* __restrict__ out = mats.out[0];
    if (count > 1) {
#pragma unroll
        for (int j = 1; j < kDirectMaxMats; j++)
            if (j < count && section >= mats.end[j - 1]) wt.w = mats.w[j], wt.n = mats.n[j], out = mats.out[j], first = mats.end[j - 1];
    }
    const int tile_n = (section - first) * 8 + at.eighth;
    if (tile_n * 32 * FN >= wt.n) return;
    const int n0 = tile_n * 32 * FN, m0 = tile_m * 32 * FM;
    // this wavefront's units of K
    constexpr int kLogWk = WK == 8 ? 3 : 2;
    static_assert(WK == 1 << kLogWk, "parts of K");
    const int log_parts = kLogWk + shares - 1, part = share * WK + wave;
    const int u0 = (int)((unsigned)units * (unsigned)part >> log_parts), u1 = (int)((unsigned)units * (unsigned)(part + 1) >> log_parts);

    constexpr int kParts = FM * FN * 4, kMine = (kParts + WK - 1) / WK;  // parts of the tile (four rows per half wavefront), of which this wavefront stores kMine
    // Four wavefronts: the parts of fragments side by side have the same rows.  (For GPTQ with bf16 rows that decides between three wavefronts a SIMD, 166 registers, and two, 170: 10512 x 2304 349 rows
    // 39.4 / 44.8 us.)
    constexpr int kRowSets = WK == 4 ? FM : kMine;
    float inv[kRowSets][4];
#pragma unroll
    for (int e = 0; e < kRowSets; e++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int part_e = WK == 4 ? 4 * FN * e + wave : min(e * WK + wave, kParts - 1), row = m0 + 32 * ((part_e >> 2) / FN) + 8 * (part_e & 3) + 4 * (lane >> 5) + r;
            inv[e][r] = inv_scales[min(row, m - 1)];
        }
    constexpr bool kUnit = ENC == QMM_GPTQ && unit_sums(ENC, W::kFlush, HILO);  // (Q4_0 and Q6_K on two fragments have no registers for them)
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
        constexpr int kPer = HILO ? 2 : 1, kAhead = direct_ahead(ENC, FM, FN, HILO, FLUSH);
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
            ap[a] = (const uint8_t*)a16 + tile * row_bytes + (int64_t)u0 * W::kSteps * 1024 * kPer;
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
            float16v P[FM][FN], U[kUnit ? FM : 1][kUnit ? FN : 1];
            half8 sf[FM];  // (Q4_K, Q5_K: four fp32 sums)
            if constexpr (W::kMin || ENC == QMM_Q4_0) {
#pragma unroll
                for (int a = 0; a < FM; a++) {
                    const int tile = min(tile_m * FM + a, (m - 1) >> 5);
                    sf[a] = *(const half8*)((const uint8_t*)(W::kMin ? (const void*)p.sums32 : (const void*)p.sums) + ((int64_t)tile * units + u) * 1024 + l16);
                }
            }
            float of[FN][4];  // Q4_K, Q5_K: offsets of the lane's four sub-blocks
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
                if constexpr (W::kMin && (t & 3) == 3) {  // the offsets, one instruction behind every fourth step (the running sums are idle until the flush)
                    constexpr int c = t >> 2;
#pragma unroll
                    for (int f = 0; f < FN; f++) {
                        if constexpr (c == 0) {
                            const float4 o = w.offsets(f);
                            of[f][0] = o.x, of[f][1] = o.y, of[f][2] = o.z, of[f][3] = o.w;
                        }
#pragma unroll
                        for (int a = 0; a < FM; a++) {
                            const float4 s = __builtin_bit_cast(float4, sf[a]);
                            T[a][f] = __builtin_amdgcn_mfma_f32_32x32x2f32(c == 0 ? s.x : c == 1 ? s.y : c == 2 ? s.z : s.w, of[f][c], T[a][f], 0, 0, 0);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
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
                            for (int r = 0; r < 16; r++) {
                                if constexpr (kUnit) U[a][f][r] = t < W::kFlush ? d * P[a][f][r] : fmaf(d, P[a][f][r], U[a][f][r]);
                                else T[a][f][r] = fmaf(d, P[a][f][r], T[a][f][r]);
                                if constexpr (kUnit && t + 1 == W::kSteps) T[a][f][r] += U[a][f][r];
                            }
                            // (left to itself the compiler puts these off and keeps the P of every scale block)
                            if constexpr (kUnit) asm volatile("" : "+v"(U[a][f]));
                            else asm volatile("" : "+v"(T[a][f]));
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
                    const float x = vv[r] * inv[WK == 4 ? e0 / (WK * FN) : e0 / WK][r];
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

int64_t direct_units(int64_t k) { return (k + 255) / 256; }

// What a call takes, in microseconds: launches and the preparation of the lhs, a fixed part per round of workgroups (Rounds), the units of K that a wavefront
// walks, terms for the weights, the lhs and the results, and one for lhs operands beyond 8 MB, which an XCD's L2 does not keep for the next column tile.
// Fitted to the problems among 205 per encoding and lhs type (512 x 512 .. 28672 x 8192, K up to 14336, 4 .. 1300 rows, weights from memory;
// profiles/direct_and_shared_gemm__plans.txt) that these kernels serve, in every plan: 7 .. 10 % off; what it picks takes 0.6 .. 1.8 % longer on average than
// the best plan (3 % for GPTQ with bf16 rows).
// unit = 0: a plan that is not built (two fragments side by side spill registers and never win with Q4_0 and Q6_K).
struct DirectCost {
    float base, round, weights, lhs, out;  // us, us, us per MB of packed weights, us per million lhs values, us per million results and share
    float unit[6];                         // us per unit of K: the plans of kDirectPlans
    float alone[3];                        // the same of the last three with a compute unit to themselves
    float far;                             // us per 10^9 lhs operands read, where they are more than 8 MB
};
constexpr DirectPlan kDirectPlans[6] = {{1, 1, 8, 0, 1}, {2, 1, 8, 0, 1}, {1, 2, 8, 0, 1}, {1, 1, 4, 0, 1}, {2, 1, 4, 0, 1}, {1, 2, 4, 0, 1}};
constexpr bool direct_built(int encoding, int fn) { return !(fn == 2 && (encoding == QMM_Q4_0 || encoding == QMM_Q6_K)); }
constexpr DirectCost kDirectCost[6][2] = {
    // bf16 lhs; fp32 lhs
    {{3.56f, 1.4f, 0.179f, 2.88f, 2.57f, {2.79f, 4.04f, 0.0f, 2.31f, 3.43f, 0.0f}, {2.12f, 2.91f, 0.0f}, 7.01f},
     {3.51f, 1.45f, 0.182f, 3.09f, 2.33f, {2.76f, 4.02f, 0.0f, 2.3f, 3.45f, 0.0f}, {2.1f, 2.89f, 0.0f}, 5.8f}},  // Q4_0
    {{4.18f, 1.15f, 0.185f, 2.87f, 2.04f, {2.51f, 3.44f, 3.82f, 2.07f, 3.02f, 3.09f}, {1.72f, 2.19f, 2.57f}, 0.0f},
     {3.74f, 1.12f, 0.184f, 4.61f, 2.31f, {3.39f, 5.19f, 5.03f, 3.09f, 5.05f, 4.46f}, {2.27f, 3.03f, 3.07f}, 20.1f}},  // Q4_K
    {{4.18f, 1.18f, 0.159f, 2.82f, 1.94f, {2.96f, 3.89f, 4.73f, 2.42f, 3.37f, 3.99f}, {1.94f, 2.42f, 3.07f}, 0.0f},
     {3.59f, 1.37f, 0.165f, 4.42f, 2.03f, {3.74f, 5.54f, 5.74f, 3.36f, 5.45f, 5.27f}, {2.44f, 3.12f, 3.47f}, 18.7f}},  // Q5_K
    {{3.49f, 1.75f, 0.158f, 2.66f, 1.36f, {3.69f, 4.77f, 0.0f, 3.14f, 4.4f, 0.0f}, {2.27f, 2.89f, 0.0f}, 11.0f},
     {2.94f, 1.78f, 0.172f, 4.48f, 1.46f, {4.9f, 7.0f, 0.0f, 4.4f, 7.37f, 0.0f}, {2.97f, 3.91f, 0.0f}, 20.8f}},  // Q6_K
    {{4.94f, 0.0025f, 0.169f, 2.65f, 3.11f, {2.5f, 3.62f, 3.56f, 1.87f, 3.17f, 2.71f}, {1.82f, 2.7f, 2.81f}, 0.0f},
     {3.74f, 1.04f, 0.178f, 4.44f, 2.88f, {3.78f, 5.21f, 4.6f, 3.27f, 5.09f, 4.22f}, {2.55f, 3.41f, 3.4f}, 15.2f}},  // GPTQ, groups of 128
    {{4.02f, 1.17f, 0.157f, 2.49f, 2.39f, {3.3f, 4.46f, 4.6f, 2.77f, 3.92f, 4.02f}, {2.36f, 3.22f, 3.52f}, 6.54f},
     {3.77f, 1.05f, 0.175f, 4.28f, 2.75f, {4.3f, 5.96f, 5.6f, 3.67f, 5.65f, 4.97f}, {3.01f, 3.8f, 3.92f}, 15.3f}},  // GPTQ, other groups
};
constexpr bool direct_costs_match_what_is_built() {
    for (int row = 0; row < 6; row++)
        for (int type = 0; type < 2; type++)
            for (int i = 0; i < 6; i++)
                if ((kDirectCost[row][type].unit[i] != 0.0f) !=
                    direct_built(row == 0 ? QMM_Q4_0 : row == 1 ? QMM_Q4_K : row == 2 ? QMM_Q5_K : row == 3 ? QMM_Q6_K : QMM_GPTQ, kDirectPlans[i].fn))
                    return false;
    return true;
}
static_assert(direct_costs_match_what_is_built());
// The rounds of a grid of wgs workgroups per XCD (column tiles go to XCDs in eights).  Two workgroups of four wavefronts fit a compute unit; an odd
// last one has it to itself and is done sooner.
struct Rounds {
    int64_t all, full, alone;
};
Rounds rounds_of(int64_t wgs, bool pairs) {
    const int64_t cus = compute_units() / 8, deep = (wgs + cus - 1) / cus;
    return pairs ? Rounds{(deep + 1) / 2, deep / 2, deep % 2} : Rounds{deep, deep, 0};
}
// When the tiles of a launch of the staged kernel are done: `full` of them and then `last`, which take a and b us, per XCD.
double staged_tiles_us(int64_t full, int64_t last, double a, double b) {
    const int64_t cus = compute_units() / 8, busy = full % cus;  // compute units that take one more of the full ones than the others
    double some = (double)(full / cus) * a, most = busy ? some + a : some, end = most;
    for (int64_t left = last; left > 0;) {
        double& free = busy && most < some ? most : some;
        left -= &free == &most ? busy : cus - busy;
        free += b;
        end = std::max(end, free);
    }
    return end;
}
double direct_us(const DirectCost& c, int plan, int shares, int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const DirectPlan& p = kDirectPlans[plan];
    if (c.unit[plan] == 0.0f) return 1e30;
    const int64_t wgs = ((m + 32 * p.fm - 1) / (32 * p.fm)) * ((n + 256 * p.fn - 1) / (256 * p.fn)) * shares, walk = (direct_units(k) + p.wk * shares - 1) / (p.wk * shares);
    const Rounds r = rounds_of(wgs, p.wk == 4);
    const double bytes = encoding == QMM_Q6_K ? 0.82 : encoding == QMM_Q5_K ? 0.69 : 0.56, per = lhs_dtype == QMM_F32 && encoding != QMM_Q4_0 ? 2 : 1;
    const double far = 2 * m * k * per > 8e6 ? c.far * (m * k * per * 1e-9) * n / (32 * p.fn) : 0.0;
    return c.base + r.all * c.round + walk * (r.full * c.unit[plan] + r.alone * c.alone[plan % 3]) + c.weights * (bytes * n * k * 1e-6) + c.lhs * (m * k * 1e-6) +
           c.out * (m * n * 1e-6) * shares + far;
}
// The same for the kernel whose wavefronts share the lhs, fitted to the same problems from 33 rows on: 5 .. 6 % off.  It wins where its tiles of 64 x 256
// (64 x 128) fill the part with most of K in a workgroup.  us, direct plans / shared: Q4_K, bf16 rows: 14336 x 4096 200 rows 59 / 49; fp32 rows:
// 14336 x 4096 500 rows 183 / 150; Q6_K 4096 x 14336 500 bf16 rows 153 / 134; but 4096 x 4096 Q4_K 64 bf16 rows 12 / 18.
struct SharedCost {
    float base, round, weights, lhs, out;
    float unit[3], unit_alone;  // the plans of kSharedPlans; four wavefronts with a compute unit to themselves
};
constexpr DirectPlan kSharedPlans[3] = {{2, 1, 1, 0, 8}, {2, 1, 2, 0, 4}, {2, 1, 1, 0, 4}};
constexpr SharedCost kSharedCost[6][2] = {
    // bf16 lhs; fp32 lhs
    {{4.93f, 0.853f, 0.094f, 1.55f, 2.62f, {3.79f, 3.93f, 3.35f}, 2.85f}, {5.01f, 0.774f, 0.1f, 1.71f, 2.52f, {3.78f, 3.92f, 3.34f}, 2.84f}},  // Q4_0
    {{4.58f, 1.97f, 0.0798f, 1.42f, 2.57f, {2.31f, 2.56f, 2.27f}, 1.78f}, {4.49f, 1.95f, 0.0749f, 2.15f, 3.19f, {3.62f, 4.15f, 3.81f}, 2.61f}},  // Q4_K
    {{4.57f, 2.11f, 0.106f, 1.38f, 2.41f, {2.72f, 3.02f, 2.78f}, 2.08f}, {3.94f, 2.46f, 0.114f, 2.06f, 3.12f, {3.97f, 4.53f, 4.17f}, 2.83f}},  // Q5_K
    {{3.74f, 2.76f, 0.132f, 1.48f, 2.48f, {3.83f, 4.16f, 3.83f}, 2.45f}, {2.61f, 3.28f, 0.124f, 1.55f, 3.33f, {5.87f, 6.55f, 6.39f}, 3.72f}},  // Q6_K
    {{5.18f, 1.29f, 0.0415f, 1.6f, 2.58f, {2.41f, 2.58f, 2.22f}, 1.87f}, {5.93f, 0.433f, 0.0638f, 2.43f, 2.93f, {3.62f, 4.06f, 3.5f}, 2.85f}},  // GPTQ, groups of 128
    {{5.89f, 0.703f, 0.0642f, 1.57f, 2.6f, {3.54f, 3.82f, 3.28f}, 2.64f}, {5.71f, 0.809f, 0.0638f, 2.23f, 2.96f, {4.56f, 5.04f, 4.56f}, 3.49f}},  // GPTQ, other groups
};
double shared_us(const SharedCost& c, int plan, int shares, int64_t m, int64_t n, int64_t k) {
    const DirectPlan& p = kSharedPlans[plan];
    const int64_t wgs = (m + 63) / 64 * ((n + 256 * p.wn - 1) / (256 * p.wn)) * shares, walk = (direct_units(k) + p.wk * shares - 1) / (p.wk * shares);
    const Rounds r = rounds_of(wgs, p.wn * p.wk == 4);
    return c.base + r.all * c.round + walk * (r.full * c.unit[plan] + r.alone * c.unit_alone) + c.weights * (0.6 * n * k * 1e-6) + c.lhs * (m * k * 1e-6) +
           c.out * (m * n * 1e-6) * shares;
}
// The same for the kernel whose lhs and weights go to LDS by themselves (gemm_staged.hip).  On 1215 problems that it was not fitted to (512 x 512 .. 28672 x 8192, K up to
// 18944, 33 .. 4096 rows, weights from memory; profiles/staged_gemm__plans.txt): 4 .. 6 % off on average by encoding and lhs type, what it has first takes 1 .. 2 % longer than
// the best plan.  (Fitted before bf16 rows' loads were spread over the steps and before a last tile of 96 or 128 rows without its last 32 left these out: such plans cost up to 7 % less than it says.)
// other: what the GEMMs behind this file (planes, tiles) take, from 200 rows on, in us: a fixed part, per MB of weights, per million lhs values, per million
// results, per 10^9 products with the rows in 256s (8 .. 12 % off beyond direct_range, where it is asked for, and what is picked there by it takes 0.9 % longer on average than the
// faster of both; none for groups that are no multiple of 128, which have no such GEMM).
struct StagedCost {
    float base, round, weights, lhs, out, share;
    float unit[7];  // the plans of kStagedPlans; 0: not built
    float other[5];
};
constexpr DirectPlan kStagedPlans[7] = {{2, 0, 4, 0, 2}, {2, 0, 2, 0, 4}, {2, 0, 1, 0, 8}, {3, 0, 2, 0, 4}, {3, 0, 1, 0, 8}, {4, 0, 2, 0, 4}, {4, 0, 1, 0, 8}};
constexpr StagedCost kStagedCost[5][2] = {
    // bf16 lhs; fp32 lhs
    {{4.97f, 2.08f, 0.0626f, 1.61f, 1.88f, 4.7f, {2.78f, 2.04f, 1.83f, 2.75f, 2.31f, 3.41f, 2.88f}, {16.1f, 0.147f, 1.61f, 0.0f, 2.11f}},
     {3.99f, 2.7f, 0.088f, 2.97f, 2.61f, 4.77f, {4.74f, 3.32f, 2.98f, 4.73f, 3.94f, 0.0f, 0.0f}, {16.3f, 4.73f, 3.8f, 4.79f, 2.69f}}},  // Q4_K
    {{5.06f, 2.12f, 0.0665f, 1.39f, 1.74f, 4.71f, {3.27f, 2.61f, 2.23f, 3.12f, 2.69f, 4.08f, 3.4f}, {14.7f, 1.05f, 2.44f, 0.107f, 1.61f}},
     {3.65f, 3.15f, 0.0849f, 2.75f, 2.55f, 4.65f, {4.94f, 3.96f, 3.3f, 5.02f, 4.28f, 0.0f, 0.0f}, {25.6f, 3.16f, 4.81f, 3.69f, 2.82f}}},  // Q5_K
    {{3.93f, 3.1f, 0.0983f, 1.55f, 2.23f, 4.61f, {4.2f, 3.56f, 3.19f, 4.28f, 3.82f, 5.69f, 5.04f}, {13.2f, 1.45f, 2.3f, 0.0f, 2.77f}},
     {2.13f, 4.38f, 0.141f, 3.05f, 3.48f, 4.43f, {6.53f, 5.51f, 4.88f, 7.3f, 6.59f, 0.0f, 0.0f}, {23.6f, 2.72f, 5.61f, 3.47f, 5.44f}}},  // Q6_K
    {{5.21f, 2.55f, 0.0331f, 1.43f, 1.55f, 4.57f, {2.45f, 1.9f, 1.77f, 2.53f, 2.21f, 3.15f, 2.72f}, {14.9f, 0.0609f, 1.56f, 0.0f, 1.88f}},
     {4.51f, 2.82f, 0.0544f, 2.78f, 2.26f, 4.62f, {4.37f, 2.93f, 2.66f, 4.4f, 3.7f, 0.0f, 0.0f}, {9.65f, 1.9f, 3.89f, 4.38f, 3.13f}}},  // GPTQ, groups of 128
    {{5.25f, 2.87f, 0.0408f, 1.41f, 1.22f, 4.49f, {3.16f, 2.72f, 2.65f, 3.77f, 3.43f, 0.0f, 0.0f}, {}},
     {4.16f, 3.4f, 0.0772f, 2.7f, 2.3f, 4.44f, {4.61f, 3.56f, 3.39f, 4.98f, 4.46f, 0.0f, 0.0f}, {}}},  // GPTQ, other groups
};
int staged_row(int encoding, int group) {
    return encoding == QMM_Q4_K ? 0 : encoding == QMM_Q5_K ? 1 : encoding == QMM_Q6_K ? 2 : encoding == QMM_GPTQ ? (group % 128 == 0 ? 3 : 4) : -1;
}
double packed_mb(int encoding, int64_t n, int64_t k) { return (encoding == QMM_Q6_K ? 0.82 : encoding == QMM_Q5_K ? 0.69 : 0.56) * n * k * 1e-6; }
// The tiles of one plan on `sections` column sections.  A last row tile of up to 32 rows takes 0.8 of the unit of one of 64.
double staged_tiles_us(const StagedCost& c, int i, int64_t m, int64_t sections, int64_t walk) {
    const DirectPlan& p = kStagedPlans[i];
    const bool short_last = staged_short_last(p.fm, m, sections);
    const int64_t full = short_last ? m / (32 * p.fm) : (m + 32 * p.fm - 1) / (32 * p.fm);
    return staged_tiles_us(full * sections, short_last ? sections : 0, c.round + walk * c.unit[i], c.round + walk * 0.8 * c.unit[p.wn == 2 ? 0 : p.wn == 4 ? 1 : 2]);
}
// What a plan's fp32 sums cost: the square of the relative error of the results (2-norm, against 64 bits) in units of 2^-48 / 6, the mean square of a rounding
// halved.  An addition counts by the share of K that its sum holds by then: `unit` times half the squares of the parts' lengths, `join` for adding the parts up
// in order; `first`: additions to zero, which are exact; `length`: what grows with K however it is cut.  Fitted to every plan on 22 K of 256 .. 28672
// (profiles/relative_error_by_plan.txt): 0.07 .. 0.4 % off on average by encoding, lhs type and kind of sums, 1.3 % at most, most of which is common to the plans of a K.
// Kinds that sum alike share a row; the shared and the staged kernel with codes from 0 do not (Q4_K 4096 x 4096, 200 bf16 rows: 1.907e-7 shared, 1.894e-7 staged).
// Of 9504 pairs of a plan and a staged one it takes the staged one in 35 where that is more than 0.05 % further off (0.4 % at most), and refuses 125 that are no further off.
struct SumsError {
    float base, unit, join, first, length;
};
constexpr SumsError kSumsError[5][2][4] = {
    // the direct kernel; the shared one, codes from 0 (fp32 rows: around their middle); the staged one, likewise; both with bf16 rows, codes around their middle
    {{{2.29f, 9.77f, 1.24f, 0.084f, -0.002f}, {54.12f, 2.12f, 0.838f, 0.922f, 0.021f}, {53.18f, 2.12f, 0.936f, 0.746f, 0.018f}, {7.92f, 1.11f, 1.25f, -1.56f, 0.03f}},
     {{37.22f, 9.76f, 1.24f, 0.054f, 0.027f}, {43.18f, 1.1f, 1.25f, -1.65f, 0.117f}, {43.18f, 1.1f, 1.25f, -1.65f, 0.117f}, {43.18f, 1.1f, 1.25f, -1.65f, 0.117f}}},  // Q4_K
    {{{4.97f, 9.75f, 1.23f, 0.018f, -0.001f}, {73.39f, 2.12f, 0.843f, 0.955f, 0.021f}, {72.41f, 2.12f, 0.932f, 0.831f, 0.018f}, {10.56f, 1.11f, 1.24f, -1.57f, 0.027f}},
     {{38.88f, 9.76f, 1.23f, 0.107f, 0.031f}, {44.89f, 1.1f, 1.23f, -1.64f, 0.116f}, {44.89f, 1.1f, 1.23f, -1.64f, 0.116f}, {44.89f, 1.1f, 1.23f, -1.64f, 0.116f}}},  // Q5_K
    {{{8.29f, 2.17f, 1.22f, -0.008f, 0.0f}, {16.1f, 1.08f, 1.28f, -0.05f, 0.0f}, {16.1f, 1.08f, 1.28f, -0.05f, 0.0f}, {}},
     {{36.48f, 2.17f, 1.23f, -0.058f, -0.001f}, {65.7f, 1.08f, 1.28f, -0.064f, 0.002f}, {65.7f, 1.08f, 1.28f, -0.064f, 0.002f}, {}}},  // Q6_K
    {{{0.66f, 2.17f, 1.26f, -0.03f, -0.001f}, {0.66f, 2.17f, 1.26f, -0.03f, -0.001f}, {0.66f, 2.17f, 1.26f, -0.03f, -0.001f}, {}},
     {{17.3f, 2.17f, 1.24f, -0.001f, 0.009f}, {17.3f, 2.17f, 1.24f, -0.001f, 0.009f}, {17.3f, 2.17f, 1.24f, -0.001f, 0.009f}, {}}},  // GPTQ, groups of 128
    {{{5.95f, 1.13f, 1.24f, -1.55f, 0.001f}, {5.95f, 1.13f, 1.24f, -1.55f, 0.001f}, {5.95f, 1.13f, 1.24f, -1.55f, 0.001f}, {}},
     {{8.41f, 8.66f, 1.25f, 0.003f, 0.007f}, {8.41f, 8.66f, 1.25f, 0.003f, 0.007f}, {8.41f, 8.66f, 1.25f, 0.003f, 0.007f}, {}}},  // GPTQ, other groups
};
// fold: units after which the staged kernel folds its sums (0: it does not).
double sums_error(const SumsError& e, const DirectPlan& p, int64_t units, int64_t fold = 0) {
    const int log_parts = __builtin_ctz((unsigned)(p.wk * p.shares));
    double squares = 0.0, join = 0.0;
    int held_parts = 0;
    for (int s = 0; s < p.shares; s++) {
        int64_t held = 0;  // units in the sum of this workgroup
        for (int i = s * p.wk; i < (s + 1) * p.wk; i++) {
            const int64_t q = (units * (i + 1) >> log_parts) - (units * i >> log_parts);
            if (q == 0) continue;
            for (int64_t done = 0; done < q;) {
                const int64_t some = fold ? std::min(fold, q - done) : q;
                squares += (double)(some * some), held_parts++;
                if (done > 0) join += (double)(done + some);
                done += some;
            }
            if (held > 0) join += (double)(held + q);
            held += q;
        }
        if (s == 1 && held < units) join += (double)units;
    }
    return e.base + e.length * (double)units + (e.unit * 0.5 * squares + e.join * join + e.first * held_parts) / (double)units;
}
// Codes around their middle: unit sums, and no plan with 128 rows a wavefront, which has no registers for them.  Row tiles of 96 (the last one of 128 may be one) have wavefronts whose loads cross from one
// 32 rows' operands to another's, with offsets of 32 bits; those 32 rows take 128 K bytes: not from K = 2^23 on.
constexpr int64_t kStagedLongRows = 1 << 23;
bool staged_has(const StagedCost& c, int plan, bool centred, int64_t k) {
    return c.unit[plan] != 0.0f && !(centred && kStagedPlans[plan].fm == 4) && (k < kStagedLongRows || kStagedPlans[plan].fm == 2);
}
// What loads to LDS want.  Scales and zeros of GPTQ lie so; only a Q6_K tensor may begin elsewhere.
bool staged_takes(const void* w) { return ((uintptr_t)w & 3) == 0; }
// The best of its plans whose parts of K are at most `longest` units and whose sums are off by no more than `most` (sums_error); returns its time (1e30: there is none).
double staged_plan(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, bool whole_tiles, bool centred, int64_t longest, double most, DirectPlan& best) {
    const int row = staged_row(encoding, group);
    // (Q6_K: the last block would be read two bytes beyond its end where it begins at a multiple of four, which it does if the blocks before it are even in number)
    if (encoding == QMM_Q6_K && (n * direct_units(k)) % 2 != 0) return 1e30;
    if (row < 0 || k % 256 || k >= 1 << 27 || m > 1 << 21 || n > 1 << 23 || kernel_disabled("staged")) return 1e30;  // (the grid's y and z have 16 bits)
    const int type = lhs_dtype == QMM_F32 ? 1 : 0;
    const StagedCost& c = kStagedCost[row][type];
    const SumsError& e = kSumsError[row][type][centred ? 3 : 2];
    double us = 1e30;
    for (int shares = 1; shares <= (whole_tiles ? 1 : 2); shares++)
        for (int i = 0; i < 7; i++) {
            DirectPlan p = kStagedPlans[i];
            p.shares = shares;
            const int64_t parts = p.wk * shares, walk = (direct_units(k) + parts - 1) / parts;
            if (!staged_has(c, i, centred, k)) continue;
            const double t = c.base + staged_tiles_us(c, i, m, (n + 256 * p.wn - 1) / (256 * p.wn) * shares, walk) + c.weights * packed_mb(encoding, n, k) + c.lhs * (m * k * 1e-6) +
                             (c.out + c.share * (shares - 1)) * (m * n * 1e-6);
            if (walk <= longest && t < us && sums_error(e, p, direct_units(k)) <= most) us = t, best = p;
            // (folded sums: 1.03, 14336 x 4096 with 160 bf16 rows 33.3 -> 35.0 us)
            p.fold = walk > kStagedFold && staged_folds(encoding, encoding == QMM_GPTQ ? (group % 128 == 0 ? 8 : 2) : 16, p.fm, type == 1);
            if (p.fold && 1.03 * t < us && sums_error(e, p, direct_units(k), kStagedFold) <= most) us = 1.03 * t, best = p;
        }
    return us;
}
// Calls that go to this file for the sake of the direct and the shared kernel: up to where the GEMMs that unpack a tile or all weights once and then share
// them take over (r = outputs, w = weights, in Mi; beyond about 1100 rows the lhs no longer stays in an L2).
bool direct_range(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    if (encoding == QMM_GPTQ && group % 128) return true;  // (the alternative is the decode kernel, eight rows a pass)
    const bool f32 = lhs_dtype == QMM_F32, few_products = encoding == QMM_Q4_0 || encoding == QMM_Q6_K;
    const double w = (double)n * k / (1 << 20), r = (double)m * n / (1 << 20);
    const double most = few_products ? 3.5 : k > 4096 && (encoding == QMM_Q4_K || encoding == QMM_GPTQ) ? 1.3 : 2.75;  // bf16 outputs
    const int64_t anyway = few_products ? 450 : 0;  // rows up to which the number of outputs does not matter
    if (r <= (f32 && encoding != QMM_Q4_0 ? 1.6 : 1)) return true;
    // fp32 rows are split in two fp16 terms here and in the other kernels, so both multiply twice; the others take K in two passes.  us, others / here:
    // Q4_K 14336 x 4096 800 rows 327 / 232, 5120 x 5120 1300 rows 239 / 198; Q6_K 14336 x 4096 800 rows 514 / 380;
    // but GPTQ 4096 x 14336 1050 rows 470 / 560.
    const bool shared = !kernel_disabled("shared");
    if (f32) {
        if (shared && encoding != QMM_Q4_0 && (m <= 1100 || (m <= 1400 && r <= 5.5)) && (encoding != QMM_GPTQ || k <= 8192)) return true;
        return m <= (w <= 24 || (encoding != QMM_Q4_0 && encoding != QMM_GPTQ) ? 720 : 450) || (k <= 1024 ? r <= 6 : m < 1100 && r <= 3.5);
    }
    // (one round of 64 x 256 tiles that fills the compute units by four fifths or more: 11008 x 4096 320 bf16 rows Q4_K 78 / 55, GPTQ 71 / 53, Q5_K 85 / 63;
    // 8192 x 8192 500 rows Q6_K 205 / 162, Q5_K 145 / 119, but Q4_K 106 / 105 and GPTQ 92 / 101)
    const int64_t tiles = (m + 63) / 64 * ((n + 255) / 256);
    if (shared && 5 * tiles >= 4 * compute_units() && tiles <= compute_units() && k <= (encoding == QMM_Q4_K || encoding == QMM_GPTQ ? 4096 : 8192)) return true;
    return m <= anyway || (m <= 1100 && r <= most);
}
// whole_tiles: one workgroup per tile (bf16 results are stored, not added up); staged: the weights lie as the staged kernel wants them; beyond: the call
// would not be this file's without that kernel (direct_range); like: with that plan's cut of K and kind of sums
DirectPlan direct_plan(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, bool whole_tiles, bool staged, bool beyond, const DirectPlan* like = nullptr) {
    const int row = encoding == QMM_Q4_0 ? 0 : encoding == QMM_Q4_K ? 1 : encoding == QMM_Q5_K ? 2 : encoding == QMM_Q6_K ? 3 : group % 128 == 0 ? 4 : 5;
    const int type = lhs_dtype == QMM_F32 ? 1 : 0;
    DirectPlan best{1, 1, 8, 1, 1};
    double us = 1e29;
    auto consider = [&](const DirectPlan& p, int shares, double t) {
        if (t >= us || (like && (p.wk != like->wk || shares != like->shares || (p.wn > 1) != (like->wn > 1)))) return;
        us = t;
        best = p;
        best.shares = shares;
    };
    if (like && like->fn == 0) {  // (several matrices that all go to the staged kernel with this cut: the tile that suits them together)
        for (const DirectPlan& p : kStagedPlans) {
            const StagedCost& c = kStagedCost[staged_row(encoding, group)][type];
            const int i = (int)(&p - kStagedPlans);
            if (!staged_has(c, i, like->centred, k) || p.wk != like->wk) continue;
            const int64_t walk = (direct_units(k) + p.wk * like->shares - 1) / (p.wk * like->shares);
            const double t = staged_tiles_us(c, i, m, (n + 256 * p.wn - 1) / (256 * p.wn) * like->shares, walk);
            if (t < us) us = t, best = p, best.shares = like->shares, best.centred = like->centred;
        }
        return best;
    }
    // Q6_K up to 64 rows, which the small-batch kernel would take in passes of 16: only plans with parts of K of up to 2048, as exact as that kernel
    // (28672 x 8192 with 64 bf16 rows, shared: parts of 2048 1.0e-7 relative error, of 4096 1.1e-7, small-batch kernel 0.98e-7; 101, 93 and 224 us).
    const int64_t longest = encoding == QMM_Q6_K && m <= 64 ? 8 : 1 << 20;  // units of K in a part
    const bool shared = m > 32 && !kernel_disabled("shared");
    for (int shares = 1; shares <= (whole_tiles ? 1 : 2); shares++) {
        for (int i = 0; i < 6; i++)
            if (direct_units(k) <= longest * kDirectPlans[i].wk * shares)
                consider(kDirectPlans[i], shares, direct_us(kDirectCost[row][type], i, shares, encoding, lhs_dtype, m, n, k));
        for (int i = 0; shared && i < 3; i++)  // (between predictions this close workgroups of four wavefronts took 3 % longer)
            if (direct_units(k) <= longest * kSharedPlans[i].wk * shares)
                consider(kSharedPlans[i], shares, shared_us(kSharedCost[row][type], i, shares, m, n, k) * (i == 2 ? 1.03 : 1.0));
    }
    // (up to 32 rows half of the staged kernel's smallest tile is empty: GPTQ 28672 x 8192 17 bf16 rows 46 .. 48 us direct, 50 .. 52 staged)
    if (like || !staged || (m <= 32 && !beyond) || (encoding == QMM_Q6_K && !beyond && (m <= 64 || best.wn == 1))) return best;
    // The staged kernel, held to the error of what it replaces (sums_error), and where that is the direct kernel with the codes of Q4_K and Q5_K around their
    // middle (KQuantWeights), as there; Q6_K, whose sums leave the matrix cores half as often as in the direct kernel, only for the shared one.
    // Beyond the range of those two anything is more exact than the GEMMs that share unpacked weights (2.2e-7 .. 3.5e-6).
    const bool k_quant = encoding == QMM_Q4_K || encoding == QMM_Q5_K;
    const bool centred = k_quant && (type == 1 || (!beyond && best.wn == 1) || (encoding == QMM_Q5_K && m <= 64));
    // As far as parts of K longer than those of that plan have been tried.
    const int64_t parts = best.wk * best.shares, part = (direct_units(k) + parts - 1) / parts;
    const int64_t chain = beyond ? 1 << 20 : std::max<int64_t>(4, k_quant && type == 1 && best.wn == 1 && part > 1 ? 5 * part : part);
    const int errors = staged_row(encoding, group);
    const double most = beyond || errors < 0 ? 1e30 : sums_error(kSumsError[errors][type][best.wn == 1 ? 0 : centred ? 3 : 1], best, direct_units(k));
    DirectPlan p;
    // (4 %: as far as the predictions are off; within it the staged kernel was slower as often as faster, GPTQ 4552 x 3072 472 fp32 rows 55.7 and 56.4 us predicted,
    // 61 and 56 taken; codes around the middle are not in its figures)
    if (staged_plan(encoding, lhs_dtype, m, n, k, group, whole_tiles, centred, chain, most, p) * (centred && type == 0 ? 1.08 : 1.04) < us) {
        best = p;
        best.centred = centred;
    }
    return best;
}

template <int ENC, int FLUSH, int FM, int FN, int WK, bool HILO>
hipError_t run_direct(const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units, int shares, hipStream_t s) {
    const int tiles_m = (int)((m + 32 * FM - 1) / (32 * FM));
    int eights = 0;
    for (int j = 0; j < mats.count; j++) mats.end[j] = eights += (mats.n[j] + 256 * FN - 1) / (256 * FN);
    constexpr int lds = WK * direct_slot<WeightsOf<ENC, FN, FLUSH, true>>(FM * FN);
    hipError_t e = allow_full_lds<gemm_direct_kernel<ENC, FLUSH, FM, FN, WK, HILO>>();
    if (e != hipSuccess) return e;
    const DirectGrid g = direct_grid(tiles_m, eights * shares);
    gemm_direct_kernel<ENC, FLUSH, FM, FN, WK, HILO><<<g.grid, dim3(64 * WK), lds, s>>>(mats.w[0], p.a16, p.inv, mats.n[0], (int)m, units, g.tiles_m, shares, mats.count, wt, mats, p, out16);
    return hipGetLastError();
}

template <int ENC, int FLUSH, bool HILO>
hipError_t run_direct_plan(const DirectPlan& pl, const WeightTensors& wt, const DirectMats& mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units,
                           hipStream_t s) {
#define QMM_GD(FM, FN, WK)                           \
    if constexpr (direct_built(ENC, FN))             \
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

bool gemm_direct_wanted(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, const void* w_at) {
    if (kernel_disabled("direct") || k % (encoding == QMM_GPTQ || encoding == QMM_Q4_0 ? 32 : 256) || n * k >= ((int64_t)1 << 32)) return false;
    if (encoding == QMM_GPTQ && (n % 8 || group % 32)) return false;
    // Served from `from` rows on, where this kernel's time crosses that of the small-batch kernels (passes of four to sixteen rows over
    // the weights; at their best on long weight matrices and on the row lengths their wavefronts divide evenly, 512, 2048 or 4096 values;
    // this kernel has no such preference), and up to where it crosses that of the GEMMs behind it (direct_range).  Both lines were fitted to
    // timings of 4700 calls, 512 x 512 .. 28672 x 4096 with K of 512 .. 14336 and 1 .. 2048 rows: within 2 % on average of always taking
    // the faster of the two.  E.g. 5120 x 5120, 17 bf16 rows: Q4_0 22 -> 16 us, Q4_K 19.6 -> 14.4, Q5_K 34 -> 15.7, Q6_K 54 -> 17.9.
    // (Up to 16 rows, and up to 64 on many shapes, the kernels for a few rows are asked first: there `from` counts where those decline, K no multiple of 256 and odd numbers of Q6_K blocks among it.)
    const bool f32 = lhs_dtype == QMM_F32, wide = n >= 6000;
    const double w = (double)n * k / (1 << 20);
    int64_t from = 17;
    switch (encoding) {
        case QMM_Q4_0:
            from = wide && k <= 1024 ? 3 : k <= 2048 ? 5 : 17;
            break;
        case QMM_Q4_K:
            from = n >= 2048 && (k <= 1024 || (k < 1536 && w <= 8)) ? 2 : 9;
            break;
        case QMM_Q5_K:
            // (5 .. 16 bf16 rows on a long K: the small-batch kernel cuts it into rounds side by side; 1024 x 14336 9 rows 22.2 / 12.5 us)
            from = wide && k <= 2048 ? 2 : n >= 2048 && (k % 512 || w <= (f32 ? 16 : 24)) ? 3 : w <= 32 && (f32 || k <= 8192 || k % 512) ? 5 : f32 ? 9 : 17;
            break;
        case QMM_Q6_K:
            // (fp32 rows with K = 4096, one round of the small-batch kernel, on a vocabulary's columns: 9 .. 16 rows on 128256 x 4096 216 / 151 us, 40960 x 4096
            // 71 / 66, but 32000 x 4096 58 / 60, 128256 x 2048 110 / 165, 65536 x 8192 209 / 238)
            if (f32) from = k % 2048 == 0 ? (k == 4096 && n > 36000 ? 17 : 9) : wide ? 3 : n >= 2048 ? 4 : 6;
            else from = k % 2048 == 0 && !(wide && k <= 2048) ? (w <= 30 && k <= 8192 ? 5 : 17) : wide ? 2 : n >= 2048 ? 3 : 6;
            break;
        case QMM_GPTQ:
            // Groups that are no multiple of 128: the alternative is the decode kernel, eight rows a pass.
            if (group % 128) return m >= (k >= 7936 && n <= 4096 ? 1 : k >= 2048 ? 2 : w >= 1 ? 3 : 5);
            from = !f32 || k < 2048 ? 17 : k <= 8192 ? 8 : 9;
            break;
        default: return false;
    }
    if (m < from) return false;
    if (direct_range(encoding, lhs_dtype, m, n, k, group)) return true;
    // Beyond, the staged kernel against the GEMMs that unpack the weights once.  us, those / here: Q4_K 14336 x 4096 320 bf16 rows 85 / 60, 800 152 / 120, 4096 x 14336 2048 rows
    // 299 / 261; Q5_K 32000 x 4096 200 rows 167 / 82; Q4_K 14336 x 4096 1300 fp32 rows 522 / 347.  With many bf16 rows on many columns those run at their best,
    // 256 x 256 results at a time, which the figures of `other` do not know (14336 x 4096 2048 rows 260 / 281, 5120 x 5120 2500 rows 163 / 191, 4096 x 4096 3000 rows 126 / 135).
    const int row = staged_row(encoding, group);
    if (row < 0 || !staged_takes(w_at) || (!f32 && m > 1600 && (n > 4096 || (m > 2048 && k <= 8192)))) return false;
    // On a short K those are the more exact ones for fp32 rows (relative error, those / here: GPTQ K = 256 7.6e-8 / 1.0e-7, 512 9.7e-8 / 1.1e-7, 768 1.1e-7 / 1.1e-7; Q6_K
    // 1.4e-7 / 2.0e-7, 1.8e-7 / 2.0e-7, 2.3e-7 / 2.0e-7).
    if (f32 && k < 768 && (encoding == QMM_GPTQ || encoding == QMM_Q6_K)) return false;
    const float(&o)[5] = kStagedCost[row][f32 ? 1 : 0].other;
    DirectPlan p;
    return staged_plan(encoding, lhs_dtype, m, n, k, group, false, false, 1 << 20, 1e30, p) <
           (f32 || m <= 1024 ? 0.95 : 0.9) * (o[0] + o[1] * packed_mb(encoding, n, k) + o[2] * (m * k * 1e-6) + o[3] * (m * n * 1e-6) + o[4] * (1e-9 * ((m + 255) / 256 * 256) * n * k));
}

bool gemm_direct_takes_staged(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    return direct_plan(encoding, lhs_dtype, m, n, k, group, false, true, !direct_range(encoding, lhs_dtype, m, n, k, group)).fn == 0;
}

int64_t gemm_direct_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t k) {
    return direct_space(nullptr, lhs_dtype == QMM_F32 && encoding != QMM_Q4_0, encoding == QMM_Q4_K || encoding == QMM_Q5_K || encoding == QMM_Q4_0,
                        encoding == QMM_Q4_K || encoding == QMM_Q5_K, m, k).bytes;
}

// Several matrices: one preparation, and one launch for all those whose own plans cut K the same way (the order of the sums is that of a
// call of its own; the tile is the one that suits them together).  q | k | v of 4096 | 1024 | 1024 x 4096 with 16 rows: one launch for three.
hipError_t launch_gemm_direct(int encoding, const void* lhs, int lhs_dtype, int count, const void* const* ws, const int64_t* ns, float* const* outs,
                              const uint16_t* scales, const uint32_t* qzeros, int group, int64_t m, int64_t k, uint16_t* out16, void* workspace,
                              hipStream_t s, bool any_rows, const GptqOrder* order) {
    const bool q40 = encoding == QMM_Q4_0, f32 = lhs_dtype == QMM_F32, sums = encoding == QMM_Q4_K || encoding == QMM_Q5_K || q40;
    if (count < 1 || count > kDirectMaxMats) return hipErrorInvalidValue;
    const DirectSpace p = direct_space(workspace, f32 && !q40, sums, sums && !q40, m, k);
    DirectPlan plans[kDirectMaxMats];
    DirectMats zero{};
    int64_t zeros = 0;
    for (int j = 0; j < count; j++) {
        plans[j] = direct_plan(encoding, lhs_dtype, m, ns[j], k, group, out16 != nullptr, staged_takes(ws[j]), !any_rows && !direct_range(encoding, lhs_dtype, m, ns[j], k, group));
        if (plans[j].shares > 1) zero.out[zero.count] = outs[j], zero.n[zero.count++] = (int)ns[j], zeros = std::max(zeros, m * ns[j]);
    }
    const unsigned grid = (unsigned)((m + 63) / 64 * 64 + std::min<int64_t>(1024, (zeros + 4095) / 4096));
    const int threads = order ? sorted_prep_threads(k) : prep_threads(k);
    if (q40) {
        if (f32) direct_prep_q8_kernel<float><<<dim3(grid), dim3(threads), 0, s>>>((const float*)lhs, (int)m, (int)k, p, zero);
        else direct_prep_q8_kernel<uint16_t><<<dim3(grid), dim3(threads), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, zero);
    } else if (order) {  // (the rest of the path takes it up to K = 32768, fp32 rows of 128 KB)
        if (encoding != QMM_GPTQ || k % 32 || k > 32768) return hipErrorInvalidValue;
        bool lhs_done;
        hipError_t e = launch_gptq_order(*order, ns[0], k, group, lhs, lhs_dtype, m, p, zero, zeros, lhs_done, s);
        if (e == hipSuccess && !lhs_done)
            e = f32 ? allow_full_lds<direct_prep_kernel<float, kOrderGptq, true>, 64>() : allow_full_lds<direct_prep_kernel<uint16_t, kOrderGptq, true>, 64>();
        if (e != hipSuccess) return e;
        const size_t row = (size_t)k * (f32 ? 4 : 2);
        const int32_t* const source = order->space.source;
        if (lhs_done) {
        } else if (f32) direct_prep_kernel<float, kOrderGptq, true><<<dim3(grid), dim3(threads), row, s>>>((const float*)lhs, (int)m, (int)k, p, sums, zero, source);
        else direct_prep_kernel<uint16_t, kOrderGptq, true><<<dim3(grid), dim3(threads), row, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, sums, zero, source);
    } else if (encoding == QMM_GPTQ) {
        if (f32) direct_prep_kernel<float, kOrderGptq><<<dim3(grid), dim3(threads), 0, s>>>((const float*)lhs, (int)m, (int)k, p, sums, zero, nullptr);
        else direct_prep_kernel<uint16_t, kOrderGptq><<<dim3(grid), dim3(threads), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, sums, zero, nullptr);
    } else {
        if (f32) direct_prep_kernel<float, kOrderK><<<dim3(grid), dim3(threads), 0, s>>>((const float*)lhs, (int)m, (int)k, p, sums, zero, nullptr);
        else direct_prep_kernel<uint16_t, kOrderK><<<dim3(grid), dim3(threads), 0, s>>>((const uint16_t*)lhs, (int)m, (int)k, p, sums, zero, nullptr);
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
            if (done[i] || plans[i].wk != pl.wk || plans[i].shares != pl.shares || (plans[i].wn > 1) != (pl.wn > 1) || (plans[i].fn == 0) != (pl.fn == 0) ||
                plans[i].centred != pl.centred)
                continue;
            mats.w[mats.count] = (const uint8_t*)ws[i], mats.out[mats.count] = outs[i], mats.n[mats.count++] = (int)ns[i];
            n += ns[i];
            done[i] = true;
        }
        if (mats.count > 1) pl = direct_plan(encoding, lhs_dtype, m, n, k, group, false, true, false, &pl);
        if (pl.fn == 0) {
            e = launch_gemm_staged(encoding, f32 && !q40, pl, wt, mats, p, out16, m, units, s);
            continue;
        }
        if (pl.wn > 1) {
            e = launch_gemm_shared(encoding, f32 && !q40, pl, wt, mats, p, out16, m, units, s);
            continue;
        }
#define QMM_GD_ENC(ENC, FLUSH) \
    e = f32 ? run_direct_plan<ENC, FLUSH, true>(pl, wt, mats, p, out16, m, units, s) : run_direct_plan<ENC, FLUSH, false>(pl, wt, mats, p, out16, m, units, s)
        if (q40) e = run_direct_plan<QMM_Q4_0, 2, false>(pl, wt, mats, p, out16, m, units, s);
        else if (encoding == QMM_Q4_K) QMM_GD_ENC(QMM_Q4_K, 16);
        else if (encoding == QMM_Q5_K) QMM_GD_ENC(QMM_Q5_K, 16);
        else if (encoding == QMM_Q6_K) QMM_GD_ENC(QMM_Q6_K, 8);
        else if (group % 128 == 0) QMM_GD_ENC(QMM_GPTQ, 8);
        else QMM_GD_ENC(QMM_GPTQ, 2);
#undef QMM_GD_ENC
    }
    return e;
}

}  // namespace qmm
