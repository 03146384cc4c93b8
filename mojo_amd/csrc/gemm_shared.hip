// The direct GEMM (gemm_direct.hip) for products large enough to fill the part without cutting K into many pieces: its wavefronts share the lhs.
//
// There every wavefront reads the lhs for itself from L2, 1 KB per matrix-core instruction with 32 columns a wavefront, and the 64 bytes per
// clock of a compute unit's vector memory path set the rate (half of what the matrix cores do).  Here WN wavefronts side by side (32 columns
// each) work on the same 32 FM rows: the lhs operands go through LDS (128 bytes per clock), loaded by the workgroup once, two chunks ahead, one
// barrier per chunk of 16 KB.  Weights as there: packed, a unit of K ahead, unpacked between the matrix-core instructions by the wavefront that
// owns the columns.  WK parts of K per workgroup.
//
// A unit of K (256 columns) of eight wavefronts takes 2.0 .. 2.3 us with bf16 rows and Q4_K, 1.4 of them the matrix cores alone; the unpacking, the
// lhs, the weights' loads and the barriers each cost about a tenth on top.  Tried without gain: operands read two steps ahead with four LDS
// buffers and the lhs requested six chunks ahead (+ 4 %, twice the barriers); the two parts of K half a unit out of phase (+ 4 %); 128 rows per
// wavefront (GPTQ - 22 % per row, but half the workgroups; the K-quants spill registers).
#include "gemm_direct.h"

namespace qmm {

namespace {

constexpr int kLhsBuffers = 2;
constexpr int64_t kFewSharedRows = 64;  // up to which Q5_K and Q6_K take their most exact sums (KQuantWeights, Q6Weights)

// Column tiles of 32 WN.  (The first arguments arrive in scalar registers with the workgroup.)
template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER>
__global__ __launch_bounds__(64 * WN * WK, 2) void gemm_shared_kernel(const uint8_t* w0, const void* a16, int rows0, int m, int units, int tiles_m, int shares, int count,
                                                                      WeightTensors wt, DirectMats mats, DirectSpace p, uint16_t* __restrict__ out16) {
    using W = WeightsOf<ENC, 1, FLUSH, CENTER>;
    constexpr int kPer = HILO ? 2 : 1, kChunk = 8 / kPer, kChunks = W::kSteps / kChunk;
    constexpr int kBuf = FM * kChunk * kPer * 1024, kLoads = FM * kChunk * kPer / WN;
    static_assert(kChunks % kLhsBuffers == 0 && kLoads * WN == FM * kChunk * kPer, "buffers alternate within a unit; whole loads per wavefront");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];  // [WK][kLhsBuffers][kBuf] lhs, [WN WK] packed rows, the inverse row scales
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wn = wave % WN, wk = wave / WN;
    float* const inv = (float*)(smem + WK * kLhsBuffers * kBuf + WN * WK * W::kStage);
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
    if (tile_n * 32 * WN >= wt.n) return;
    const int n0 = tile_n * 32 * WN + 32 * wn, m0 = tile_m * 32 * FM;
    // this wavefront's units of K; the workgroup's barriers are those of its longest part
    constexpr int kLogWk = WK == 2 ? 1 : 0;
    const int log_parts = kLogWk + shares - 1, part = share * WK + wk, walk = (units + (1 << log_parts) - 1) >> log_parts;
    const int u0 = (int)((unsigned)units * (unsigned)part >> log_parts), u1 = (int)((unsigned)units * (unsigned)(part + 1) >> log_parts);

    constexpr bool kUnit = unit_sums(ENC, W::kFlush, HILO);
    float16v T[FM];
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) T[a][r] = 0.0f;

    const float16v zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Q4_K, Q5_K: the steps at which the sums of the lhs are asked for and multiplied (asked for at step 12 and waited for behind the last one they cost 8 .. 13 % with CENTER)
    constexpr int kSumsAt = 2, kOffsetsAt = 13;
    const uint32_t l16 = lane * 16;
    uint8_t* const bufs = smem + wk * kLhsBuffers * kBuf;
    W w;
    w.init(wt, n0, lane, smem + WK * kLhsBuffers * kBuf + wave * W::kStage);
    // the lhs: piece j of a chunk (1 KB) is operand j % (kChunk kPer) of row tile j / (kChunk kPer); this wavefront brings pieces wn, wn + WN, ...
    const int64_t row_bytes = (int64_t)units * W::kSteps * 1024 * kPer;
    const int last_tile = (m - 1) >> 5;
    const uint8_t* src[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int piece = wn + WN * j;
        src[j] = (const uint8_t*)a16 + min(tile_m * FM + piece / (kChunk * kPer), last_tile) * row_bytes +
                 ((int64_t)u0 * W::kSteps * kPer + piece % (kChunk * kPer)) * 1024;
    }
    // chunk c is computed on while c + 1 goes from registers to LDS and c + 2 is on its way
    gd_u4 held[kLoads];
    const int last_chunk = (u1 - u0) * kChunks - 1;
    auto load_lhs = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kLoads; j++) held[j] = *(const gd_u4*)(src[j] + min(chunk, last_chunk) * (kChunk * kPer * 1024) + l16);
    };
    auto store_lhs = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kLoads; j++) *(gd_u4*)(bufs + slot * kBuf + (wn + WN * j) * 1024 + l16) = held[j];
    };
    half8 af[2][FM][kPer];  // operands of a step, read a step ahead within a chunk
    auto read_lhs = [&](int chunk, int step, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < FM; a++)
#pragma unroll
            for (int q = 0; q < kPer; q++) af[slot][a][q] = *(const half8*)(bufs + chunk % kLhsBuffers * kBuf + ((a * kChunk + step) * kPer + q) * 1024 + l16);
    };
    if (u0 < u1) {
        load_lhs(0);
        if constexpr (ENC == QMM_GPTQ) w.load_first(u0);
        else w.load(u0);
        store_lhs(0);
        load_lhs(1);
    }
    if (threadIdx.x < 32 * FM) inv[threadIdx.x] = p.inv[min(m0 + (int)threadIdx.x, m - 1)];
    for (int it = 0; it < walk; it++) {
        const int u = u0 + it;
        if (u >= u1) {  // (a shorter part)
#pragma unroll
            for (int c = 0; c < kChunks; c++) __syncthreads();
            continue;
        }
        const bool more = u + 1 < u1;
        w.open();
        if (more) w.load(u + 1);
        half8 sf[FM];
        auto load_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int a = 0; a < FM; a++)
                sf[a] = *(const half8*)((const uint8_t*)p.sums + ((int64_t)min(tile_m * FM + a, last_tile) * units + u) * 1024 + l16);
        };
        if constexpr (ENC == QMM_Q4_0) load_sums();
        float16v P[FM], U[kUnit ? FM : 1], M[W::kMin ? FM : 1];
        half8 b[2][W::kPlanes];
        float offset_unit = 0.0f;
        w.template step<0>(0, b[0]);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<W::kSteps>([&](auto tt) __attribute__((always_inline)) {
            constexpr int t = decltype(tt)::value, chunk = t / kChunk, in = t % kChunk, cur = t & 1;
            constexpr int kMfma = FM * kPer * W::kPlanes + (W::kMin && t == kOffsetsAt ? (CENTER ? 2 : 1) * FM : 0);
            if constexpr (in == 0) {
                __syncthreads();  // this chunk has arrived, the one before it is used up
                store_lhs((chunk + 1) % kLhsBuffers);
                load_lhs(it * kChunks + chunk + 2);
                read_lhs(chunk, 0, cur);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (in + 1 < kChunk) read_lhs(chunk, in + 1, cur ^ 1);
            if constexpr (W::kMin && t == kSumsAt) load_sums();
            if constexpr (W::kMin && t == kOffsetsAt) {
                const half8 first = CENTER ? w.offsets_lo() : w.min_operand(0);
#pragma unroll
                for (int a = 0; a < FM; a++) M[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[a], first, zero16, 0, 0, 0);
                if constexpr (CENTER)
#pragma unroll
                    for (int a = 0; a < FM; a++) M[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[a], w.offsets_hi(), M[a], 0, 0, 0);
            }
#pragma unroll
            for (int pl = 0; pl < W::kPlanes; pl++)
#pragma unroll
                for (int q = 0; q < kPer; q++)
#pragma unroll
                    for (int a = 0; a < FM; a++) {
                        if (t % W::kFlush == 0 && pl == 0 && q == 0) P[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[cur][a][q], b[cur][pl], zero16, 0, 0, 0);
                        else P[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[cur][a][q], b[cur][pl], P[a], 0, 0, 0);
                    }
            if constexpr (W::kMin && CENTER && t >= kOffsetsAt - 5 && t < kOffsetsAt) {
                if constexpr (t == kOffsetsAt - 5) offset_unit = w.open_offsets();
                else w.template add_offsets<t - (kOffsetsAt - 4)>();
            }
            if constexpr (t + 1 < W::kSteps) {
                w.template before_step<t>();
                w.template step<t + 1>(0, b[cur ^ 1]);
            }
            if (more) {
                if constexpr (t > 0) w.template after_step<t - 1>(u + 1);
                if constexpr (t + 1 == W::kSteps) w.template after_step<t>(u + 1);
            }
            if constexpr (in + 1 < kChunk) __builtin_amdgcn_sched_group_barrier(0x100, FM * kPer, 0);  // the next operands first, then the weights in between
            unrolled<kMfma>([&](auto) __attribute__((always_inline)) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, (W::kPlanes == 2 ? 28 : W::kMin ? 17 : 11) / kMfma + 1, 0);
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (t % W::kFlush == W::kFlush - 1) {
                if constexpr (ENC == QMM_Q4_0) {
                    const half8 dw = w.template scale_operand<t / 2>(0);
#pragma unroll
                    for (int a = 0; a < FM; a++) {
                        const float16v S = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[a], dw, zero16, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            U[a][r] = t < W::kFlush ? P[a][r] * S[r] : fmaf(P[a][r], S[r], U[a][r]);
                            if constexpr (t + 1 == W::kSteps) T[a][r] += U[a][r];
                        }
                        asm volatile("" : "+v"(U[a]));
                    }
                } else {
                    float d = 0.0f;
                    if constexpr (ENC == QMM_GPTQ) d = w.template scale_at<t / W::kFlush>(0);
                    else d = w.scale(0);
                    const float per_unit = CENTER ? w.scale_per_unit() : 0.0f, dmin = w.min_scale(0);
#pragma unroll
                    for (int a = 0; a < FM; a++) {
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            if constexpr (kUnit) U[a][r] = t < W::kFlush ? d * P[a][r] : fmaf(d, P[a][r], U[a][r]);
                            else if constexpr (W::kMin && CENTER) T[a][r] = fmaf(offset_unit, fmaf(per_unit, P[a][r], M[a][r]), T[a][r]);
                            else if constexpr (W::kMin) T[a][r] = fmaf(dmin, M[a][r], fmaf(d, P[a][r], T[a][r]));
                            else T[a][r] = fmaf(d, P[a][r], T[a][r]);
                            if constexpr (kUnit && t + 1 == W::kSteps) T[a][r] += U[a][r];
                        }
                        if constexpr (kUnit) asm volatile("" : "+v"(U[a]));
                        else asm volatile("" : "+v"(T[a]));
                    }
                }
            }
        });
    }
    __syncthreads();  // (the lhs buffers are used up; inv has arrived where there was no unit)

    // Two parts of K: each of the two wavefronts of a column group takes half of the rows and adds what the other has for them.
    constexpr int kOwn = FM / WK;
    if constexpr (WK == 2) {
        float4* const red = (float4*)smem + wn * FM * 256;
#pragma unroll
        for (int a = 0; a < FM; a++)
            if (a / kOwn != wk)
#pragma unroll
                for (int j = 0; j < 4; j++) red[a * 256 + j * 64 + lane] = make_float4(T[a][4 * j], T[a][4 * j + 1], T[a][4 * j + 2], T[a][4 * j + 3]);
        __syncthreads();
#pragma unroll
        for (int a = 0; a < FM; a++)
            if (a / kOwn == wk)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 x = red[a * 256 + j * 64 + lane];
                    T[a][4 * j] += x.x; T[a][4 * j + 1] += x.y; T[a][4 * j + 2] += x.z; T[a][4 * j + 3] += x.w;
                }
    }
    const int col = n0 + (lane & 31), g = lane >> 5;
    if (col >= wt.n) return;
    // (the kind of result chosen once, not at each value)
    auto each = [&](auto&& store) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < FM; a++) {
            if (WK == 2 && a / kOwn != wk) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4 s = *(const float4*)(inv + 32 * a + 8 * j + 4 * g);
                const float sv[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = m0 + 32 * a + 8 * j + 4 * g + r;
                    if (row < m) store((int64_t)row * wt.n + col, T[a][4 * j + r] * sv[r]);
                }
            }
        }
    };
    if (shares > 1) each([&](int64_t at, float x) __attribute__((always_inline)) { unsafeAtomicAdd(out + at, x); });
    else if (out16) each([&](int64_t at, float x) __attribute__((always_inline)) { out16[at] = f2bf(x); });
    else each([&](int64_t at, float x) __attribute__((always_inline)) { out[at] = x; });
}

template <int ENC, int FLUSH, int FM, int WN, int WK, bool HILO, bool CENTER>
hipError_t run_shared(const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units, int shares, hipStream_t s) {
    using W = WeightsOf<ENC, 1, FLUSH, CENTER>;
    constexpr int kBuf = FM * 8 * 1024;
    constexpr int lds = WK * kLhsBuffers * kBuf + WN * WK * W::kStage + 32 * FM * 4;
    static_assert(WK == 1 || WN * FM * 4096 <= lds - 32 * FM * 4, "the partial results fit in front of the row scales");
    static_assert(lds <= kLdsPerCu, "fits a compute unit");
    const int tiles_m = (int)((m + 32 * FM - 1) / (32 * FM));
    int eights = 0;
    for (int j = 0; j < mats.count; j++) mats.end[j] = eights += (mats.n[j] + 256 * WN - 1) / (256 * WN);
    hipError_t e = allow_full_lds<gemm_shared_kernel<ENC, FLUSH, FM, WN, WK, HILO, CENTER>>();
    if (e != hipSuccess) return e;
    const DirectGrid g = direct_grid(tiles_m, eights * shares);
    gemm_shared_kernel<ENC, FLUSH, FM, WN, WK, HILO, CENTER><<<g.grid, dim3(64 * WN * WK), lds, s>>>(mats.w[0], p.a16, mats.n[0], (int)m, units, g.tiles_m, shares, mats.count, wt, mats, p, out16);
    return hipGetLastError();
}

template <int ENC, int FLUSH, bool HILO, bool CENTER = false>
hipError_t run_shared_plan(const DirectPlan& pl, const WeightTensors& wt, const DirectMats& mats, const DirectSpace& p, uint16_t* out16, int64_t m, int units,
                           hipStream_t s) {
#define QMM_GS(FM, WN, WK) \
    if (pl.fm == FM && pl.wn == WN && pl.wk == WK) return run_shared<ENC, FLUSH, FM, WN, WK, HILO, CENTER>(wt, mats, p, out16, m, units, pl.shares, s)
    QMM_GS(2, 8, 1);
    QMM_GS(2, 4, 2);
    QMM_GS(2, 4, 1);
#undef QMM_GS
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm_shared(int encoding, bool hilo, const DirectPlan& pl, const WeightTensors& wt, DirectMats mats, const DirectSpace& p, uint16_t* out16,
                              int64_t m, int units, hipStream_t s) {
    const bool few = m <= kFewSharedRows;
#define QMM_GS_RUN(...) return run_shared_plan<__VA_ARGS__>(pl, wt, mats, p, out16, m, units, s)
#define QMM_GS_ENC(ENC, FLUSH)                \
    do {                                      \
        if (hilo) QMM_GS_RUN(ENC, FLUSH, true); \
        QMM_GS_RUN(ENC, FLUSH, false);        \
    } while (0)
    switch (encoding) {
        case QMM_Q4_0: QMM_GS_RUN(QMM_Q4_0, 2, false);
        case QMM_Q4_K:
            if (hilo) QMM_GS_RUN(QMM_Q4_K, 16, true, true);
            QMM_GS_RUN(QMM_Q4_K, 16, false);
        case QMM_Q5_K:
            if (hilo) QMM_GS_RUN(QMM_Q5_K, 16, true, true);
            if (few) QMM_GS_RUN(QMM_Q5_K, 16, false, true);
            QMM_GS_RUN(QMM_Q5_K, 16, false);
        case QMM_Q6_K:
            if (few) QMM_GS_ENC(QMM_Q6_K, 8);
            QMM_GS_ENC(QMM_Q6_K, 16);
        case QMM_GPTQ:
            if (wt.group % 128 == 0) QMM_GS_ENC(QMM_GPTQ, 8);
            QMM_GS_ENC(QMM_GPTQ, 2);
        default: return hipErrorInvalidValue;
    }
#undef QMM_GS_RUN
#undef QMM_GS_ENC
}

}  // namespace qmm
