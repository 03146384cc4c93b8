// GPTQ with a few lhs rows (1 .. 16 bf16, 1 .. 8 fp32 a workgroup, up to four times as many side by side) on the matrix cores, K any multiple of 256, groups of 32, 64, 128 or 256: one launch, no workspace needed.
//
// Shape of the work: that of gemv_kquant_small.hip.  A workgroup has as many wavefronts, up to 16, as divide the 256-column parts of K evenly into groups; a wavefront keeps the lhs operands
// of its part in 32 registers and walks the workgroup's tiles of CW output columns with them.  An item, 32 rows of CW words and the scales and zeros over them (2.2 or 4.3 KB), goes
// global -> LDS directly into a private ring of two slots, one item ahead of the one being multiplied.
//
// What bounds it: the way to the first product (launch, lhs from L2 and its conversion, some 4 us with up to four rows, 6 with sixteen), then memory, 4.5 TB/s at 14336 x 4096 (vector
// instructions issued in half of a wavefront's life, waiting 0.43 .. 0.46 of it).  The tensor lies
// K row by K row, so a tile is 64 or 128 bytes of every row: 32 columns fill the cache lines, 16 leave it to the L2 of the XCD that neighbouring tiles share.  The kernels before had the loads of
// one group per wavefront in flight, held in registers, and a workgroup per 64 (one row: 16) columns: figures at the dispatch (qmm_api.hip).
//
// Arithmetic.  lhs: see small_narrow.  A word holds eight k of one column, what a lane supplies of the B operand of v_mfma_f32_16x16x32_f16: a masked nibble is the subnormal q * 2^-24 (or
// 16 q * 2^-24), one packed multiply-add leaves (q - zero) * 2^-14, so every product is exact; per group  acc += scale * 2^14 * P.

#include <algorithm>
#include <type_traits>

#include "small_lhs.h"

namespace qmm {

namespace {

constexpr int kGsWaves = 16;

// CW: columns of a tile.  GS: steps of 32 k in a group.  Words of an item: 16-byte pieces, row by row; behind them its scales, then its zeros, a dword per lane.
template <int CW, int GS>
struct GptqItem {
    static constexpr int kGroups = 8 / GS, kScales = kGroups * CW / 2, kDwords = kScales + kGroups * CW / 8;
    static constexpr int kWordLoads = CW / 8, kParamLoads = (kDwords + 63) / 64, kLoads = kWordLoads + kParamLoads;
    static constexpr int kWords = kWordLoads * 1024, kSlot = kWords + kParamLoads * 256;
};

struct GptqSmallCut {
    int per, stride;           // tiles of a workgroup at most, workgroups across the tiles
    int waves, groups, chunk;  // wavefronts; groups of K; items whose partial results fit LDS together
    bool apart, bf16;          // a group of K per workgroup; bf16 results
    uint32_t packed() const { return (uint32_t)waves | (uint32_t)chunk << 8 | (uint32_t)apart << 16 | (uint32_t)bf16 << 17 | (uint32_t)groups << 18; }
};

}  // namespace

template <int CW, int GS, int MROWS, typename AT>
__global__ __launch_bounds__(64 * kGsWaves) void gemv_gptq_small_kernel(const uint32_t* __restrict__ qweight, const uint16_t* __restrict__ scales, const uint32_t* __restrict__ qzeros,
                                                                       const AT* __restrict__ a, int n, int m, int k, int stride, int per, uint32_t packed, float* __restrict__ out) {
    using I = GptqItem<CW, GS>;
    constexpr int PL = sizeof(AT) == 4 ? 2 : 1, LR = MROWS <= 4 ? 1 : MROWS / 4, RN = LR * PL, kPass = std::min(MROWS, 4 / PL), H = CW / 16;
    static_assert(RN <= 4, "operand rows");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nn = lane & 15, kg = lane >> 4;
    const int waves = (int)(packed & 0xffu), chunk = (int)(packed >> 8) & 0xff, groups = (int)(packed >> 18) & 0x1fff;
    const bool apart = (packed >> 16) & 1, bf16 = (packed >> 17) & 1;
    // Neighbouring tiles run on one XCD (ids congruent mod 8), whose L2 then fetches the lines that they share once.
    int share, of_k = (int)blockIdx.y, row0 = 0;  // this workgroup's tiles, group of K, first lhs row
    if (MROWS == small_rows<AT>() && (packed >> 31)) {
        // several tiles of lhs rows: those that read the same weights side by side (blockIdx.y) on one XCD, every XCD the same number of them
        row0 = (int)blockIdx.y * MROWS, share = (int)blockIdx.x * ((stride * (apart ? groups : 1) + 7) >> 3) + (int)blockIdx.z, of_k = apart ? share / stride : 0;
        share -= of_k * stride;
        if (apart && of_k >= groups) return;
    } else share = ((int)blockIdx.x & 7) * ((stride + 7) >> 3) + ((int)blockIdx.x >> 3);
    if (share >= stride) return;  // (the whole workgroup)
    const int parts = k >> 8;
    const int g_first = apart ? of_k : 0, g_end = apart ? g_first + 1 : groups;
    uint8_t* const ring = smem + wave * (2 * I::kSlot);
    const uint32_t ring_lds = lds_address(ring);
    float* const accs = (float*)(smem + waves * (2 * I::kSlot));  // [chunk][waves][H LR][64]
    float* const totals = accs + chunk * waves * (H * LR) * 64;    // [chunk][H LR][64], with more than one group
    const int ntiles = (n + CW - 1) / CW, my_items = share + (per - 1) * stride < ntiles ? per : per - 1;

    // (the last tile ends with the matrix and may share columns with the one before)
    auto first_column = [&](int item) __attribute__((always_inline)) { return min((share + item * stride) * CW, n - CW); };
    constexpr int kPieces = CW / 4, kRows = 64 / kPieces;  // 16-byte pieces of a row of words; rows of a load
    const uint32_t word_lane = (uint32_t)(lane / kPieces) * (uint32_t)n * 4u + 16u * (uint32_t)(lane % kPieces);
    auto issue = [&](int part, int item, int slot) __attribute__((always_inline)) {
        const int n0 = first_column(item);
        const uint8_t* const words = (const uint8_t*)(qweight + (int64_t)(32 * part) * n + n0);
#pragma unroll
        for (int i = 0; i < I::kWordLoads; i++) small_stream16<CW == 32>(word_lane, words + (int64_t)(i * kRows) * n * 4, ring_lds + slot * I::kSlot + i * 1024);
        const uint8_t* const sc = (const uint8_t*)(scales + (int64_t)(part * I::kGroups) * n + n0);
        const uint8_t* const zr = (const uint8_t*)(qzeros + (int64_t)(part * I::kGroups) * (n >> 3) + (n0 >> 3));
#pragma unroll
        for (int j = 0; j < I::kParamLoads; j++) {
            const int d = min(lane + 64 * j, I::kDwords - 1), e = d - I::kScales;
            const uint8_t* const at = d < I::kScales ? sc + (uint32_t)(d / (CW / 2)) * (uint32_t)n * 2u + 4u * (uint32_t)(d % (CW / 2))
                                                     : zr + (uint32_t)(e / (CW / 8)) * (uint32_t)(n >> 1) + 4u * (uint32_t)(e % (CW / 8));
            load4_to_lds(at, ring_lds + slot * I::kSlot + I::kWords + j * 256);
        }
    };

    // lhs operands of the wavefront's part: operand row nn is lhs row nn / 4 + 4 j, hi part or (fp32) residual, j and part by nn % 4; fragment s of lane quarter kg holds columns
    // 32 s + 8 kg + (0,4,1,5,2,6,3,7)
    half8 fa[8];
    float bs[LR];  // inverse lhs scales of this lane's results
#pragma unroll
    for (int s = 0; s < 8; s++) fa[s] = pack4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int j = 0; j < LR; j++) bs[j] = 0.0f;
    typedef typename std::conditional<sizeof(AT) == 4, u32x4, u32x2>::type xraw_t;
    auto narrow = [&](const xraw_t (&xr)[MROWS], uint8_t* area) __attribute__((always_inline)) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));  // (what is computed from it here is not kept in registers between the groups)
        const int nn = lane & 15, kg = lane >> 4, my_row = (nn >> 2) + 4 * ((nn & 3) / PL), my_part = (nn & 3) % PL;
        float* const row_scales = (float*)(area + 4 * kSmallPlane);
        float common = 1.0f;
        if constexpr (PL == 2) common = small_common_scale<14>(xr);
#pragma unroll
        for (int r0 = 0; r0 < MROWS; r0 += kPass) {
            const float inverse = small_narrow<PL, kPass, kSmallOrderGptq, 14>(xr, r0, common, area, row_scales, lane);
            __builtin_amdgcn_wave_barrier();
            if ((nn & 3) < RN && my_row >= r0 && my_row < r0 + kPass) {
                const uint8_t* const pl = area + ((my_row - r0) * PL + my_part) * kSmallPlane + 16 * kg;
#pragma unroll
                for (int s = 0; s < 8; s++) fa[s] = *(const half8*)(pl + 64 * s);
            }
#pragma unroll
            for (int j = 0; j < LR; j++)
                if (kg + 4 * j >= r0 && kg + 4 * j < r0 + kPass) bs[j] = inverse == 0.0f ? row_scales[kg + 4 * j - r0] : inverse;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the operands are in registers before the next item's load may overwrite the slot
    };
    const uint32_t a_lane = 4 * (uint32_t)sizeof(AT) * lane;

    int slot = 0;
    {
        xraw_t xr[MROWS];
        const int part = min(g_first * waves + wave, parts - 1);
#pragma unroll
        for (int j = 0; j < MROWS; j++) hidden_load(xr[j], a_lane, a + (int64_t)min(row0 + j, m - 1) * k + part * 256);
        issue(part, 0, 0);
        wait_vmcnt<I::kLoads>();
#pragma unroll
        for (int j = 0; j < MROWS; j++) tie(xr[j]);
        narrow(xr, ring + I::kSlot);
    }
    const ks_float4 zero4 = {0.f, 0.f, 0.f, 0.f};

    int held = g_first;  // the group whose lhs operands are in the registers
    for (int c0 = 0; c0 < my_items; c0 += chunk) {
        const int ct = min(chunk, my_items - c0);
        for (int g = g_first; g < g_end; g++) {
            const int part = g * waves + wave;
            if (part < parts) {  // (all wavefronts but for the last group)
                if (g != held) {
                    held = g;
                    xraw_t xr[MROWS];
#pragma unroll
                    for (int j = 0; j < MROWS; j++) xr[j] = *(const xraw_t*)((const uint8_t*)(a + (int64_t)min(row0 + j, m - 1) * k + part * 256) + a_lane);
                    narrow(xr, ring + (slot ^ 1) * I::kSlot);
                }
                for (int t = 0; t < ct; t++) {
                    // the next item: of the chunk, of the next group, of the next chunk
                    int ng = g, nt = c0 + t + 1;
                    if (t + 1 == ct) {
                        ng = g + 1, nt = c0;
                        if (ng == g_end || part + waves >= parts) ng = g_first, nt = c0 + ct;
                    }
                    if (nt < my_items) {
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (what was read from that slot is in registers)
                        issue(ng * waves + wave, nt, slot ^ 1);
                        wait_vmcnt<I::kLoads>();
                    } else {
                        wait_vmcnt<0>();
                    }
                    // lane (nn, kg) holds column n0 + H nn + h
                    const uint8_t* const item = ring + slot * I::kSlot;
                    const uint32_t* const sc = (const uint32_t*)(item + I::kWords);
                    float v[H][LR];
#pragma unroll
                    for (int h = 0; h < H; h++)
#pragma unroll
                        for (int j = 0; j < LR; j++) v[h][j] = 0.0f;
#pragma unroll
                    for (int gi = 0; gi < I::kGroups; gi++) {
                        const int c = H * nn;
                        const uint32_t s2 = CW == 32 ? sc[gi * 16 + nn] : ((const uint16_t*)sc)[gi * 16 + nn];
                        const uint32_t z2 = sc[I::kScales + gi * (CW / 8) + (c >> 3)] >> (4 * (c & 7));
                        ks_float4 P[H];
                        uint32_t nz[H];
#pragma unroll
                        for (int h = 0; h < H; h++) {
                            const float z = (float)(((z2 >> (4 * h)) & 0xFu) + 1u) * -6.103515625e-05f;  // -zero * 2^-14
                            nz[h] = to_half2_bits(z, z);
                            P[h] = zero4;
                        }
#pragma unroll
                        for (int s = gi * GS; s < gi * GS + GS; s++) {
                            uint32_t w[H];
                            if constexpr (H == 2) {
                                const uint2 pair = *(const uint2*)(item + s * 512 + 8 * lane);
                                w[0] = pair.x, w[1] = pair.y;
                            } else {
                                w[0] = *(const uint32_t*)(item + s * 256 + 4 * lane);
                            }
#pragma unroll
                            for (int h = 0; h < H; h++) {
                                constexpr uint32_t M1 = 0x000F000Fu, M2 = 0x00F000F0u, kLow = 0x64006400u, kHigh = 0x54005400u;  // 2^10, 2^6
                                const uint32_t y = w[h] >> 8;
                                const half8 b = pack4(pk_fma(w[h] & M1, kLow, nz[h]), pk_fma(w[h] & M2, kHigh, nz[h]), pk_fma(y & M1, kLow, nz[h]), pk_fma(y & M2, kHigh, nz[h]));
                                P[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[s], b, P[h], 0, 0, 0);
                            }
                        }
#pragma unroll
                        for (int h = 0; h < H; h++) {
                            const float scale = h2f((uint16_t)(s2 >> (16 * h))) * 16384.0f;
#pragma unroll
                            for (int j = 0; j < LR; j++) v[h][j] = fmaf(scale, PL == 2 ? P[h][PL * j] + P[h][PL * j + PL - 1] : P[h][j], v[h][j]);
                        }
                    }
                    float* const mine = accs + ((t * waves + wave) * (H * LR)) * 64 + lane;
#pragma unroll
                    for (int h = 0; h < H; h++)
#pragma unroll
                        for (int j = 0; j < LR; j++) mine[(h * LR + j) * 64] = bs[j] * v[h][j];
                    slot ^= 1;
                }
            }
            __syncthreads();
            // the group's result (lhs row kg + 4 j, column n0 + H nn + h): dealt to the wavefronts, which add it to that of the groups before
            const int live = min(waves, parts - g * waves);
            for (int q = wave; q < ct * (H * LR); q += waves) {
                const int t = q / (H * LR), hj = q % (H * LR), h = hj / LR, row = row0 + kg + 4 * (hj % LR);
                const float* const src = accs + ((t * waves) * (H * LR) + hj) * 64 + lane;
                float c[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                int w = 0;
                for (; w + 4 <= live; w += 4)
#pragma unroll
                    for (int i = 0; i < 4; i++) c[i] += src[(w + i) * (H * LR) * 64];
#pragma unroll
                for (int i = 0; i < 3; i++)
                    if (w + i < live) c[i] += src[(w + i) * (H * LR) * 64];
                float r = (c[0] + c[1]) + (c[2] + c[3]);
                if (groups > 1) {
                    float* const total = totals + (t * (H * LR) + hj) * 64 + lane;
                    if (g > g_first) r = *total + r;
                    if (g + 1 < g_end) *total = r;
                }
                if (g + 1 < g_end || row >= m) continue;
                const int64_t at = (int64_t)row * n + first_column(c0 + t) + H * nn + h;
                if (bf16) ((uint16_t*)out)[at] = f2bf(r);
                else out[at + (int64_t)of_k * m * n] = r;
            }
            if (g + 1 < g_end || c0 + chunk < my_items) __syncthreads();
        }
    }
}

namespace {

struct GptqSmallPlan {
    GptqSmallCut cut;
    int cw, grid, parts, per_cu, row_tiles;
    size_t lds;
};
// Groups of K: of its length only, so that results do not depend on what else a call has.
int gptq_small_groups(int64_t k) {
    const int groups = (int)((k / 256 + kGsWaves - 1) / kGsWaves);
    return groups == 3 ? 4 : groups;
}
int gptq_small_slot(int cw, int group) {
    const int dwords = 256 / group * (cw / 2 + cw / 8);
    return cw * 128 + (dwords + 63) / 64 * 256;
}
// apart: workgroups that share a tile, one group of K each
bool gptq_small_cut(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, bool apart, int cw, GptqSmallPlan& p) {
    p.row_tiles = (int)((m + small_most_rows(lhs_dtype) - 1) / small_most_rows(lhs_dtype));
    m = std::min(m, small_most_rows(lhs_dtype));
    const int parts = (int)(k / 256), groups = gptq_small_groups(k), lr = m <= 4 ? 1 : m <= 8 ? 2 : 4;
    if (n < cw) return false;
    GptqSmallCut& c = p.cut;
    p.cw = cw;
    c.groups = groups;
    c.waves = (parts + groups - 1) / groups;
    c.apart = apart;
    p.parts = apart ? groups : 1;
    const int64_t tiles = (n + cw - 1) / cw;
    p.per_cu = std::max(1, kGsWaves / c.waves);
    const int64_t most = std::max<int64_t>(1, small_places(p.per_cu, p.row_tiles) / p.parts);
    c.per = (int)((tiles + most - 1) / most);
    c.stride = (int)((tiles + c.per - 1) / c.per);
    p.grid = (c.stride + 7) / 8 * 8;
    const int ring = c.waves * 2 * gptq_small_slot(cw, group), each = (c.waves + (groups > p.parts ? 1 : 0)) * lr * (cw / 16) * 256;
    c.chunk = std::min(std::min(c.per, 254), (kLdsPerCu / p.per_cu - ring) / each);
    p.lds = (size_t)ring + (size_t)std::max(c.chunk, 0) * each;
    return c.chunk > 0;
}
// Tiles of 16 or 32 columns, groups of K walked in a workgroup or a workgroup for each: the lowest of fitted costs (what differs between the four).  us per conversion of the lhs
// of a group of K, per item of 16 wavefronts with 16 and with 32 columns, by rows; 19 matrices of 1024 x 1024 .. 128256 x 4096, groups of 128, weights from memory: what it picks takes 0.3 .. 2.5 % longer
// on average than the best of the four.
// Groups side by side only below 2^27 weights (8192 x 28672 one row 27.4 us walked, 31 apart, 8 fp32 rows 45 and 52).  32 columns: whole cache lines, 14336 x 4096 4 bf16 rows 9.0 against
// 11.3 us; 16 columns where that spreads the matrix more evenly over the part, 4096 x 4096 5.5 against 6.0, and always with nine rows and more, whose results do not fit LDS next to the
// larger ring.
struct GptqSmallCost {
    float convert, item[2];
};
constexpr GptqSmallCost kGptqSmallCost[2][4] = {
    // rows up to 2, 4, 8, 16
    {{1.16f, {1.19f, 1.57f}}, {1.38f, {1.14f, 1.49f}}, {2.07f, {0.94f, 1.37f}}, {4.2f, {0.5f, 0.0f}}},  // bf16
    {{0.96f, {1.25f, 1.67f}}, {2.03f, {1.0f, 1.31f}}, {3.3f, {0.5f, 0.8f}}, {}},                        // fp32
};
bool gptq_small_plan(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group, bool may_part, GptqSmallPlan& best) {
    const GptqSmallCost& cost = kGptqSmallCost[lhs_dtype == QMM_F32 ? 1 : 0][m <= 2 ? 0 : m <= 4 ? 1 : m <= 8 || lhs_dtype == QMM_F32 ? 2 : 3];
    const int groups = gptq_small_groups(k);
    double us = 1e30;
    for (int apart = 0; apart <= (may_part && groups > 1 && n * k < (int64_t)1 << 27 ? 1 : 0); apart++)
        for (int cw = 16; cw <= (m <= 8 || lhs_dtype == QMM_F32 ? 32 : 16); cw += 16) {
            GptqSmallPlan p;
            if (!gptq_small_cut(lhs_dtype, m, n, k, group, apart != 0, cw, p)) continue;
            const int walk = apart ? 1 : groups, chunks = (p.cut.per + p.cut.chunk - 1) / p.cut.chunk, workgroups = (int)(((int64_t)p.cut.stride * p.parts * p.row_tiles + compute_units() - 1) / compute_units());
            const double t = cost.convert * ((walk > 1 ? walk * chunks : 1) + 0.3 * (workgroups - 1)) + cost.item[cw / 16 - 1] * p.cut.per * walk * p.cut.waves * p.per_cu / kGsWaves +
                             0.15 * (chunks * walk - 1) + 2.8 * apart;
            if (t < us) us = t, best = p;
        }
    return us < 1e29;
}

template <int CW, int GS, int MROWS, typename AT>
hipError_t run_gptq_small(const GptqSmallPlan& p, const uint32_t* qweight, const uint16_t* scales, const uint32_t* qzeros, const AT* a, float* out, int n, int m, int k, hipStream_t s) {
    hipError_t e = allow_full_lds<gemv_gptq_small_kernel<CW, GS, MROWS, AT>>();
    if (e != hipSuccess) return e;
    const dim3 grid = p.row_tiles > 1 ? dim3(8, (unsigned)p.row_tiles, (unsigned)((p.cut.stride * p.parts + 7) / 8)) : dim3((unsigned)p.grid, (unsigned)p.parts);
    gemv_gptq_small_kernel<CW, GS, MROWS, AT><<<grid, dim3((unsigned)(64 * p.cut.waves)), p.lds, s>>>(qweight, scales, qzeros, a, n, m, k, p.cut.stride, p.cut.per, p.cut.packed() | (uint32_t)(p.row_tiles > 1) << 31, out);
    return hipGetLastError();
}

template <int CW, int GS>
hipError_t run_gptq_small_rows(const GptqSmallPlan& p, const uint32_t* qweight, const uint16_t* scales, const uint32_t* qzeros, const void* a, int lhs_dtype, float* out, int n, int m, int k,
                               hipStream_t s) {
    if (lhs_dtype == QMM_F32) {
        const float* const f = (const float*)a;
        if (m == 1) return run_gptq_small<CW, GS, 1>(p, qweight, scales, qzeros, f, out, n, m, k, s);
        if (m == 2) return run_gptq_small<CW, GS, 2>(p, qweight, scales, qzeros, f, out, n, m, k, s);
        if (m <= 4) return run_gptq_small<CW, GS, 4>(p, qweight, scales, qzeros, f, out, n, m, k, s);
        return run_gptq_small<CW, GS, 8>(p, qweight, scales, qzeros, f, out, n, m, k, s);
    }
    const uint16_t* const b = (const uint16_t*)a;
    if (m == 1) return run_gptq_small<CW, GS, 1>(p, qweight, scales, qzeros, b, out, n, m, k, s);
    if (m == 2) return run_gptq_small<CW, GS, 2>(p, qweight, scales, qzeros, b, out, n, m, k, s);
    if (m <= 4) return run_gptq_small<CW, GS, 4>(p, qweight, scales, qzeros, b, out, n, m, k, s);
    if (m <= 8 || CW > 16) return run_gptq_small<CW, GS, 8>(p, qweight, scales, qzeros, b, out, n, m, k, s);  // (more rows come with 16 columns only)
    return run_gptq_small<CW, GS, (CW > 16 ? 8 : 16)>(p, qweight, scales, qzeros, b, out, n, m, k, s);
}

}  // namespace

bool gemv_gptq_small_supported(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    // (with the name of the older small-batch kernel this one goes too)
    if (kernel_disabled("gptq_small") || kernel_disabled("gptq_mm") || (group != 32 && group != 64 && group != 128 && group != 256)) return false;
    if (m < 1 || m > 4 * small_most_rows(lhs_dtype) || n < 16 || n % 8 || n > 1 << 23 || k < 256 || k % 256 || k > 1 << 20) return false;
    // Nine rows and more, us, older small-batch kernel / this one: two workgroups on a compute unit convert the lhs twice, 5632 x 2048 7.3 / 8.6, 8192 x 1024 5.6 / 6.1; large matrices with several groups of
    // K, few results in LDS at a time, 28672 x 8192 38 / 45; but 2048 x 2048 6.7 / 6.0, 8192 x 8192 17.7 / 16.1.
    // One row, groups of 32, whose scales and zeros leave the larger ring no room: 28672 x 8192 33 .. 36 / 38, but 14336 x 4096 15.2 / 11.5.
    if (m == 1 && group == 32 && k > 4096 && n * k >= (int64_t)1 << 27) return false;
    return m <= 8 || lhs_dtype == QMM_F32 || ((k > 2048 || n <= 16 * compute_units()) && (k <= 4096 || n * k < (int64_t)1 << 27));
}

// What groups of K side by side take (without it a workgroup walks all of K: the same sums).
int64_t gemv_gptq_small_workspace_bytes(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    GptqSmallPlan p;
    return gptq_small_groups(k) > 1 && gptq_small_plan(lhs_dtype, m, n, k, group, true, p) && p.cut.apart ? p.parts * m * n * 4 : 0;
}

// The caller has asked gemv_gptq_small_supported.  out_bf16: `out` is a bf16 array.  workspace: null, or gemv_gptq_small_workspace_bytes.
hipError_t launch_gemv_gptq_small(const void* a, int lhs_dtype, const uint32_t* qweight, const uint16_t* scales, const uint32_t* qzeros, int64_t m, int64_t n, int64_t k, int group, float* out,
                                  bool out_bf16, void* workspace, hipStream_t s) {
    GptqSmallPlan p;
    if (!gptq_small_plan(lhs_dtype, m, n, k, group, workspace != nullptr, p)) return hipErrorInvalidValue;
    const bool apart = p.cut.apart;
    p.cut.bf16 = out_bf16 && !apart;
    float* const to = apart ? (float*)workspace : out;
#define QMM_GS(CW, GS) run_gptq_small_rows<CW, GS>(p, qweight, scales, qzeros, a, lhs_dtype, to, (int)n, (int)m, (int)k, s)
#define QMM_GS_GROUP(CW) (group == 32 ? QMM_GS(CW, 1) : group == 64 ? QMM_GS(CW, 2) : group == 128 ? QMM_GS(CW, 4) : QMM_GS(CW, 8))
    hipError_t e = p.cw == 32 ? QMM_GS_GROUP(32) : QMM_GS_GROUP(16);
#undef QMM_GS_GROUP
#undef QMM_GS
    if (e != hipSuccess || !apart) return e;
    return out_bf16 ? launch_sum_shares_bf16((const float*)workspace, (uint16_t*)out, m * n, p.parts, s) : launch_sum_shares((const float*)workspace, out, m * n, p.parts, s);
}

}  // namespace qmm
