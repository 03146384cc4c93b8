// Q4_0, Q4_K, Q5_K and Q6_K with a few lhs rows (1 .. 16 bf16, 1 .. 8 fp32 a workgroup, up to four times as many side by side) on the matrix cores, K any multiple of 256: one launch, no workspace (groups of K side
// by side: a second launch and their sums in the workspace).
//
// Shape of the work.  A workgroup has as many wavefronts, up to 16, as divide the super-blocks of a row evenly into groups: wavefront w owns super-block
// w + waves g of group g (K = 4096: one group of 16; 14336: four of 14).  It converts the lhs columns of its super-block into matrix-core operands once a
// group, keeps them in 32 registers, and walks the workgroup's tiles of 16 weight rows with them.  The super-block of a tile's 16 rows (2.3 .. 3.8 KB) goes global -> LDS
// directly into a private ring of two slots, one item ahead of the one being multiplied: no wavefront waits for another before the end.  Partial results
// stay in LDS and are added in wavefront order, so their order depends on K only, not on N or on timing
// (the last bits of a row also on the rows beside it, whose values have a part in how it is scaled: small_lhs.h).
//
// Why 16 wavefronts with one super-block each (two before, eight wavefronts): an item is a chain LDS reads -> unpacking -> matrix cores of some 150 vector instructions, and with two
// wavefronts a SIMD most of it was waiting.  Why the rows of the lhs go where they go (row j to operand row 4 j mod 16, fp32 residuals in the rows between): a
// lane of the result holds operand rows 4 (lane / 16) + 0 .. 3, so with up to four rows every lane has one wanted result (two with fp32 residuals), and
// what is done to results (scales, sums, LDS) shrinks to a quarter.
//
// What bounds it: the way to the first product (launch, lhs from L2, conversion: some 4 us with four rows, 6 with sixteen), then memory (14336 x 4096, 4 bf16 rows: a tile of 16 rows, 37 .. 54 KB
// a compute unit, every 1.4 / 1.75 / 2.1 us).  Counters: vector instructions are issued in 0.57 .. 0.65 of a wavefront's life (403 of them in the 4.7 us of 4096 x 4096 with 4 fp32 rows, most for the lhs, and a SIMD's
// four wavefronts do it at the same time), 0.40 .. 0.46 of it is spent waiting, matrix cores are busy 0.09 .. 0.16.  us, the kernels before / this one, 14336 x 4096 4 bf16 rows, weights from memory: Q4_K 11.2 / 9.4, Q5_K 17.8 / 10.8, Q6_K 20.3 / 12.6; 16 bf16 rows
// 18.6 / 12.7, 17.5 / 13.9, 22.6 / 17.5; 4096 x 14336 4 fp32 rows 13.9 / 12.2, 22.7 / 13.9, 23.1 / 15.7; 2048 x 1024 4 bf16 rows 9.2 / 3.9.  Relative error, K = 4096, before / now: fp32 rows Q4_K
// 4.0e-7 / 1.1e-7, Q5_K 1.7e-7 / 1.2e-7, Q6_K 1.6e-7 / 1.0e-7; bf16 rows 2.5e-7 / 0.8e-7, 1.0e-7 / 0.85e-7, 0.97e-7 / 0.84e-7 (codes around their middle, residuals to nearest, super-blocks added in
// four chains).
//
// More rows than one workgroup takes: each streams all weights, the second one from its XCD's L2, which still beats preparing the lhs with a launch of its own where that launch and the next one's way to its first product
// are most of the time: 4096 x 4096 Q4_K 16 fp32 rows 11.7 / 9.2 us, 1024 x 14336 23.9 / 11.4 (rule and lines: qmm_api.hip).
//
// Arithmetic.  lhs: scaled by powers of two, then fp16 (see small_narrow; bf16 rows: one term; fp32 rows: hi part and residual, 22 bits).  Weights: integers sc * (q - mid) (Q4_K, Q5_K) or q (Q6_K) as fp16, so every product is exact and the sums are fp32.
//   Q4_K: a masked nibble is the subnormal q * 2^-24 (or 16 q * 2^-24), one packed multiply-add leaves sc * (q - 8) * 2^-18.
//   Q5_K: a byte permute puts nibble and fifth bit under 0x54: 64 + q; one packed multiply-add, (64 + q) * sc - 80 * sc, leaves sc * (q - 16) (exact: below 2^11).
//   Q6_K: the same with 96 taken off; sc * q may need 13 bits, so the scale multiplies the results of its 16 weights instead.
//   Q4_0 (an item is 16 rows x eight blocks): the lhs as Q8_0, quantised as any Q8_0 lhs here, int8 products of 16 (q - 8), whose sums over a block are exact; sum of (sum / 16) * (d_w d_a).
//   What codes around their middle leave out (Q4_K, Q5_K): mid * d * sc - dmin * mn times the sum of 32 lhs values, both as two fp16 terms, one more matrix product a super-block.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "small_lhs.h"

namespace qmm {

namespace {

constexpr int kSmallWaves = 16;

// The item of a wavefront: 16 rows of one super-block.  kRow: bytes of a row in LDS; Q6_K blocks lie at even addresses, loads to LDS want multiples of
// four: 212 bytes from the last such address on, the last 16 of them as a piece of their own (which overlaps the one before), and one piece of padding that
// spreads the rows over the banks.
template <int ENC>
struct SmallItem {
    static constexpr int kBpb = ENC == QMM_Q4_0 ? 8 * Q4_0_BPB : ENC == QMM_Q4_K ? Q4_K_BPB : ENC == QMM_Q5_K ? Q5_K_BPB : Q6_K_BPB;  // of 256 columns
    static constexpr int kRow = ENC == QMM_Q6_K ? 240 : kBpb, kRowPieces = kRow / 16, kPieces = 16 * kRowPieces, kLoads = (kPieces + 63) / 64, kSlot = 16 * kRow;
    static_assert(4 * kSmallPlane + 16 <= kSlot, "four planes of lhs rows and their scales fit a ring slot");
};

enum { kSmallPlain = 0, kSmallMats = 1, kSmallGated = 2, kSmallPairs = 3 };

}  // namespace

// MROWS: lhs rows of a workgroup, 1, 2, 4, 8 or 16 (rows past m repeat the last one and their results are dropped); more go side by side, in workgroups of their own.
// MODE: one matrix; several that share the lhs (their tiles numbered through); gate and up (result silu(gate) * up), eight rows of each in a tile, or a tile of gate and one of up after the other.
struct SmallCut {
    int per, stride;  // tiles (pairs of them) of a workgroup at most, workgroups across the tiles
    uint32_t packed;  // wavefronts; << 8: items (tile of a matrix, or of both) of a workgroup whose partial results fit LDS together; << 16: bf16 results; << 17: a group of K per workgroup; << 18: groups of a workgroup; << 31: several tiles of lhs rows
};
template <int ENC, int MROWS, typename AT, int MODE>
__device__ __forceinline__ void small_body(const MmMats& mats, const AT* __restrict__ a, int m, int k, const SmallCut& cut) {
    using I = SmallItem<ENC>;
    constexpr bool kQ8 = ENC == QMM_Q4_0;                   // the lhs as Q8_0 codes and block scales
    constexpr int PL = sizeof(AT) == 4 && !kQ8 ? 2 : 1;     // operand rows of an lhs row
    constexpr int LR = MROWS <= 4 ? 1 : MROWS / 4;          // lhs rows of a lane's results: lane / 16 + 4 j
    constexpr int RN = LR * PL;
    constexpr int kPass = std::min(MROWS, 4 / PL);          // lhs rows that change lanes together
    static_assert(RN <= 4, "operand rows");
    constexpr bool kMin = ENC == QMM_Q4_K || ENC == QMM_Q5_K;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    // (what follows from the launch comes as arguments: the compiler fetches blockDim and gridDim with a vector load and waits for it)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)(cut.packed & 0xffu), chunk = (int)(cut.packed >> 8) & 0xff, per = cut.per, stride = cut.stride;
    const bool out_bf16 = (cut.packed >> 16) & 1, apart = (cut.packed >> 17) & 1;
    const int nn = lane & 15, kg = lane >> 4;
    const int nblk = k >> 8, groups = (int)(cut.packed >> 18) & 0x1fff;
    int share = (int)blockIdx.x, part = (int)blockIdx.y, row0 = 0;  // this workgroup's tiles, group of K, first lhs row
    if (MROWS == small_rows<AT>() && (cut.packed >> 31)) {
        // several tiles of lhs rows: those that read the same weights side by side (blockIdx.y) on one XCD (ids congruent mod 8), every XCD the same number of them
        row0 = (int)blockIdx.y * MROWS, share = (int)blockIdx.z * 8 + (int)blockIdx.x, part = apart ? share / stride : 0;
        share -= part * stride;
        if (share >= stride || (apart && part * waves >= nblk)) return;  // (the whole workgroup)
    }
    // One group per workgroup (then groups is 1, and the operands of the first conversion serve every item), or all of them.  (A flag or a comparison of the group's number instead, as `groups > 1` below, took Q6_K 1184 x 1024
    // with 33 rows from 4.95 to 5.11 us.)
    const int g_first = apart ? part : 0, g_end = apart ? g_first + 1 : groups;
    const uint32_t row_bytes = (uint32_t)(nblk * I::kBpb);
    uint8_t* const ring = smem + wave * (2 * I::kSlot);
    const uint32_t ring_lds = lds_address(ring);
    float* const accs = (float*)(smem + waves * (2 * I::kSlot));  // [chunk][waves][LR][64]
    float* const totals = accs + chunk * waves * LR * 64;  // [chunk][LR][64], with more than one group
    // Weight rows of a matrix in a tile.  Gated, eight of gate and the same eight of up: a workgroup has results whole with half as many of them.  14336 x 4096 4 bf16 rows: seven such tiles for each
    // of 256 compute units, where 896 pairs of whole tiles were four (eight tiles) for each of 224, 15.3 -> 13.9 us; Q6_K 13824 x 5120 28.8 -> 26.9, Q4_K 1000 x 4096 3 rows 6.9 -> 5.8.  The same sums.
    // Pairs of whole tiles are left to small_gated_plan's choice.
    constexpr int kTile = MODE == kSmallGated ? 8 : 16, kEach = MODE == kSmallPairs ? 2 : 1;  // kEach: items that make a result
    const int ntiles = MODE == kSmallMats ? mats.tile_end[kLanesMaxMats - 1] : (mats.n[0] + kTile - 1) / kTile;
    const int my_items = kEach * (share + (per - 1) * stride < ntiles ? per : per - 1);  // (the grid has no workgroup without a tile)

    // item i of the workgroup: its matrix, and the first row there
    auto matrix_of = [&](int i, int& n0, int& n) __attribute__((always_inline)) {
        const int tile = share + i / kEach * stride;
        int j = 0;
        if constexpr (MODE == kSmallMats) {  // (entries past the last repeat it)
#pragma unroll
            for (int i = 0; i + 1 < kLanesMaxMats; i++) j += tile >= mats.tile_end[i] ? 1 : 0;
        }
        n0 = (MODE == kSmallMats && j ? tile - mats.tile_end[j - 1] : tile) * kTile;
        if constexpr (MODE == kSmallPairs) j = i & 1;
        n = mats.n[j];
        return j;
    };
    // piece p = lane + 64 i of an item: row p / kRowPieces
    uint32_t full[I::kLoads];  // byte offset of the piece (Q6_K: of its row) in a tile that lies inside the matrix
    uint32_t at_row = 0;       // Q6_K: where it begins in the row, eight bits each
#pragma unroll
    for (int i = 0; i < I::kLoads; i++) {
        const int p = min(lane + 64 * i, I::kPieces - 1), pr = p / I::kRowPieces, pc = p - pr * I::kRowPieces;
        full[i] = (uint32_t)(pr % kTile) * row_bytes + (ENC == QMM_Q6_K ? 0u : 16u * (uint32_t)pc);
        if constexpr (ENC == QMM_Q6_K) at_row |= (pc < 13 ? 16u * (uint32_t)pc : 196u) << (8 * i);
    }
    auto issue = [&](int sb, int item, int slot) {
        int n0, n;
        const int j = matrix_of(item, n0, n);
        const uint8_t* const base = mats.w[j] + (int64_t)n0 * row_bytes + (ENC == QMM_Q6_K ? 0 : sb * I::kBpb);
        const uint8_t* const base2 = MODE == kSmallGated ? mats.w[1] + (base - mats.w[0]) : base;
        const int last = n - 1 - n0;  // rows past the matrix repeat its last row (their results are dropped)
#pragma unroll
        for (int i = 0; i < I::kLoads; i++) {
            uint32_t off = full[i];
            if (last < kTile - 1) {  // (the last tile of a ragged matrix only)
                const int pr = min(lane + 64 * i, I::kPieces - 1) / I::kRowPieces % kTile;
                off -= (uint32_t)(pr - min(pr, last)) * row_bytes;
            }
            if constexpr (ENC == QMM_Q6_K) off = ((off + (uint32_t)(sb * Q6_K_BPB)) & ~3u) + ((at_row >> (8 * i)) & 0xffu);
            if (i < I::kLoads - 1 || I::kPieces % 64 == 0 || lane < I::kPieces - 64 * (I::kLoads - 1)) {
                const uint32_t to = ring_lds + slot * I::kSlot + i * 1024;
                constexpr int kGate = 8 * I::kRowPieces;  // pieces of the first of two matrices
                if (MODE != kSmallGated || 64 * (i + 1) <= kGate) small_stream16(off, base, to);
                else if (64 * i >= kGate) small_stream16(off, base2, to);
                else load16_to_lds_once((lane + 64 * i < kGate ? base : base2) + off, to);
            }
        }
    };

    // ---- lhs operands of the wavefront's super-block.  Operand row nn: lhs row nn / 4 + 4 j, hi part or (fp32) residual, j and part by nn % 4.
    // Q4_K, Q5_K: fragment (p, h) of lane quarter kg holds columns 64 kg + 32 h + 8 p + (0 .. 7; Q4_K in the order 0,2,1,3,4,6,5,7); Q6_K: fragment g holds 16 g + 4 kg + 0 .. 3.
    // Q4_0: block b of lane quarter kg holds the codes of columns 4 kg .. + 3 and 16 + 4 kg .. + 3; block scales of this lane's results, two fp16 numbers a register.
    half8 fa[kMin ? 4 : 1][2], fs;
    ks_half4 fq[ENC == QMM_Q6_K ? 16 : 1];
    u32x2 fc[kQ8 ? 8 : 1];
    u32x4 fd[kQ8 ? LR : 1];
    float bs[LR];  // inverse lhs scales of this lane's results
#pragma unroll
    for (int b = 0; b < (kQ8 ? 8 : 1); b++) fc[b] = u32x2{0u, 0u};
#pragma unroll
    for (int j = 0; j < (kQ8 ? LR : 1); j++) fd[j] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < (kMin ? 4 : 1); p++) fa[p][0] = fa[p][1] = pack4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int g = 0; g < (ENC == QMM_Q6_K ? 16 : 1); g++) fq[g] = ks_half4{0, 0, 0, 0};
    fs = pack4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int j = 0; j < LR; j++) bs[j] = 0.0f;
    typedef typename std::conditional<sizeof(AT) == 4, u32x4, u32x2>::type xraw_t;
    // xr: columns 4 lane .. 4 lane + 3 of every lhs row; area: a free ring slot
    auto narrow = [&](const xraw_t (&xr)[MROWS], uint8_t* area) __attribute__((always_inline)) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));  // (what is computed from it here is not kept in registers between the groups)
        const int nn = lane & 15, kg = lane >> 4, my_row = (nn >> 2) + 4 * ((nn & 3) / PL), my_part = (nn & 3) % PL;
        if constexpr (kQ8) {
#pragma unroll
            for (int r0 = 0; r0 < MROWS; r0 += kPass) {
                small_quantize<kPass>(xr, r0, area, lane);
                asm volatile("" ::: "memory");  // (scales are written as 16-bit numbers and read as vectors: not to be reordered)
                __builtin_amdgcn_wave_barrier();
                if ((nn & 3) < RN && my_row >= r0 && my_row < r0 + kPass) {
                    const uint8_t* const pl = area + (my_row - r0) * kSmallCodes;
#pragma unroll
                    for (int b = 0; b < 8; b++) fc[b] = *(const u32x2*)(pl + 32 * b + 8 * kg);
                }
#pragma unroll
                for (int j = 0; j < LR; j++)
                    if (kg + 4 * j >= r0 && kg + 4 * j < r0 + kPass) fd[j] = *(const u32x4*)(area + (kg + 4 * j - r0) * kSmallCodes + 256);
            }
        } else {
            float* const scales = (float*)(area + 4 * kSmallPlane);
            constexpr int kTop = kMin ? 9 : 14;
            float common = 1.0f;
            if constexpr (PL == 2) common = small_common_scale<kTop>(xr);
#pragma unroll
            for (int r0 = 0; r0 < MROWS; r0 += kPass) {
                const float inverse = small_narrow<PL, kPass, ENC == QMM_Q4_K ? kSmallOrderK : kSmallOrderPlain, kTop>(xr, r0, common, area, scales, lane);
                __builtin_amdgcn_wave_barrier();
                if ((nn & 3) < RN && my_row >= r0 && my_row < r0 + kPass) {
                    const uint8_t* const pl = area + ((my_row - r0) * PL + my_part) * kSmallPlane;
                    if constexpr (ENC == QMM_Q6_K) {
#pragma unroll
                        for (int g = 0; g < 16; g++) fq[g] = *(const ks_half4*)(pl + 32 * g + 8 * kg);
                    } else {
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            fa[p][0] = *(const half8*)(pl + 128 * kg + 16 * p);
                            fa[p][1] = *(const half8*)(pl + 128 * kg + 64 + 16 * p);
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < LR; j++)
                    if (kg + 4 * j >= r0 && kg + 4 * j < r0 + kPass) bs[j] = inverse == 0.0f ? scales[kg + 4 * j - r0] : inverse;
            }
        }
        if constexpr (kMin) {
            // Sums of the operand rows over 32 columns on the matrix cores: column j < 4 of the product is sub-block 2 j (the lane quarter kg = j supplies the ones),
            // column 4 + j sub-block 2 j + 1.  Through LDS they come to the lane that supplies them: (row nn, sub-blocks 2 kg, 2 kg + 1), as two fp16 terms.
            const uint32_t e0 = nn == kg ? 0x3C003C00u : 0u, e1 = nn == kg + 4 ? 0x3C003C00u : 0u;
            const half8 ones0 = pack4(e0, e0, e0, e0), ones1 = pack4(e1, e1, e1, e1);
            ks_float4 S = {0.f, 0.f, 0.f, 0.f}, S1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < 4; p++) {
                S = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][0], ones0, S, 0, 0, 0);
                S1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][1], ones1, S1, 0, 0, 0);
            }
            S += S1;
            float* const st = (float*)area;
            __builtin_amdgcn_wave_barrier();
            if (nn < 8) {
#pragma unroll
                for (int r = 0; r < RN; r++) st[(4 * kg + r) * 9 + nn] = S[r];
            }
            __builtin_amdgcn_wave_barrier();
            const float s0 = (nn & 3) < RN ? st[nn * 9 + kg] : 0.0f, s1 = (nn & 3) < RN ? st[nn * 9 + 4 + kg] : 0.0f;
            const half2v sh = to_half2(s0, s1), sl = to_half2(fmaf((float)sh.x, -1.0f, s0), fmaf((float)sh.y, -1.0f, s1));
            const uint32_t h = __builtin_bit_cast(uint32_t, sh), l = __builtin_bit_cast(uint32_t, sl);
            fs = pack4((h & 0xffffu) | (l << 16), h, (l >> 16) | (h & 0xffff0000u), 0u);  // (sh0, sl0), (sh0, sh1), (sl1, sh1)
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the operands are in registers before the next item's load may overwrite the slot
    };
    const uint32_t a_lane = 4 * (uint32_t)sizeof(AT) * lane;

    // first group: the lhs, then the first weights, which stay on their way while the lhs is converted.  (Straight-line code: nothing may move a register that such a load has
    // not filled yet.  A wavefront without a super-block, in the last group, takes the last one and drops it.)
    int slot = 0;
    {
        xraw_t xr[MROWS];
        const int sb = min(g_first * waves + wave, nblk - 1);
#pragma unroll
        for (int j = 0; j < MROWS; j++) hidden_load(xr[j], a_lane, a + (int64_t)min(row0 + j, m - 1) * k + sb * 256);
        issue(sb, 0, 0);
        wait_vmcnt<I::kLoads>();
#pragma unroll
        for (int j = 0; j < MROWS; j++) tie(xr[j]);
        narrow(xr, ring + I::kSlot);
    }
    // (constants of the unpack in vector registers: an and-or in one instruction takes no literal and one scalar at most)
    uint32_t m_low = ENC == QMM_Q5_K ? 0x01010101u : 0x03030303u, c54 = 0x54545454u;
    if constexpr (ENC == QMM_Q5_K || ENC == QMM_Q6_K) asm volatile("" : "+v"(m_low), "+v"(c54));
    const ks_float4 zero4 = {0.f, 0.f, 0.f, 0.f};

    for (int c0 = 0; c0 < my_items; c0 += chunk) {
        const int ct = min(chunk, my_items - c0);
        for (int g = g_first; g < g_end; g++) {
            const int sb = g * waves + wave;
            if (sb < nblk) {  // (all wavefronts but for the last group)
            if (groups > 1 && c0 + g > g_first) {
                xraw_t xr[MROWS];
#pragma unroll
                for (int j = 0; j < MROWS; j++) xr[j] = *(const xraw_t*)((const uint8_t*)(a + (int64_t)min(row0 + j, m - 1) * k + sb * 256) + a_lane);
                narrow(xr, ring + (slot ^ 1) * I::kSlot);
            }
            for (int t = 0; t < ct; t++) {
                // the next item: of the chunk, of the next group, of the next chunk
                int ng = g, nt = c0 + t + 1;
                if (t + 1 == ct) {
                    ng = g + 1, nt = c0;
                    if (ng == g_end || sb + waves >= nblk) ng = g_first, nt = c0 + ct;
                }
                if (nt < my_items) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (what was read from that slot is in registers)
                    issue(ng * waves + wave, nt, slot ^ 1);
                    wait_vmcnt<I::kLoads>();
                } else {
                    wait_vmcnt<0>();
                }
                const uint8_t* const lb = ring + slot * I::kSlot + nn * I::kRow;
                float v[LR];
                if constexpr (kQ8) {
                    // codes less 8, times 16, as signed bytes: the dot products of a block come out exact; v = sum of dot / 16 * (d_w d_a), the product of two fp16 numbers exact in fp32
                    const uint32_t* const l32 = (const uint32_t*)lb;
                    float u[2][LR];  // two chains of sums
#pragma unroll
                    for (int j = 0; j < LR; j++) u[0][j] = u[1][j] = 0.0f;
#pragma unroll
                    for (int b = 0; b < 8; b++) {
                        const int at = (18 * b + 2) >> 2;
                        uint32_t x;  // the block begins at 0 or 2 mod 4
                        if ((18 * b + 2) % 4 == 0) x = l32[at + kg];
                        else x = __builtin_amdgcn_alignbyte(l32[at + kg + 1], l32[at + kg], 2);
                        const half2v dp = __builtin_bit_cast(half2v, l32[(18 * b) >> 2]);
                        const _Float16 dw = (18 * b) % 4 ? dp.y : dp.x;
                        const u32x2 w = {((x << 4) & 0xF0F0F0F0u) ^ 0x80808080u, (x & 0xF0F0F0F0u) ^ 0x80808080u};
                        const ks_int4 dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, fc[b]), __builtin_bit_cast(long, w), ks_int4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < LR; j++) {
                            const uint32_t pair = fd[j][b >> 1];  // (a bit cast of the element itself takes the first one)
                            const half2v da2 = __builtin_bit_cast(half2v, pair);
                            u[b & 1][j] = fmaf((float)dot[j], fmaf((float)dw, (float)(b & 1 ? da2.y : da2.x), 0.0f), u[b & 1][j]);
                        }
                    }
#pragma unroll
                    for (int j = 0; j < LR; j++) v[j] = 0.0625f * (u[0][j] + u[1][j]);
                } else if constexpr (ENC == QMM_Q6_K) {
                    const uint32_t* const l32 = (const uint32_t*)lb;
                    const uint32_t skew = 2u * (((uint32_t)nn * (uint32_t)nblk + (uint32_t)sb) & 1u);  // (16 rows of a tile: n0 is even)
                    auto rd = [&](int dw) __attribute__((always_inline)) { return __builtin_amdgcn_alignbyte(l32[dw + 1], l32[dw], skew); };
                    const uint4 s4 = *(const uint4*)(lb + 192);
                    const uint32_t tail = l32[55];  // bytes 208 .. 211
                    const uint32_t sd[4] = {__builtin_amdgcn_alignbyte(s4.y, s4.x, skew), __builtin_amdgcn_alignbyte(s4.z, s4.y, skew),
                                            __builtin_amdgcn_alignbyte(s4.w, s4.z, skew), __builtin_amdgcn_alignbyte(tail, s4.w, skew)};
                    const float d = h2f((uint16_t)(tail >> (8 * skew)));
                    const ks_half4 off96 = {(_Float16)96.0f, (_Float16)96.0f, (_Float16)96.0f, (_Float16)96.0f};
                    float u[2][RN];  // two chains of sums
#pragma unroll
                    for (int r = 0; r < RN; r++) u[0][r] = u[1][r] = 0.0f;
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int e2 = 0; e2 < 2; e2++) {
                            if constexpr (RN == 4) __builtin_amdgcn_sched_barrier(0);  // (with more results on their way at once the compiler spills)
                            const uint32_t QH = rd(32 + 8 * h + 4 * e2 + kg);
#pragma unroll
                            for (int c = 0; c < 4; c++) {
                                const int gr = 8 * h + 2 * c + e2;  // scale group: weights 128 h + 32 c + 16 e2 + (0..15)
                                const uint32_t QL = rd(16 * h + 8 * (c & 1) + 4 * e2 + kg);
                                const uint32_t lo = (c >> 1) ? QL & 0xF0F0F0F0u : (QL << 4) & 0xF0F0F0F0u;
                                const uint32_t hi = ((QH >> (2 * c)) & m_low) | c54;
                                const uint2 bq = make_uint2(__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u));
                                const ks_half4 bw = __builtin_bit_cast(ks_half4, bq) - off96;
                                const float cs = (float)((int)(sd[gr >> 2] << (24 - 8 * (gr & 3))) >> 24);
                                const ks_float4 P = __builtin_amdgcn_mfma_f32_16x16x16f16(fq[gr], bw, zero4, 0, 0, 0);
#pragma unroll
                                for (int r = 0; r < RN; r++) u[h][r] = fmaf(cs, P[r], u[h][r]);
                            }
                        }
#pragma unroll
                    for (int j = 0; j < LR; j++) v[j] = d * (PL == 2 ? (u[0][PL * j] + u[1][PL * j]) + (u[0][PL * j + PL - 1] + u[1][PL * j + PL - 1]) : u[0][j] + u[1][j]);
                } else {
                    const uint4 hdr = *(const uint4*)lb;
                    constexpr int kQs = ENC == QMM_Q4_K ? 16 : 48;
                    const uint4 q0 = *(const uint4*)(lb + kQs + 32 * kg), q1 = *(const uint4*)(lb + kQs + 16 + 32 * kg);
                    // 6-bit scales and mins of sub-blocks 2 kg, 2 kg + 1 (4 .. 7 use the split encoding)
                    const int sh = 16 * (kg & 1);
                    const uint32_t p0 = (hdr.y >> sh) & 0xffffu, p1 = (hdr.z >> sh) & 0xffffu, p2 = (hdr.w >> sh) & 0xffffu;
                    const uint32_t sc_pair = kg >= 2 ? ((p2 & 0x0F0Fu) | ((p0 >> 2) & 0x3030u)) : (p0 & 0x3F3Fu);
                    const uint32_t mn_pair = kg >= 2 ? (((p2 >> 4) & 0x0F0Fu) | ((p1 >> 2) & 0x3030u)) : (p1 & 0x3F3Fu);
                    float d = h2f((uint16_t)(hdr.x & 0xffffu));
                    // what the codes around their middle leave out: (mid d sc - dmin mn) times the sums of the lhs, both as two fp16 terms, the former times a power of two that
                    // brings the largest it can be below 2^15
                    constexpr float kMid = ENC == QMM_Q4_K ? 8.0f : 16.0f;
                    const float dm = kMid * d, dmin = h2f((uint16_t)(hdr.x >> 16)), e0 = (float)(sc_pair & 0xffu), e1 = (float)(sc_pair >> 8);
                    const int scale = 15 - __builtin_amdgcn_frexp_expf(63.0f * (fabsf(dm) + fabsf(dmin)));
                    const float o0 = __builtin_amdgcn_ldexpf(fmaf(dm, e0, -(dmin * (float)(mn_pair & 0xffu))), scale), o1 = __builtin_amdgcn_ldexpf(fmaf(dm, e1, -(dmin * (float)(mn_pair >> 8))), scale);
                    const half2v oh = to_half2(o0, o1), ol = to_half2(fmaf((float)oh.x, -1.0f, o0), fmaf((float)oh.y, -1.0f, o1));
                    const uint32_t ohb = __builtin_bit_cast(uint32_t, oh), olb = __builtin_bit_cast(uint32_t, ol);
                    const half8 offs = pack4(__builtin_amdgcn_perm(ohb, ohb, 0x01000100u), (olb & 0xffffu) | (ohb & 0xffff0000u), (ohb >> 16) | (olb & 0xffff0000u), 0u);
                    const uint32_t qd[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
                    ks_float4 P = zero4, Q = zero4;  // two chains: low and high nibbles
                    if constexpr (ENC == QMM_Q4_K) {
                        const uint32_t M1 = 0x000F000Fu, M2 = 0x00F000F0u;
                        // 64 sc for the low nibbles (q * 2^-24), 4 sc for the high ones (16 q * 2^-24): the operand is sc * (q - 8) * 2^-18 (as sc * q * 2^-24, always a subnormal, the matrix core
                        // drops low bits of the products)
                        const uint32_t sp_lo = to_half2_bits(64.0f * e0, 64.0f * e0), sp_hi = to_half2_bits(4.0f * e1, 4.0f * e1);
                        const uint32_t np_lo = pk_mul(sp_lo, 0x80088008u), np_hi = pk_mul(sp_hi, 0x80808080u);  // -8 * 2^-24, -128 * 2^-24 times it
                        d *= 262144.0f;
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            const uint32_t x0 = qd[2 * p], x1 = qd[2 * p + 1], y0 = x0 >> 8, y1 = x1 >> 8;
                            const half8 blo = pack4(pk_fma(x0 & M1, sp_lo, np_lo), pk_fma(y0 & M1, sp_lo, np_lo), pk_fma(x1 & M1, sp_lo, np_lo), pk_fma(y1 & M1, sp_lo, np_lo));
                            const half8 bhi = pack4(pk_fma(x0 & M2, sp_hi, np_hi), pk_fma(y0 & M2, sp_hi, np_hi), pk_fma(x1 & M2, sp_hi, np_hi), pk_fma(y1 & M2, sp_hi, np_hi));
                            P = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][0], blo, P, 0, 0, 0);
                            Q = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][1], bhi, Q, 0, 0, 0);
                        }
                    } else {
                        const uint4 h0 = *(const uint4*)(lb + 16), h1 = *(const uint4*)(lb + 32);  // fifth bits: bit j of byte i, column i of sub-block j
                        const uint32_t hd[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
                        const uint32_t s_lo = to_half2_bits(e0, e0), s_hi = to_half2_bits(e1, e1), n_lo = to_half2_bits(-80.0f * e0, -80.0f * e0), n_hi = to_half2_bits(-80.0f * e1, -80.0f * e1);
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            uint32_t lo[4], hi[4];
#pragma unroll
                            for (int i = 0; i < 2; i++) {
                                const uint32_t x = qd[2 * p + i], f = hd[2 * p + i] >> (2 * kg);
                                const uint32_t xl = (x << 4) & 0xF0F0F0F0u, xh = x & 0xF0F0F0F0u, fl = (f & m_low) | c54, fh = ((f >> 1) & m_low) | c54;
                                lo[2 * i] = pk_fma(__builtin_amdgcn_perm(fl, xl, 0x05010400u), s_lo, n_lo);
                                lo[2 * i + 1] = pk_fma(__builtin_amdgcn_perm(fl, xl, 0x07030602u), s_lo, n_lo);
                                hi[2 * i] = pk_fma(__builtin_amdgcn_perm(fh, xh, 0x05010400u), s_hi, n_hi);
                                hi[2 * i + 1] = pk_fma(__builtin_amdgcn_perm(fh, xh, 0x07030602u), s_hi, n_hi);
                            }
                            P = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][0], pack4(lo[0], lo[1], lo[2], lo[3]), P, 0, 0, 0);
                            Q = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[p][1], pack4(hi[0], hi[1], hi[2], hi[3]), Q, 0, 0, 0);
                        }
                    }
                    const ks_float4 O = __builtin_amdgcn_mfma_f32_16x16x32_f16(fs, offs, zero4, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < LR; j++) {
                        float sum = P[PL * j] + Q[PL * j], off = O[PL * j];
                        if constexpr (PL == 2) sum += P[PL * j + PL - 1] + Q[PL * j + PL - 1], off += O[PL * j + PL - 1];
                        v[j] = fmaf(d, sum, __builtin_amdgcn_ldexpf(off, -scale));
                    }
                }
                float* const mine = accs + ((t * waves + wave) * LR) * 64 + lane;
#pragma unroll
                for (int j = 0; j < LR; j++) mine[j * 64] = kQ8 ? v[j] : bs[j] * v[j];
                slot ^= 1;
            }
            }
            __syncthreads();
            // the group's result (matrix row 16 tile + nn, lhs row kg + 4 j): dealt to the wavefronts, which add it to that of the groups before
            const int live = min(waves, nblk - g * waves);
            for (int q = wave; q < ct / kEach * LR; q += waves) {
                const int t = q / LR * kEach, j = q % LR, row = row0 + kg + 4 * j;
                float s[kEach];
#pragma unroll
                for (int h = 0; h < kEach; h++) {
                    const float* const src = accs + (((t + h) * waves) * LR + j) * 64 + lane;
                    float c[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    int w = 0;
                    for (; w + 4 <= live; w += 4)
#pragma unroll
                        for (int i = 0; i < 4; i++) c[i] += src[(w + i) * LR * 64];
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        if (w + i < live) c[i] += src[(w + i) * LR * 64];
                    s[h] = (c[0] + c[1]) + (c[2] + c[3]);
                    if (groups > 1) {
                        float* const total = totals + ((t + h) * LR + j) * 64 + lane;
                        if (g > g_first) s[h] = *total + s[h];
                        if (g + 1 < g_end) *total = s[h];
                    }
                }
                if (g + 1 < g_end) continue;
                int n0, n;
                const int mat = matrix_of(c0 + t, n0, n);
                float r = s[0];
                if constexpr (MODE == kSmallGated) r = r / (1.0f + expf(-r)) * dpp_move<0x128>(r);  // (lanes nn < 8: gate, times up eight lanes on)
                if constexpr (MODE == kSmallPairs) r = r / (1.0f + expf(-r)) * s[kEach - 1];
                const int64_t at = (int64_t)row * n + n0 + nn;
                if (row < m && nn < kTile && n0 + nn < n) {
                    if (out_bf16) ((uint16_t*)mats.out[mat])[at] = f2bf(r);
                    else mats.out[mat][at + (int64_t)part * m * n] = r;
                }
            }
            if (g + 1 < g_end || c0 + chunk < my_items) __syncthreads();
        }
    }
}

// Wavefronts a SIMD that the compiler may aim at.  A launch has four, but for six it packs one and two bf16 rows of Q6_K into 80 registers where 90 keep an item's unpacking in flight: 4096 | 1024 | 1024
// x 4096 2 rows 8.4 / 7.8 us, 3664 | 3664 | 3664 x 1024 one row 5.3 / 4.95.
constexpr int small_simd_waves(int enc, int rows, int size, int mode) { return enc == QMM_Q6_K && rows <= 2 && size == 2 && mode == kSmallMats ? 5 : 8; }
template <int ENC, int MROWS, typename AT, int MODE>
__global__ __launch_bounds__(64 * kSmallWaves) __attribute__((amdgpu_waves_per_eu(4, small_simd_waves(ENC, MROWS, sizeof(AT), MODE)))) void gemv_kquant_small_mats_kernel(const MmMats mats, const AT* __restrict__ a, int m, int k, const SmallCut cut) {
    small_body<ENC, MROWS, AT, MODE>(mats, a, m, k, cut);
}

// The plain call: one matrix [n, k].  Twelve dwords of arguments.
template <int ENC, int MROWS, typename AT>
__global__ __launch_bounds__(64 * kSmallWaves) void gemv_kquant_small_kernel(const uint8_t* __restrict__ w, const AT* __restrict__ a, float* __restrict__ out, int n, int m, int k,
                                                                          int per, int stride, uint32_t packed) {
    MmMats mats;
    mats.w[0] = w;
    mats.out[0] = out;
    mats.n[0] = n;
    small_body<ENC, MROWS, AT, kSmallPlain>(mats, a, m, k, SmallCut{per, stride, packed});
}

namespace {

struct SmallPlan {
    int waves, groups, grid, parts, per, chunk, row_tiles;
    bool pairs;
    size_t lds;
};
// Groups of K: of its length only, so that results do not depend on what else a call has.
int small_groups(int64_t k) {
    const int groups = (int)((k / 256 + kSmallWaves - 1) / kSmallWaves);
    return groups == 3 ? 4 : groups;
}
// tiles: of 16 weight rows, gated: of eight of each matrix, or pairs of them (each = 2 items); parts: workgroups that share a tile, one group of K each; per: tiles of a workgroup, 0: as few as there are places for
SmallPlan small_plan(int encoding, int lhs_dtype, int64_t m, int64_t tiles, int64_t k, bool parts, int each = 1, int per = 0) {
    SmallPlan p;
    p.row_tiles = (int)((m + small_most_rows(lhs_dtype) - 1) / small_most_rows(lhs_dtype));
    m = std::min(m, small_most_rows(lhs_dtype));
    const int nblk = (int)(k / 256), groups = small_groups(k);
    p.groups = groups;
    p.waves = (nblk + groups - 1) / groups;
    p.parts = parts ? groups : 1;
    // one workgroup per compute unit (as many as 16 wavefronts allow with few each), all with the same number of tiles or one fewer
    const int per_cu = std::max(1, kSmallWaves / p.waves);
    const int64_t most = std::max<int64_t>(1, small_places(per_cu, p.row_tiles) / p.parts);
    p.per = per ? per : (int)((tiles + most - 1) / most);
    p.grid = (int)((tiles + p.per - 1) / p.per);
    const int slot = encoding == QMM_Q4_0 || encoding == QMM_Q4_K ? SmallItem<QMM_Q4_K>::kSlot : encoding == QMM_Q5_K ? SmallItem<QMM_Q5_K>::kSlot : SmallItem<QMM_Q6_K>::kSlot;
    // (as many items between two barriers as fit: a barrier after each, with two buffers, took Q6_K 28672 x 8192 with 16 rows from 65 to 92 us)
    const int lr = m <= 4 ? 1 : m <= 8 ? 2 : 4, ring = p.waves * 2 * slot, bytes = (p.waves + (groups > p.parts ? 1 : 0)) * lr * 256;
    p.chunk = std::min(std::min(each * p.per, 254), (kLdsPerCu / per_cu - ring) / bytes) / each * each;
    p.lds = (size_t)ring + (size_t)p.chunk * bytes;
    p.pairs = each == 2;
    return p;
}
// us: a tile of one group of K, the lhs of one
double small_item_us(int encoding) { return encoding == QMM_Q4_0 || encoding == QMM_Q4_K ? 1.4 : encoding == QMM_Q5_K ? 1.75 : 2.1; }
double small_convert_us(int encoding, int lhs_dtype, int64_t m) {
    return encoding == QMM_Q4_0 ? (m <= 2 ? 1.2 : m <= 4 ? 1.6 : m <= 8 ? 2.6 : 5.0)
           : lhs_dtype == QMM_F32 ? (m <= 2 ? 1.7 : m <= 4 ? 2.2 : 3.7) : (m <= 2 ? 1.5 : m <= 4 ? 1.7 : m <= 8 ? 3.0 : encoding == QMM_Q6_K ? 3.6 : 4.4);
}
// A gated pair: tiles with eight rows of each matrix, or pairs of whole ones?  By what the fullest compute unit gets, its workgroups' lhs and items one after the other.  The former may leave it an item less, but
// where several workgroups fit a compute unit they are more workgroups, and each converts the lhs: Q4_K 2816 x 1024 16 fp32 rows 6.5 / 7.3 us, Q4_0 4864 x 1024 8 fp32 rows 5.8 / 6.4 in pairs / halves.
// With more than four lhs rows a workgroup, pairs also where nothing is gained: half as many results to a wavefront's store is 2 .. 8 % there (9728 x 2560 16 fp32 rows Q4_0 13.6 / 14.4, 18944 x 3584
// 16 bf16 rows Q4_K 23.4 / 24.3); up to four rows, halves dealt like pairs (Q5_K 2816 x 1024 4 rows in pairs, halves, so dealt 4.5 / 4.3 / 4.15).  Over 460 calls, 1 .. 24 rows, 1.02 of the time of pairs at
// worst, 0.95 on average; always halves 0.96, up to 1.15.
SmallPlan small_gated_plan(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const SmallPlan halves = small_plan(encoding, lhs_dtype, m, (n + 7) / 8, k, false), pairs = small_plan(encoding, lhs_dtype, m, (n + 15) / 16, k, false, 2);
    const int64_t rows = std::min(m, small_most_rows(lhs_dtype));
    auto us = [&](const SmallPlan& p, int items) {
        const int64_t workgroups = ((int64_t)p.grid * p.row_tiles + compute_units() - 1) / compute_units();
        return workgroups * (small_convert_us(encoding, lhs_dtype, rows) + items * p.per * small_item_us(encoding));
    };
    if (rows > 4) return us(halves, 1) < 0.99 * us(pairs, 2) ? halves : pairs;
    return us(halves, 1) <= us(pairs, 2) ? halves : small_plan(encoding, lhs_dtype, m, (n + 7) / 8, k, false, 1, 2 * pairs.per);
}
// A K of several groups: a workgroup per (share of the tiles, group), whose results a launch of their own adds in group order, or all groups in each workgroup?
// The latter converts the lhs again for every group; both give the same bits.  us, walk / apart: Q4_K 1024 x 14336 4 bf16 rows 13.7 / 7.9, 4096 x 14336 2 bf16 rows
// 13.7 / 11.8, 8 fp32 rows 23.2 / 14.7; but two groups and many tiles, 28672 x 8192 4 bf16 rows 27.7 / 29.7, 8192 x 8192 11.5 / 12.1.
bool small_parts(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const int groups = small_groups(k);
    if (groups < 2) return false;
    const double item = small_item_us(encoding), convert = small_convert_us(encoding, lhs_dtype, m);
    const int64_t tiles = (n + 15) / 16;
    const SmallPlan w = small_plan(encoding, lhs_dtype, m, tiles, k, false), a = small_plan(encoding, lhs_dtype, m, tiles, k, true);
    const double walk = groups * ((w.per + w.chunk - 1) / w.chunk) * convert + groups * w.per * item;
    return convert + a.per * item + (a.per - 1) / a.chunk * 1.0 + 2.3 + 1.6e-6 * (4.0 * m * n * groups) < walk;
}

template <int ENC, int MROWS, typename AT>
hipError_t run_small(const MmMats& mats, const SmallPlan& p, const AT* a, int m, int k, bool gated, bool out_bf16, hipStream_t s) {
    const dim3 grid = p.row_tiles > 1 ? dim3(8, (unsigned)p.row_tiles, (unsigned)((p.grid * p.parts + 7) / 8)) : dim3((unsigned)p.grid, (unsigned)p.parts), block((unsigned)(64 * p.waves));
    const SmallCut cut{p.per, p.grid, (uint32_t)p.waves | (uint32_t)p.chunk << 8 | (uint32_t)out_bf16 << 16 | (uint32_t)(p.parts > 1) << 17 | (uint32_t)(p.parts > 1 ? 1 : p.groups) << 18 | (uint32_t)(p.row_tiles > 1) << 31};
    hipError_t e;
    if (gated && p.pairs) {
        if constexpr (MROWS > 4) {
            if ((e = allow_full_lds<gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallPairs>>()) != hipSuccess) return e;
            gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallPairs><<<grid, block, p.lds, s>>>(mats, a, m, k, cut);
        } else {
            return hipErrorInvalidValue;
        }
    } else if (gated) {
        if ((e = allow_full_lds<gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallGated>>()) != hipSuccess) return e;
        gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallGated><<<grid, block, p.lds, s>>>(mats, a, m, k, cut);
    } else if (mats.count > 1) {
        if ((e = allow_full_lds<gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallMats>>()) != hipSuccess) return e;
        gemv_kquant_small_mats_kernel<ENC, MROWS, AT, kSmallMats><<<grid, block, p.lds, s>>>(mats, a, m, k, cut);
    } else {
        if ((e = allow_full_lds<gemv_kquant_small_kernel<ENC, MROWS, AT>>()) != hipSuccess) return e;
        gemv_kquant_small_kernel<ENC, MROWS, AT><<<grid, block, p.lds, s>>>(mats.w[0], a, mats.out[0], mats.n[0], m, k, cut.per, cut.stride, cut.packed);
    }
    return hipGetLastError();
}

template <int ENC>
hipError_t run_small_rows(const MmMats& mats, const SmallPlan& p, const void* a, int lhs_dtype, int m, int k, bool gated, bool out_bf16, hipStream_t s) {
    if (lhs_dtype == QMM_F32) {
        const float* const f = (const float*)a;
        if (m == 1) return run_small<ENC, 1>(mats, p, f, m, k, gated, out_bf16, s);
        if (m <= 2) return run_small<ENC, 2>(mats, p, f, m, k, gated, out_bf16, s);
        if (m <= 4) return run_small<ENC, 4>(mats, p, f, m, k, gated, out_bf16, s);
        return run_small<ENC, 8>(mats, p, f, m, k, gated, out_bf16, s);
    }
    const uint16_t* const b = (const uint16_t*)a;
    if (m == 1) return run_small<ENC, 1>(mats, p, b, m, k, gated, out_bf16, s);
    if (m <= 2) return run_small<ENC, 2>(mats, p, b, m, k, gated, out_bf16, s);
    if (m <= 4) return run_small<ENC, 4>(mats, p, b, m, k, gated, out_bf16, s);
    if (m <= 8) return run_small<ENC, 8>(mats, p, b, m, k, gated, out_bf16, s);
    return run_small<ENC, 16>(mats, p, b, m, k, gated, out_bf16, s);
}

}  // namespace

bool gemv_kquant_small_supported(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, const void* w) {
    if (encoding != QMM_Q4_0 && encoding != QMM_Q4_K && encoding != QMM_Q5_K && encoding != QMM_Q6_K) return false;
    // (with the name of an encoding's older small-batch kernel this one goes too)
    if (kernel_disabled("kquant_small") || kernel_disabled(encoding == QMM_Q4_0 ? "q4_0_small" : encoding == QMM_Q4_K ? "q4k_mm" : encoding == QMM_Q5_K ? "q5k_mm" : "q6k_mm")) return false;
    if (m < 1 || m > small_most_rows(lhs_dtype) * 4 || n < 1 || n > 0x7fffff00 || k < 256 || k % 256 || k > (1 << 20)) return false;
    if (encoding == QMM_Q4_K || encoding == QMM_Q5_K) return ((uintptr_t)w & 15) == 0;
    if (encoding == QMM_Q4_0) return ((uintptr_t)w & 3) == 0;
    // (loads of four bytes at least: the last block of the matrix has to end at a multiple of four)
    return ((uintptr_t)w & 3) == 0 && n * (k / 256) % 2 == 0;
}

// What the fullest compute unit gets of a call whose workgroups walk K, a tile being 16 weight rows: small_tiles_wanted.
SmallLoad small_load(int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const SmallPlan p = small_plan(QMM_Q4_K, lhs_dtype, m, (n + 15) / 16, k, false);
    const int workgroups = ((int64_t)p.grid * p.row_tiles + compute_units() - 1) / compute_units();
    return {workgroups, workgroups * p.waves};
}

// What the parts of K of a plain call with few tiles take (without it a workgroup walks all of K: the same sums).
int64_t gemv_kquant_small_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return small_parts(encoding, lhs_dtype, m, n, k) ? small_groups(k) * m * n * 4 : 0;
}

namespace {
__global__ __launch_bounds__(256) void small_sum_bf16_kernel(const float* __restrict__ part, uint16_t* __restrict__ out, int64_t count, int parts) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    float v = 0.0f;
    for (int j = 0; j < parts; j++) v += part[j * count + i];
    out[i] = f2bf(v);
}
// The same for matrices that share a launch: matrix j has the values from end[j - 1] to end[j], and their shares at part[j], one after the other.
struct SmallSums {
    const float* part[kLanesMaxMats];
    float* out[kLanesMaxMats];
    int64_t end[kLanesMaxMats];
};
__global__ __launch_bounds__(256) void small_sum_mats_kernel(SmallSums sums, int parts) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= sums.end[kLanesMaxMats - 1]) return;
    const float* part = sums.part[0];
    float* out = sums.out[0];
    int64_t first = 0, end = sums.end[0];
#pragma unroll
    for (int j = 1; j < kLanesMaxMats; j++)
        if (i >= sums.end[j - 1]) part = sums.part[j], out = sums.out[j], first = sums.end[j - 1], end = sums.end[j];
    float v = 0.0f;
    for (int j = 0; j < parts; j++) v += part[j * (end - first) + i - first];
    out[i - first] = v;
}
}  // namespace
// out[i] = bf16(part[i] + part[count + i] + ...), in that order
hipError_t launch_sum_shares_bf16(const float* part, uint16_t* out, int64_t count, int shares, hipStream_t s) {
    small_sum_bf16_kernel<<<dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s>>>(part, out, count, shares);
    return hipGetLastError();
}

// count matrices [ns[j], k] that share the lhs; gated: two of the same size, gate and up, outs[0] = silu(lhs gate^T) * (lhs up^T).  The caller has asked
// gemv_kquant_small_supported for each.  out_bf16: the outputs are bf16 arrays.  workspace: null, or (not gated) gemv_kquant_small_workspace_bytes with n = the sum of ns.
hipError_t launch_gemv_kquant_small(int encoding, const void* lhs, int lhs_dtype, int count, const void* const* ws, const int64_t* ns, float* const* outs, int64_t m, int64_t k,
                                    bool gated, bool out_bf16, void* workspace, hipStream_t s) {
    if (count < 1 || count > kLanesMaxMats || (gated && (count != 2 || ns[0] != ns[1]))) return hipErrorInvalidValue;
    MmMats mats;
    int64_t tiles = 0;
    for (int j = 0; j < kLanesMaxMats; j++) {
        const int i = std::min(j, count - 1);
        if (j < count) tiles += (ns[j] + 15) / 16;
        mats.w[j] = (const uint8_t*)ws[i];
        mats.out[j] = outs[gated ? 0 : i];
        mats.n[j] = (int)ns[i];
        mats.tile_end[j] = (int)tiles;
    }
    mats.count = count;
    int64_t all = 0;
    for (int j = 0; j < count; j++) all += ns[j];
    const bool parts = !gated && workspace && small_parts(encoding, lhs_dtype, m, all, k);
    SmallSums sums;
    int64_t values = 0;
    if (parts)
        for (int j = 0; j < kLanesMaxMats; j++) {
            sums.part[j] = mats.out[j] = (float*)workspace + values * small_groups(k);
            sums.out[j] = outs[std::min(j, count - 1)];
            if (j < count) values += m * ns[j];
            sums.end[j] = values;
        }
    const SmallPlan p = gated ? small_gated_plan(encoding, lhs_dtype, m, ns[0], k) : small_plan(encoding, lhs_dtype, m, tiles, k, parts);
    const bool store_bf16 = out_bf16 && !parts;
    hipError_t e = encoding == QMM_Q4_0   ? run_small_rows<QMM_Q4_0>(mats, p, lhs, lhs_dtype, (int)m, (int)k, gated, store_bf16, s)
                   : encoding == QMM_Q4_K ? run_small_rows<QMM_Q4_K>(mats, p, lhs, lhs_dtype, (int)m, (int)k, gated, store_bf16, s)
                   : encoding == QMM_Q5_K ? run_small_rows<QMM_Q5_K>(mats, p, lhs, lhs_dtype, (int)m, (int)k, gated, store_bf16, s)
                                          : run_small_rows<QMM_Q6_K>(mats, p, lhs, lhs_dtype, (int)m, (int)k, gated, store_bf16, s);
    if (e != hipSuccess || !parts) return e;
    if (count > 1) {  // (fp32 results: the callers with several matrices have no others)
        small_sum_mats_kernel<<<dim3((unsigned)((values + 255) / 256)), dim3(256), 0, s>>>(sums, p.parts);
        return hipGetLastError();
    }
    if (!out_bf16) return launch_sum_shares((const float*)workspace, outs[0], values, p.parts, s);
    return launch_sum_shares_bf16((const float*)workspace, (uint16_t*)outs[0], values, p.parts, s);
}

}  // namespace qmm
