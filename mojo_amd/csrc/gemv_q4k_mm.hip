// Q4_K small-batch kernel (9 to 16 lhs rows over prepared lhs planes): weight rows streamed through LDS, 16 x 16 x 32
// matrix-core products over exact integer codes.
//
// Arithmetic is that of the prefill kernel (gemm_q4k.hip): a masked nibble is the fp16 subnormal
// q*2^-24, one packed fp16 multiply folds the 6-bit sub-block scale in (times 64), the lhs was narrowed to fp16
// (hi, plus a residual plane) by a separate pass (gemm_lhs.h) after an exact power-of-two scaling of the row, the fp32 super-block scale is
// applied in the lanes and the min term is one extra matrix product per super-block.  An fp32 lhs costs a second matrix product per operand.
//
// Shape of the work: a workgroup of 8 wavefronts walks a list of up to 4 weight tiles of 16 rows.
// The super-blocks of a row are dealt to the wavefronts in groups of 16, two per wavefront; a
// wavefront's lhs fragments for its two super-blocks of a group are held in registers and reused
// for every tile of the workgroup.  The weights of a (group, tile) item, 288 contiguous bytes of
// each of the 16 rows, travel from global memory straight into a wavefront-private ring of three
// LDS slots (global_load_lds_dwordx4: no registers are held while they are in flight), two items
// ahead of the one being decoded; the wavefront waits with a vmcnt that leaves the younger items
// in flight.  Lane (row n = lane % 16, chunk c = lane / 16) decodes the 32 code bytes of chunk c of
// its row: sub-block 2c in the low nibbles, 2c + 1 in the high ones, so it needs only those two
// scales and mins; 8 code bytes feed two matrix-core instructions.  A wavefront accumulates its
// partial result of a tile over the groups in a private LDS slot; one barrier at the end, then the
// 8 partial results of a tile are added in a fixed order.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "gemm_lhs.h"
#include "lds_stream.h"
#include "qmm_internal.h"

namespace qmm {

typedef float float4v __attribute__((ext_vector_type(4)));

namespace {

constexpr int kRunBlk = 2;                      // super-blocks per item
constexpr int kRowBytes = kRunBlk * Q4_K_BPB;   // 288: bytes of a row in an item (18 pieces of 16 bytes)
constexpr int kPieces = 16 * kRowBytes / 16;    // 288 pieces per item, piece p at LDS offset 16 p
constexpr int kLoads = (kPieces + 63) / 64;     // 5 load instructions per item, the last one by 32 lanes
constexpr int kSlotBytes = kPieces * 16;        // 4608
constexpr int kSlots = 3;                       // ring: one item being decoded, two in flight
constexpr float kTwo18f = 262144.0f;
constexpr int kWaves = 8;                       // wavefronts per workgroup
constexpr int kMaxTiles = 4;                    // tiles per workgroup (private LDS accumulators per wavefront)
constexpr int kRingBytes = kWaves * kSlots * kSlotBytes;
constexpr int kAccBytes = kWaves * kMaxTiles * 4 * 64 * 4;
constexpr int kLdsBytes = kRingBytes + kAccBytes;
__device__ __forceinline__ half8 zero_half8() { return pack4(0u, 0u, 0u, 0u); }

}  // namespace

// NPART: matrix products per weight operand (2: hi and residual planes).
template <int NPART>
__global__ __launch_bounds__(512) void gemv_q4_k_mm_kernel(const MmMats mats, const _Float16* __restrict__ a16, const _Float16* __restrict__ a16_lo,
                                                           const _Float16* __restrict__ asum, const float* __restrict__ inv, int m, int k) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nblk = k >> 8;
    const int64_t row_bytes = (int64_t)nblk * Q4_K_BPB;
    const int nn = lane & 15, kg = lane >> 4;
    uint8_t* ring = smem + wave * (kSlots * kSlotBytes);
    const uint32_t ring_lds = lds_address(ring);
    float* accs = (float*)(smem + kRingBytes);  // [kWaves][kMaxTiles][4][64]
    const int ntiles = mats.tile_end[kLanesMaxMats - 1];  // 16-row tiles, numbered through the matrices (entries past count repeat the last)
    // One matrix (the plain call) needs nothing from the argument block per item; with several, the tile's matrix is
    // looked up there (dependent scalar loads per item).
    const bool single = mats.count == 1;
    const uint8_t* const w_first = mats.w[0];
    float* const out_first = mats.out[0];
    const int n_first = mats.n[0];
    const int my_tiles = min(kMaxTiles, (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x);
    // group g is super-blocks [16 g, 16 g + 16): two per wavefront, or, when 8 or fewer are left, one
    const int ngrp = (nblk + kRunBlk * kWaves - 1) / (kRunBlk * kWaves), total = ngrp * my_tiles;
    auto group_share = [&](int g, int& first, int& cnt) {
        const int left = nblk - kRunBlk * kWaves * g;  // > 0
        const int per = left > kWaves ? kRunBlk : 1;
        first = kRunBlk * kWaves * g + per * wave;
        cnt = max(0, min(per, nblk - first));
        first = min(first, nblk - 1);  // (no share: a valid address, the data is not used)
    };

    int last_issued = -1;  // newest item whose loads into LDS have been issued
    // piece p = lane + 64 i of an item: row p / 18, 16-byte piece p % 18
    int prow[kLoads], pidx[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int p = min(lane + 64 * i, kPieces - 1);
        prow[i] = p / 18;
        pidx[i] = p - prow[i] * 18;
    }
    // item (group g, tile index t) -> ring slot `slot`
    auto issue = [&](int g, int t, int slot) {
        const int tile = (int)blockIdx.x + t * (int)gridDim.x;
        int n0 = tile * 16, n = n_first;
        const uint8_t* wj = w_first;
        if (!single) {
            int j = 0;
            while (j + 1 < mats.count && tile >= mats.tile_end[j]) j++;  // (uniform: a few scalar compares)
            n0 = (tile - (j ? mats.tile_end[j - 1] : 0)) * 16;
            n = mats.n[j];
            wj = mats.w[j];
        }
        int bc, cnt;
        group_share(g, bc, cnt);
        const int last_piece = max(cnt, 1) * 9 - 1;
        const uint8_t* base = wj + (int64_t)bc * Q4_K_BPB;
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const uint8_t* src = base + (int64_t)min(n0 + prow[i], n - 1) * row_bytes + 16 * min(pidx[i], last_piece);
            if (i < kLoads - 1 || lane < kPieces - 64 * (kLoads - 1))  // the last instruction: 32 lanes
                load16_to_lds_once(src, ring_lds + slot * kSlotBytes + i * 1024);
        }
    };

    // items in flight: it + 1 and it + 2
    int ig = 0, it_t = 0, islot = 0;  // next item to issue
    auto issue_next = [&]() {
        issue(ig, it_t, islot);
        last_issued++;
        islot = islot == kSlots - 1 ? 0 : islot + 1;
        if (++it_t == my_tiles) { it_t = 0; ig++; }
    };
    if (total > 0) issue_next();
    if (total > 1) issue_next();

    const int mrow = min(nn, m - 1);  // lhs operand row of this lane
    const uint32_t M1 = 0x000F000Fu, M2 = 0x00F000F0u;
    const int sh = 16 * (kg & 1);  // byte pair (2c, 2c + 1) mod 4 inside a dword of the 6-bit fields
    const bool upper = kg >= 2;    // sub-blocks 4..7 use the split encoding

    half8 fa[kRunBlk][4][2][NPART], fs[kRunBlk];
#pragma unroll
    for (int bb = 0; bb < kRunBlk; bb++) {
        fs[bb] = zero_half8();
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int q = 0; q < NPART; q++) fa[bb][p][h][q] = zero_half8();
    }

    int grp = 0, ti = 0, slot = 0;
    for (int it = 0; it < total; it++) {
        int gb0, nb;
        group_share(grp, gb0, nb);
        if (ti == 0) {
            // lhs fragments of the group's super-blocks: registers, reused for every tile.
            // Fragment (p, h) of chunk kg holds lhs columns 64 kg + 32 h + 8 p + (0,2,1,3,4,6,5,7).
#pragma unroll
            for (int bb = 0; bb < kRunBlk; bb++) {
                const int blk = min(gb0 + bb, nblk - 1);
                const _Float16* ah = a16 + (int64_t)mrow * k + (int64_t)blk * 256 + 64 * kg;
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    fa[bb][p][0][0] = *(const half8*)(ah + 8 * p);
                    fa[bb][p][1][0] = *(const half8*)(ah + 32 + 8 * p);
                }
                if constexpr (NPART == 2) {
                    const _Float16* al = a16_lo + (int64_t)mrow * k + (int64_t)blk * 256 + 64 * kg;
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        fa[bb][p][0][1] = *(const half8*)(al + 8 * p);
                        fa[bb][p][1][1] = *(const half8*)(al + 32 + 8 * p);
                    }
                }
                // asum: 8 hi parts then 8 lo parts per super-block
                const uint16_t* as = (const uint16_t*)asum + ((int64_t)mrow * nblk + blk) * 16 + 2 * kg;
                const uint32_t hi = *(const uint32_t*)as, lo = *(const uint32_t*)(as + 8);  // (ah0, ah1), (al0, al1)
                fs[bb] = pack4((hi & 0xffffu) | (lo << 16), hi, (lo >> 16) | (hi & 0xffff0000u), 0u);
            }
        }
        // the slot of item it - 1 is free: its reads fed matrix products whose results are already stored
        while (last_issued < min(it + 2, total - 1)) issue_next();
        // item `it` has landed when only the loads of later items are outstanding
        wait_items<kLoads, 0>(last_issued - it, false);
        const uint8_t* wbuf = ring + slot * kSlotBytes;

        float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int bb = 0; bb < kRunBlk; bb++) {
            if (bb >= nb) break;
            const uint8_t* lb = wbuf + nn * kRowBytes + bb * Q4_K_BPB;
            const uint4 hdr = *(const uint4*)lb;
            const uint4 q0 = *(const uint4*)(lb + 16 + 32 * kg), q1 = *(const uint4*)(lb + 32 + 32 * kg);
            // 6-bit scales and mins of sub-blocks 2 kg, 2 kg + 1
            const uint32_t p0 = (hdr.y >> sh) & 0xffffu, p1 = (hdr.z >> sh) & 0xffffu, p2 = (hdr.w >> sh) & 0xffffu;
            const uint32_t sc_pair = upper ? ((p2 & 0x0F0Fu) | ((p0 >> 2) & 0x3030u)) : (p0 & 0x3F3Fu);
            const uint32_t mn_pair = upper ? (((p2 >> 4) & 0x0F0Fu) | ((p1 >> 2) & 0x3030u)) : (p1 & 0x3F3Fu);
            // 64 * sc for the low nibbles (q * 2^-24), 4 * sc for the high ones (16 q * 2^-24): the operand is
            // sc * q * 2^-18, a normal fp16 number from sc * q = 16 on (as sc * q * 2^-24, always a subnormal, the
            // matrix core drops low bits of the products of small sc * q towards minus infinity: a bias growing with K)
            const float e0 = 64.0f * (float)(sc_pair & 0xffu), e1 = 4.0f * (float)(sc_pair >> 8);
            const uint32_t sp_lo = pack_half2(e0, e0), sp_hi = pack_half2(e1, e1);
            // min term: weight slots (bh0, bh0, bl0, bh1, bh1, bl1, 0, 0) of -(dmin * mn_j), hi and residual parts
            float4v Bk = {0.f, 0.f, 0.f, 0.f};
            {
                const uint32_t ndm = ((hdr.x >> 16) ^ 0x8000u) * 0x00010001u;  // (-dmin, -dmin)
                const uint32_t mp = pack_half2((float)(mn_pair & 0xffu), (float)(mn_pair >> 8));
                const uint32_t hi = pk_mul(ndm, mp);
                const uint32_t lo = pk_fma(ndm, mp, hi ^ 0x80008000u);
                const half8 bmin = pack4((hi & 0xffffu) * 0x00010001u, (lo & 0xffffu) | (hi & 0xffff0000u),
                                         (hi >> 16) | (lo & 0xffff0000u), 0u);
                Bk = __builtin_amdgcn_mfma_f32_16x16x32_f16(fs[bb], bmin, Bk, 0, 0, 0);
            }
            float4v P = {0.f, 0.f, 0.f, 0.f}, Q = {0.f, 0.f, 0.f, 0.f};  // two chains: low and high nibbles
            const uint32_t qd[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const uint32_t x0 = qd[2 * p], x1 = qd[2 * p + 1], y0 = x0 >> 8, y1 = x1 >> 8;
                const half8 blo = pack4(pk_mul(x0 & M1, sp_lo), pk_mul(y0 & M1, sp_lo), pk_mul(x1 & M1, sp_lo),
                                        pk_mul(y1 & M1, sp_lo));
                const half8 bhi = pack4(pk_mul(x0 & M2, sp_hi), pk_mul(y0 & M2, sp_hi), pk_mul(x1 & M2, sp_hi),
                                        pk_mul(y1 & M2, sp_hi));
                P = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[bb][p][0][0], blo, P, 0, 0, 0);
                Q = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[bb][p][1][0], bhi, Q, 0, 0, 0);
                if constexpr (NPART == 2) {
                    P = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[bb][p][0][1], blo, P, 0, 0, 0);
                    Q = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[bb][p][1][1], bhi, Q, 0, 0, 0);
                }
            }
            const float dsc = h2f((uint16_t)(hdr.x & 0xffffu)) * kTwo18f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float v = fmaf(dsc, P[r] + Q[r], Bk[r]);
                acc[r] += v;
            }
        }
        // this wavefront's running sum of the tile over its groups
        float* mine = accs + (wave * kMaxTiles + ti) * 4 * 64 + lane;
#pragma unroll
        for (int r = 0; r < 4; r++) mine[r * 64] = grp == 0 ? acc[r] : mine[r * 64] + acc[r];

        slot = slot == kSlots - 1 ? 0 : slot + 1;
        if (++ti == my_tiles) { ti = 0; grp++; }
    }
    __syncthreads();
    // lane holds lhs rows 4 kg + r of weight row 16 tile + nn; (tile, r) pairs are dealt to the wavefronts
    for (int pr = wave; pr < my_tiles * 4; pr += kWaves) {
        const int t = pr >> 2, r = pr & 3;
        const int tile = (int)blockIdx.x + t * (int)gridDim.x;
        int n = n_first, tile0 = 0;
        float* out = out_first;
        if (!single) {
            int j = 0;
            while (j + 1 < mats.count && tile >= mats.tile_end[j]) j++;
            n = mats.n[j];
            out = mats.out[j];
            tile0 = j ? mats.tile_end[j - 1] : 0;
        }
        const int col = (tile - tile0) * 16 + nn, row = 4 * kg + r;
        float v = 0.0f;
#pragma unroll
        for (int ww = 0; ww < kWaves; ww++) {
            v += accs[((ww * kMaxTiles + t) * 4 + r) * 64 + lane];
        }
        if (row < m && col < n) out[(int64_t)row * n + col] = v * inv[row];
    }
}

int64_t gemv_q4_k_mm_workspace_bytes(int lhs_dtype, int64_t m, int64_t k) {
    return m <= 8 ? 0 : lhs_planes(nullptr, lhs_dtype, m, k).bytes;
}

// count matrices [ns[j], k] that share the lhs (count = 1: the plain call); out[j] is fp32 [m, ns[j]], dense.
hipError_t launch_gemv_q4_k_mm_grouped(const void* lhs, int lhs_dtype, int count, const uint8_t* const* ws, const int64_t* ns,
                                       float* const* outs, int64_t m, int64_t k, void* workspace, hipStream_t s) {
    if (count < 1 || count > kLanesMaxMats || m < 9) return hipErrorInvalidValue;
    MmMats mats;
    int64_t ntiles = 0;
    for (int j = 0; j < kLanesMaxMats; j++) {
        const int jj = j < count ? j : count - 1;
        if (j < count) ntiles += (ns[j] + 15) / 16;
        mats.w[j] = ws[jj];
        mats.out[j] = outs[jj];
        mats.n[j] = (int)ns[jj];
        mats.tile_end[j] = (int)ntiles;
    }
    mats.count = count;
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return hipGetLastError();
        cus = prop.multiProcessorCount;
    }
    hipError_t e = allow_full_lds<gemv_q4_k_mm_kernel<1>>();
    if (e == hipSuccess) e = allow_full_lds<gemv_q4_k_mm_kernel<2>>();
    if (e != hipSuccess) return e;
    // every workgroup gets the same number of tiles (at most kMaxTiles), one workgroup per compute unit when that fits
    // (more tiles on fewer workgroups is slower at every size: 4096 x 14336, 4 rows: 18.1 / 23.8 / 36.0 us with 1 / 2 / 4 tiles)
    const int64_t per_wg = std::min<int64_t>(kMaxTiles, (ntiles + cus - 1) / cus);
    const int64_t wgs = (ntiles + per_wg - 1) / per_wg;
    dim3 grid((unsigned)wgs), block(64 * kWaves);
    const LhsPlanes p = lhs_planes(workspace, lhs_dtype, m, k);
    e = launch_prep_lhs<kLhsOrderQ4K16>(lhs, lhs_dtype, m, k, p, s);
    if (e != hipSuccess) return e;
    if (!p.a16_lo)
        gemv_q4_k_mm_kernel<1><<<grid, block, kLdsBytes, s>>>(mats, p.a16, nullptr, p.asum, p.inv, (int)m, (int)k);
    else
        gemv_q4_k_mm_kernel<2><<<grid, block, kLdsBytes, s>>>(mats, p.a16, p.a16_lo, p.asum, p.inv, (int)m, (int)k);
    return hipGetLastError();
}

hipError_t launch_gemv_q4_k_mm(const void* lhs, int lhs_dtype, const uint8_t* w, int64_t m, int64_t n, int64_t k,
                               float* out, void* workspace, hipStream_t s) {
    return launch_gemv_q4_k_mm_grouped(lhs, lhs_dtype, 1, &w, &n, &out, m, k, workspace, s);
}

}  // namespace qmm
