// Act-order GPTQ checkpoints (desc_act = True) with several lhs rows: the columns of K sorted by group, so that the kernels for plain
// groups serve the call.
//
// The kernel that looks the group of every k up (gemv_gptq.hip) passes over the weights once per four rows and multiplies on the vector
// units: 14336 x 4096 with 400 bf16 rows took 2.4 ms, this way 103 us.  Sorting costs one small launch and one pass over the packed weights: the words of
// some columns of the output lie in LDS (all of K), from which every word of the sorted matrix takes its eight nibbles; other workgroups
// of that launch sort the columns of the lhs.  What bounds the pass is reading and writing the packed weights (2 x 29 MB at 14336 x 4096: 17 us with 400 rows of
// lhs, 3.8 TB/s; the sort, one workgroup, 6; profiles/direct_gemm_act_order_quantisers__kernel_trace.txt).
//
// A sorted column list is a plain-group matrix only if every group has exactly group_size columns, which is so in any checkpoint that was
// quantised group by group.  The device finds out: where it is not so, the sort leaves a mark, the order as it was (the products are then
// meaningless) and the look-up kernel, launched behind them, replaces the whole result; otherwise that launch returns at once.
#include <algorithm>

#include "qmm_internal.h"

namespace qmm {

namespace {

typedef uint32_t go_u4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(4))) GoWords4 {  // (qweight is 4-byte aligned)
    go_u4 v;
};

constexpr int kSortWaves = 16;

// source[p]: the column of K at sorted position p.  Stable (within a group the columns keep their order).  One workgroup; wavefront w
// takes a sixteenth of K.  Group indices outside [0, groups) are clamped, as in the look-up kernel.
__global__ __launch_bounds__(64 * kSortWaves) void gptq_order_sort_kernel(const int32_t* __restrict__ g_idx, int k, int group, int bits,
                                                                          int32_t* __restrict__ source, int32_t* __restrict__ uneven) {
    extern __shared__ uint32_t counts[];  // [kSortWaves][groups], then whether any group has another size
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = k / group;
    uint32_t* const bad = counts + kSortWaves * groups;
    for (int i = tid; i <= kSortWaves * groups; i += 64 * kSortWaves) counts[i] = 0;
    __syncthreads();
    const int per = ((k + kSortWaves - 1) / kSortWaves + 63) / 64 * 64, lo = min(k, wave * per), hi = min(k, lo + per);
    uint32_t* const mine = counts + wave * groups;
    auto group_of = [&](int i) __attribute__((always_inline)) { return min(max(g_idx[i], 0), groups - 1); };
    for (int i = lo + lane; i < hi; i += 64) atomicAdd(mine + group_of(i), 1u);
    __syncthreads();
    for (int g = tid; g < groups; g += 64 * kSortWaves) {  // where each wavefront's columns of the group begin
        uint32_t at = 0;
        for (int w = 0; w < kSortWaves; w++) {
            const uint32_t c = counts[w * groups + g];
            counts[w * groups + g] = at;
            at += c;
        }
        if (at != (uint32_t)group) *bad = 1;
    }
    __syncthreads();
    const bool as_is = *bad != 0;
    if (tid == 0) *uneven = as_is;
    if (as_is) {
        for (int i = tid; i < k; i += 64 * kSortWaves) source[i] = i;
        return;
    }
    for (int i0 = lo; i0 < hi; i0 += 64) {
        const int i = i0 + lane;
        const bool live = i < hi;
        const int g = live ? group_of(i) : 0;
        uint64_t same = __ballot(live);  // the lanes with this lane's group
        for (int b = 0; b < bits; b++) {
            const bool set = (g >> b) & 1;
            const uint64_t with = __ballot(set);
            same &= set ? with : ~with;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1)), count = __popcll(same);
        if (live) {
            const uint32_t at = mine[g];
            source[g * group + (int)at + rank] = i;
            if (rank == count - 1) mine[g] = at + (uint32_t)count;
        }
        // (the next turn of this wavefront reads what its lanes wrote: LDS operations of a wavefront are performed in order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The first 8 * per_xcd workgroups: COLS columns of the weights each, neighbours on one XCD (they share cache lines).  Then one per lhs row.
template <typename AT, int COLS>
__global__ __launch_bounds__(512) void gptq_order_permute_kernel(const uint32_t* __restrict__ qweight, const AT* __restrict__ a, int n, int k, int per_xcd,
                                                                 const int32_t* __restrict__ source, uint32_t* __restrict__ sorted_w,
                                                                 AT* __restrict__ sorted_a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, b = (int)blockIdx.x;
    if (b < 8 * per_xcd) {
        constexpr int kPieces = COLS / 4;
        const int col = ((b & 7) * per_xcd + (b >> 3)) * COLS + 4 * (tid & (kPieces - 1));
        const int rows = k >> 3, r0 = tid / kPieces;
        constexpr int kRows = 512 / kPieces;  // rows per turn
        const bool in_n = col < n;            // (N is a multiple of 8)
        const uint32_t* from = qweight + (in_n ? col : 0);
        uint32_t* const words = (uint32_t*)smem + 4 * (tid & (kPieces - 1));
#pragma unroll 8
        for (int r = r0; r < rows; r += kRows) *(go_u4*)(words + r * COLS) = ((const GoWords4*)(from + (int64_t)r * n))->v;
        __syncthreads();
        if (!in_n) return;
#pragma unroll 2
        for (int r = r0; r < rows; r += kRows) {
            const int4 s0 = *(const int4*)(source + 8 * r), s1 = *(const int4*)(source + 8 * r + 4);
            const int src[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
            go_u4 o = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const go_u4 x = *(const go_u4*)(words + (src[j] >> 3) * COLS);
                const int at = 4 * (src[j] & 7);
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] |= ((x[c] >> at) & 0xFu) << (4 * j);
            }
            *(go_u4*)(sorted_w + (int64_t)r * n + col) = o;
        }
        return;
    }
    const int64_t row = b - 8 * per_xcd;
    AT* const held = (AT*)smem;
    const AT* ar = a + row * k;
    constexpr int kPer = 16 / sizeof(AT);
    for (int i = tid * kPer; i < k; i += 512 * kPer) *(go_u4*)(held + i) = *(const go_u4*)(ar + i);
    __syncthreads();
    for (int i = tid * kPer; i < k; i += 512 * kPer) {
        AT v[kPer] __attribute__((aligned(16)));
#pragma unroll
        for (int j = 0; j < kPer; j += 4) {
            const int4 s = *(const int4*)(source + i + j);
            v[j] = held[s.x];
            v[j + 1] = held[s.y];
            v[j + 2] = held[s.z];
            v[j + 3] = held[s.w];
        }
        *(go_u4*)(sorted_a + row * k + i) = *(const go_u4*)v;
    }
}

}  // namespace

GptqOrderSpace gptq_order_space(void* workspace, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    GptqOrderSpace p;
    char* base = (char*)workspace;
    p.uneven = (int32_t*)base;
    int64_t off = 256;
    p.source = (int32_t*)(base + off);
    off += up(k * 4);
    p.qweight = (uint32_t*)(base + off);
    off += up(n * k / 2);
    p.lhs = base + off;
    off += up(m * k * (lhs_dtype == QMM_F32 ? 4 : 2));
    p.bytes = off;
    return p;
}

// The look-up kernel or the sort and the direct GEMM: the predicted time of both in microseconds.  The look-up kernel walks K with one workgroup per 64
// columns, in passes of up to four rows; where its table of scales does not fit LDS (small groups on a long K), every weight reads its
// scale from memory.  The sorted way is five launches and one pass over the weights, whatever the number of rows up to 32.  Fitted to timings of
// 20 matrices (512 x 512 .. 8192 x 28672, groups of 32 and 128) with 1 .. 16 rows: 9 .. 12 % off, and what it picks takes 0.4 % longer on average than
// the faster of the two.  us, look-up / sorted: 14336 x 4096 4 bf16 rows 25 / 38, 6 rows 45 / 38, fp32 8 rows 41 / 40; 4096 x 4096 4 / 5 rows
// 23 / 25, 35 / 25; 512 x 512 8 / 16 rows 11 / 14, 21 / 13; 4096 x 14336 one row 39 / 51, two 66 / 51; group 32 one row 182 / 57.
bool gptq_order_wanted(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    if (k > 32768 || n % 8 || k % 32 || kernel_disabled("gptq_order")) return false;
    const bool f32 = lhs_dtype == QMM_F32;
    const double kk = k / 1024.0, w = (double)n * k / (1 << 20);
    const double rows[4] = {0.0, 1.0, f32 ? 1.06 : 1.45, f32 ? 1.42 : 1.7};  // a pass of that many, over a pass of one
    double one = 1.9 + 2.75 * kk * std::max(1.0, n / (64.0 * compute_units())) + 0.06 * w;
    if (!gptq_act_order_table_fits(m, k, group)) one *= f32 ? 1.9 : 3.0;
    const double look_up = one * ((m / 4) * rows[3] + rows[std::min<int64_t>(m % 4, 3)]);
    return look_up > 13.0 + 2.1 * kk + 0.31 * w + 0.12 * (n / 1024.0);
}

hipError_t launch_gptq_order(const void* lhs, int lhs_dtype, const uint32_t* qweight, const int32_t* g_idx, int64_t m, int64_t n, int64_t k, int group,
                             const GptqOrderSpace& p, hipStream_t s) {
    const int groups = (int)(k / group);
    int bits = 0;
    while ((1 << bits) < groups) bits++;
    hipError_t e = allow_full_lds<gptq_order_sort_kernel>();
    if (e != hipSuccess) return e;
    gptq_order_sort_kernel<<<dim3(1), dim3(64 * kSortWaves), (size_t)(kSortWaves * groups + 1) * 4, s>>>(g_idx, (int)k, group, bits, p.source, p.uneven);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // columns per workgroup: the most (whole cache lines with 32) with which two workgroups fit a compute unit
#define QMM_GO(AT, COLS)                                                                                                                                  \
    do {                                                                                                                                                  \
        const int per_xcd = (int)((n + 8 * COLS - 1) / (8 * COLS));                                                                                       \
        if ((e = allow_full_lds<gptq_order_permute_kernel<AT, COLS>>()) != hipSuccess) return e;                                                          \
        gptq_order_permute_kernel<AT, COLS><<<dim3((unsigned)(8 * per_xcd + m)), dim3(512), (size_t)k * COLS / 2, s>>>(                                    \
            qweight, (const AT*)lhs, (int)n, (int)k, per_xcd, p.source, p.qweight, (AT*)p.lhs);                                                           \
    } while (0)
#define QMM_GO_COLS(AT)                              \
    do {                                             \
        if (k <= kLdsPerCu / 32) QMM_GO(AT, 32);     \
        else if (k <= kLdsPerCu / 16) QMM_GO(AT, 16); \
        else QMM_GO(AT, 8);                          \
    } while (0)
    if (lhs_dtype == QMM_F32) QMM_GO_COLS(float);
    else QMM_GO_COLS(uint16_t);
#undef QMM_GO_COLS
#undef QMM_GO
    return hipGetLastError();
}

}  // namespace qmm
