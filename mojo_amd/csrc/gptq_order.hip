// Act-order GPTQ checkpoints (desc_act = True) with several lhs rows: the columns of K sorted by group, so that the kernels for plain
// groups serve the call.
//
// The kernel that looks the group of every k up (gemv_gptq.hip) passes over the weights once per four rows and multiplies on the vector
// units: 14336 x 4096 with 400 bf16 rows took 2.4 ms, this way 75 us.  Sorting costs one launch and one pass over the packed weights: a workgroup holds some
// columns of the output in LDS (all of K), sorts the columns of K by group while those are on their way, and takes the eight nibbles of every word of the sorted
// matrix from there.  Workgroups of the same launch hold rows of the lhs there instead and leave the operands of the direct GEMM in the same order; where the launch has no room for them,
// that GEMM's own preparation does.
// What bounds the pass, at 14336 x 4096 (2 x 29 MB and 400 rows of the lhs, 18 us in a trace with nothing in the caches, 3.6 TB/s): loads (the sort hides behind them but for its start), nibbles (about 2 us) and stores one
// after the other, since all workgroups run at once.
// us of the whole call with the sort as a launch of its own and a sorted copy of the lhs / this way, nothing in the caches: 14336 x 4096 400 rows 127 / 122, 8 rows 50 / 44;
// 4096 x 14336 64 rows 76 / 63; 4096 x 4096 64 rows 37 / 30; 8192 x 8192 300 rows 130 / 123; 1024 x 4096 20 rows 29 / 22; 8192 x 28672 20 rows 184 / 174;
// 3584 x 18944 33 rows 90 / 90.  With the lhs as a launch of its own / in the same one: 14336 x 4096 400 rows 81.5 / 77.6, 8 rows 36.5 / 32.9, 100 fp32 rows 56.7 / 52.0; 4096 x 4096
// 64 rows 25.0 / 24.3; 1024 x 4096 20 rows 17.4 / 14.6; 3584 x 18944 33 rows 68.4 / 63.9; 2560 x 9088 9 fp32 rows 38.4 / 33.3; 28672 x 8192 40 rows 108.7 / 107.0.
//
// A sorted column list is a plain-group matrix only if every group has exactly group_size columns, which is so in any checkpoint that was
// quantised group by group.  The device finds out: where it is not so, the sort leaves a mark, the order as it was (the products are then
// meaningless) and the look-up kernel, launched behind them, replaces the whole result; otherwise that launch returns at once.
#include <algorithm>

#include "gemm_direct.h"
#include "lds_stream.h"
#include "qmm_internal.h"

namespace qmm {

namespace {

typedef uint32_t go_u4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 16, kThreads = 64 * kWaves;

// The lhs: its rows (the first workgroups of the grid), where their operands and inverse scales go, and the results that are added to (the next ones zero them).
struct OrderLhs {
    const void* a;
    _Float16* a16;
    float* inv;
    int m, workgroups, zeroing;  // multiples of 8
    DirectMats zero;
};
struct __attribute__((packed, aligned(4))) OrderWords {  // (qweight begins at any multiple of four)
    go_u4 v;
};
constexpr int lhs_rows(int cols, int size) { return cols / (size == 4 ? 8 : 4); }  // of a workgroup: as many bytes as its words of the weights

// The bits of a row's largest magnitude, of the finite ones, by one wavefront: every wavefront of a row for itself (LDS is full of words and order).
template <typename AT>
__device__ __forceinline__ uint32_t wave_largest(const AT* x, int k, int lane) {
    uint32_t top = 0;
    for (int pc = lane; pc < k >> 3; pc += 64) top = largest_bits(top, load_piece(x + pc * 8));
    float mx = largest_of<AT>(top);
    if (any_not_finite(mx)) {
        mx = 0.0f;
        for (int pc = lane; pc < k >> 3; pc += 64) mx = largest_finite(mx, load_piece(x + pc * 8));
    }
    return wave_max_nonneg_bits(mx);
}

// Eight words of eight nibbles: nibble j of word i and nibble i of word j change places.
__device__ __forceinline__ void transpose_nibbles(uint32_t (&a)[8]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t lo = a[i], hi = a[i + 4];
        a[i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        a[i + 4] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
    }
#pragma unroll
    for (int i = 0; i < 6; i += i == 1 ? 3 : 1) {
        const uint32_t lo = a[i], hi = a[i + 2];
        a[i] = __builtin_amdgcn_perm(hi, lo, 0x06020400u);
        a[i + 2] = __builtin_amdgcn_perm(hi, lo, 0x07030501u);
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const uint32_t lo = a[i], hi = a[i + 1];
        a[i] = (lo & 0x0f0f0f0fu) | ((hi << 4) & 0xf0f0f0f0u);
        a[i + 1] = ((lo >> 4) & 0x0f0f0f0fu) | (hi & 0xf0f0f0f0u);
    }
}
// LDS holds, for every column of K, the nibbles of the slab's columns of N side by side.  Where column k lies, in such rows: the eight of a word are exchanged, so that the
// wavefronts that write them use all banks.  Its own inverse.
template <int COLS>
__device__ __forceinline__ uint32_t place_of(uint32_t k) { return k ^ ((k >> (COLS == 32 ? 4 : COLS == 16 ? 5 : 6)) & 7u); }

// How the nibbles are taken.  Turned: the words go through registers on their way to LDS and are transposed there, eight columns of K by eight of N; a word of the sorted matrix is then eight
// dwords transposed back: 1.4 vector instructions a nibble, 3 where every nibble is shifted out of a word as it came (loads go straight to LDS then).  Against that, us of the whole call, as
// they come / turned: 14336 x 4096 400 rows 77.6 / 74.6, 8 rows 32.9 / 31.1, 100 fp32 rows 52.0 / 48.0; 4096 x 4096 64 rows 24.3 / 23.6; 28672 x 8192 40 rows 107.0 / 100.9; 5120 x 20480 64
// rows 90.6 / 87.9; 8192 x 8192 500 rows (32 columns, 128 registers) 96.9 / 92.7.  Not for slabs of 8 columns, whose loads would be 16 bytes a row and instruction (1024 x 4096 2000 rows 45.1 / 45.9,
// 8192 x 28672 300 rows 271 / 280), and not with eight turns and two workgroups a compute unit: 64 registers do not hold the words beside the groups (8192 x 8192 with spills 98 / 104).
constexpr bool order_turned(int cols, int turns) { return cols > 8 && turns != 8; }

// Workgroup: COLS columns of the weights, neighbours on one XCD (they share cache lines).  It sorts for itself while its words are on their way to LDS: where the
// sort was a launch of one workgroup it took 6.6 us at K = 4096 and 18 at 14336.
// Stable sort (within a group the columns keep their order), wavefront w takes a sixteenth of K, TURNS times 64 columns; group indices outside [0, groups) are
// clamped, as in the look-up kernel.  The first workgroup leaves the order (source[p]: the column of K at sorted position p) and the mark in memory.
// LDS: [k / 8][COLS] words (turned: [k][COLS / 8], see place_of), uint16 [k] order, uint16 [kWaves][groups] counts.
// Where that is more than a compute unit has (K beyond 26208, less with groups of 32 or 64), or leaves room for one workgroup and there are several for each compute unit: a launch of
// one workgroup without words (qweight null) that only sorts, then TURNS = 0, which takes the order from memory.
template <typename AT, int COLS, int TURNS>
__global__ __launch_bounds__(kThreads, TURNS <= 8 ? 8 : 4) void gptq_order_kernel(const uint32_t* __restrict__ qweight, const int32_t* __restrict__ g_idx, int n, int k, int group, int bits,
                                                                                  int per_xcd, int32_t* __restrict__ source, int32_t* __restrict__ uneven,
                                                                                  uint32_t* __restrict__ sorted_w, OrderLhs lhs) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr bool kTurned = order_turned(COLS, TURNS);
    constexpr int kPieces = COLS / (kTurned ? 8 : 4), kRows = kThreads / kPieces;  // threads to a row of words, rows a turn
    constexpr int kHeld = TURNS == 0 ? 2 : COLS == 32 && TURNS == 16 ? 5 : (TURNS * COLS + 63) / 64;  // turns of words in registers while the sort runs
    constexpr int kLhsRows = lhs_rows(COLS, sizeof(AT)), kRowWaves = kWaves / kLhsRows;
    const int b = (int)blockIdx.x - lhs.workgroups - lhs.zeroing, slab = ((b & 7) * per_xcd + (b >> 3)) * COLS;
    if (b >= 0 && slab >= n) return;
    if (b < 0 && b >= -lhs.zeroing) {
        zero_out(lhs.zero, lhs.m, b + lhs.zeroing, lhs.zeroing);
        return;
    }
    // (rows of one group of eight on one XCD: a 128-byte line of an operand holds eight rows)
    const bool of_lhs = b < 0;
    const int turn = (int)blockIdx.x >> 3, row0 = (turn / (8 / kLhsRows) * 8 + ((int)blockIdx.x & 7)) * 8 + turn % (8 / kLhsRows) * kLhsRows;
    if (of_lhs && row0 >= lhs.m) return;
    const int col = slab + (kTurned ? 8 : 4) * (tid & (kPieces - 1)), rows = qweight ? k >> 3 : 0, r0 = tid / kPieces, groups = k / group;
    const bool in_n = col < n;  // (N is a multiple of 8)
    uint16_t* const order = (uint16_t*)(smem + (size_t)rows * COLS * 4);
    uint16_t* const counts = order + k;
    uint32_t* const pairs = (uint32_t*)counts;  // (k is even)
    uint32_t* const bad = (uint32_t*)order;     // until the order is written

    auto place = [&](uint32_t src) __attribute__((always_inline)) { return kTurned && !of_lhs ? place_of<COLS>(src) : src; };
    uint32_t* const nibbles = (uint32_t*)smem + (tid & (kPieces - 1));
    OrderWords held[kHeld][2];
    auto load_words = [&](int turn0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kHeld; i++) {
            const uint32_t* const from = qweight + (int64_t)min((turn0 + i) * kRows + r0, rows - 1) * n + min(col, n - 8);
            held[i][0] = *(const OrderWords*)from;
            held[i][1] = *(const OrderWords*)(from + 4);
        }
    };
    auto spread_words = [&](int turn0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kHeld; i++) {
            const int r = (turn0 + i) * kRows + r0;
            if (r < rows) {
                uint32_t a[8];
#pragma unroll
                for (int c = 0; c < 4; c++) a[c] = held[i][0].v[c], a[4 + c] = held[i][1].v[c];
                transpose_nibbles(a);
                const uint32_t mixed = place_of<COLS>(8 * r) & 7u;
#pragma unroll
                for (int c = 0; c < 8; c++) nibbles[(8 * r + (c ^ mixed)) * kPieces] = a[c];
            }
        }
    };
    auto load_16s = [&](const uint8_t* from, int bytes) __attribute__((always_inline)) {  // (of the lhs)
        for (int i = 0; i * (kThreads * 16) < bytes; i++)
            if (i * (kThreads * 16) + tid * 16 < bytes) load16_to_lds(from + i * (kThreads * 16) + tid * 16, lds_address(smem) + wave * 1024 + i * (kThreads * 16));
    };
    auto load_lds = [&]() __attribute__((always_inline)) {
        if (of_lhs) {
            load_16s((const uint8_t*)lhs.a + (int64_t)row0 * k * sizeof(AT), min(kLhsRows, lhs.m - row0) * k * (int)sizeof(AT));
        } else if constexpr (!kTurned) {
            const uint32_t* const from = qweight + (in_n ? col : 0);
            for (int i = 0; i * kRows < rows; i++)
                if (i * kRows + r0 < rows) load16_to_lds(from + (int64_t)(i * kRows + r0) * n, lds_address(smem) + wave * 1024 + i * (kThreads * 16));
        }
    };
    if constexpr (TURNS == 0) {
        if (of_lhs || !kTurned) {
            load_lds();
            wait_vmcnt<0>();
        } else {
            for (int turn = 0; turn * kRows < rows; turn += kHeld) {
                load_words(turn);
                spread_words(turn);
            }
        }
        __syncthreads();
    } else {
        // (asked for before the words: a wait for these would be one for everything asked for earlier)
        const int per = (k + 64 * kWaves - 1) / (64 * kWaves) * 64, lo = wave * per;
        int g[TURNS];
    #pragma unroll
        for (int t = 0; t < TURNS; t++) g[t] = g_idx[min(lo + 64 * t + lane, k - 1)];
        for (int i = tid; i < (kWaves * groups + 1) / 2; i += kThreads) pairs[i] = 0;
        if (tid == 0) *bad = 0;
    #pragma unroll
        for (int t = 0; t < TURNS; t++) {
            g[t] = min(max(g[t], 0), groups - 1);
            tie(g[t]);
        }
        if (of_lhs || !kTurned) load_lds();
        else load_words(0);

        const int turns = min(per, max(0, k - lo));  // columns of this wavefront
        __syncthreads();
    #pragma unroll
        for (int t = 0; t < TURNS; t++)
            if (64 * t + lane < turns) {
                const int at = wave * groups + g[t];
                atomicAdd(pairs + (at >> 1), 1u << (16 * (at & 1)));
            }
        __syncthreads();
        for (int i = tid; i < groups; i += kThreads) {  // where each wavefront's columns of the group begin
            uint32_t c[kWaves], at = 0;
    #pragma unroll
            for (int w = 0; w < kWaves; w++) c[w] = counts[w * groups + i];
    #pragma unroll
            for (int w = 0; w < kWaves; w++) {
                counts[w * groups + i] = (uint16_t)at;
                at += c[w];
            }
            if (at != (uint32_t)group) *bad = 1;
        }
        __syncthreads();
        const bool as_is = *bad != 0;
        __syncthreads();
        if (as_is) {
            for (int i = tid; i < k; i += kThreads) order[i] = (uint16_t)place(i);
        } else {
            uint16_t* const mine = counts + wave * groups;
    #pragma unroll
            for (int t = 0; t < TURNS; t++) {
                if (64 * t >= turns) break;
                const bool live = 64 * t + lane < turns;
                uint64_t same = __ballot(live);  // the lanes with this lane's group
                for (int bit = 0; bit < bits; bit++) {
                    const bool set = (g[t] >> bit) & 1;
                    const uint64_t with = __ballot(set);
                    same &= set ? with : ~with;
                }
                const int rank = __popcll(same & ((1ull << lane) - 1)), count = __popcll(same);
                if (live) {
                    const uint32_t at = mine[g[t]];
                    order[g[t] * group + (int)at + rank] = (uint16_t)place(lo + 64 * t + lane);
                    if (rank == count - 1) mine[g[t]] = (uint16_t)(at + (uint32_t)count);
                }
                // (the next turn of this wavefront reads what its lanes wrote: LDS operations of a wavefront are performed in order)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (of_lhs || !kTurned) wait_vmcnt<0>();
        else spread_words(0);
        __syncthreads();
        if (b == 0) {
            if (tid == 0) *uneven = as_is;
            if (source)
                for (int i = tid; i < k; i += kThreads) source[i] = (int32_t)place(order[i]);
        }
    }
    auto sources = [&](int r) __attribute__((always_inline)) {  // of sorted columns 8 r .. 8 r + 7
        if constexpr (TURNS == 0) {
            const go_u4 s0 = *(const go_u4*)(source + 8 * r), s1 = *(const go_u4*)(source + 8 * r + 4);
            return go_u4{s0.x | s0.y << 16, s0.z | s0.w << 16, s1.x | s1.y << 16, s1.z | s1.w << 16};
        } else {
            return *(const go_u4*)(order + 8 * r);
        }
    };
    if (of_lhs) {
        const int row = row0 + wave / kRowWaves, pieces = k >> 3, steps = (k + 255) / 256 * 16;
        if (row >= lhs.m) return;
        const AT* const x = (const AT*)smem + wave / kRowWaves * k;
        float v[8], inv;
        const float scale = row_scale(wave_largest(x, k, lane), kRowTop, inv);
        if (wave % kRowWaves == 0 && lane == 0) lhs.inv[row] = inv;
        for (int pc = wave % kRowWaves * 64 + lane; pc < 2 * steps; pc += 64 * kRowWaves) {  // (zeros up to a whole unit)
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = 0.0f;
            if (pc < pieces) {
                const go_u4 s = sources(pc);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const AT y = x[(j & 1) ? s[j >> 1] >> 16 : s[j >> 1] & 0xffffu];
                    if constexpr (sizeof(AT) == 4) v[j] = y;
                    else v[j] = __uint_as_float((uint32_t)y << 16);
                }
            }
            store_piece<AT, kOrderGptq>(lhs.a16, steps, row, pc, scale, v);
        }
        return;
    }
    if (!in_n) return;
#pragma unroll 2
    for (int r = r0; r < rows; r += kRows) {
        const go_u4 s = sources(r);
        go_u4* const to = (go_u4*)(sorted_w + (int64_t)r * n + col);
        if constexpr (kTurned) {
            uint32_t a[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t src = (j & 1) ? s[j >> 1] >> 16 : s[j >> 1] & 0xffffu;
                a[j] = nibbles[(TURNS == 0 ? place(src) : src) * kPieces];
            }
            transpose_nibbles(a);
            to[0] = go_u4{a[0], a[1], a[2], a[3]};
            to[1] = go_u4{a[4], a[5], a[6], a[7]};
        } else {
            go_u4 o = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t src = (j & 1) ? s[j >> 1] >> 16 : s[j >> 1] & 0xffffu;
                const go_u4 x = *(const go_u4*)(smem + 16 * (tid & (kPieces - 1)) + (src >> 3) * (COLS * 4));
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = __builtin_amdgcn_alignbit(x[c] >> ((src << 2) & 31u), o[c], 4);
            }
            to[0] = o;
        }
    }
}

}  // namespace

GptqOrderSpace gptq_order_space(void* workspace, int64_t n, int64_t k) {
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    GptqOrderSpace p;
    char* base = (char*)workspace;
    p.uneven = (int32_t*)base;
    int64_t off = 256;
    p.source = (int32_t*)(base + off);
    off += up(k * 4);
    p.qweight = (uint32_t*)(base + off);
    off += up(n * k / 2);
    p.bytes = off;
    return p;
}

// The look-up kernel or the sort and the direct GEMM: the predicted time of both in microseconds.  The look-up kernel walks K with one workgroup per 64
// columns, in passes of up to four rows; where its table of scales does not fit LDS (small groups on a long K), every weight reads its
// scale from memory.  The sorted way is three launches (up to five where the lhs or the sort has one of its own) and one pass over the weights, whatever the number of rows up to 32.  Fitted to timings of
// 15 matrices (512 x 512 .. 28672 x 8192, groups of 32 and 128, weights from memory) with 1 .. 12 rows; what is taken, the second line included, takes 0.14 % longer on
// average than the faster of the two (profiles/gptq_act_order__look_up_against_sorted.txt, 576 calls, from when the lhs had a launch of its own and nibbles were sorted one by one: the sorted way has become 4 .. 8 us
// cheaper, and up to a fifth is lost near the line).  us, look-up / sorted, now: 14336 x 4096 4 bf16 rows 29.9 / 30.2, 5 rows 42.9 / 29.9, fp32 4 rows 21.1 / 32.0, 6 rows 39.2 / 32.2; 11008 x 4096 4 bf16 rows
// 27.9 / 28.5; 4096 x 4096 2 / 3 bf16 rows 21.9 / 17.7, 26.6 / 17.9; 8192 x 8192 4 rows 57.8 / 39.2; 512 x 512 8 / 12 fp32 rows 9.7 / 10.0, 14.8 / 10.0; 1024 x 14336 one bf16 row 40 / 32.5, one fp32 row 41.9 / 37.1.
bool gptq_order_wanted(int lhs_dtype, int64_t m, int64_t n, int64_t k, int group) {
    if (k > 32768 || n % 8 || k % 32 || kernel_disabled("gptq_order")) return false;
    const bool f32 = lhs_dtype == QMM_F32;
    const double kk = k / 1024.0, w = (double)n * k / (1 << 20);
    const double rows[4] = {0.0, 1.0, f32 ? 1.06 : 1.7, f32 ? 1.42 : 1.7};  // a pass of that many, over a pass of one
    double one = 1.9 + 2.75 * kk * std::max(1.0, n / (64.0 * compute_units())) + 0.06 * w;
    if (!gptq_act_order_table_fits(m, k, group)) one *= f32 ? 1.9 : 3.0;
    const double look_up = one * ((m / 4) * rows[3] + rows[std::min<int64_t>(m % 4, 3)]);
    // Beyond some 60 M weights that line finds the look-up kernel ahead with one row more or two, but there it is two to four times further off: the second line, from when
    // the sort was a launch of its own.  Relative error, us, look-up / sorted: 5504 x 18944 4 fp32 rows 5.7e-7 / 1.3e-7, 99 / 79; 18944 x 4096 6 rows 2.8e-7 / 1.2e-7,
    // 69 / 48; groups of 32, 11648 x 12032 2 rows 4.7e-7 / 1.5e-7, 83 / 87; 32000 x 28672 4 bf16 rows 6.1e-7 / 1.4e-7, 419 / 479.
    return look_up > std::min(11.0 + (f32 ? 1.8 : 1.5) * kk + (f32 ? 0.40 : 0.35) * w, 13.0 + 2.1 * kk + 0.31 * w + 0.12 * (n / 1024.0));
}

// How many workgroups zero results beside those of the lhs (`rows` rows each) and `slabs` others, in a launch of which the part takes `at_once`; -1: the lhs has a launch of its own.  zeros: results of the
// largest matrix that is added to.
// Workgroups go to the eight XCDs in turn, and there to four groups of compute units in turn, whichever of those is free: one long workgroup more than a group has places for costs the time of a slab.  Those
// that zero, and those of the lhs beyond its rows, end at once, but count in turn; so their number decides where the others go, and a few with nothing to do may help.  us by that number: 7840 x 5504 18 bf16 rows (31 slabs and a workgroup of
// the lhs for the 32 places of an XCD) 8 / 16 / 32 / 40 36.1 / 36.0 / 29.3 / 35.9, 7400 x 8832 29 rows 8 / 16 / 32 / 56 41.7 / 41.8 / 41.9 / 57, 7560 x 8064 13 rows 8 / 16 / 24 35.6 / 48.9 / 48.8.  Of 5048 ways to launch 210
// calls 5022 are faster or slower than with a launch for the lhs as this has them.  That launch costs 4 .. 7 us (14336 x 4096 400 rows 69 / 74, 5120 x 20480 64 rows 88 / 95), less than a slab (4096 x 14336 400
// rows 101 / 93, 4056 x 18176 13 rows 70 / 63, 6984 x 25088 2283 rows 1013 / 919); two to a compute unit and in several rounds they end at different times, and one more costs less (24440 x 8192 42 rows 100 / 104,
// 30688 x 5120 1126 rows 388 / 397; of 60 such calls none took longer so).
int order_lhs_room(int64_t slabs, int64_t at_once, int64_t m, int64_t rows, int64_t zeros) {
    // of the first XCD, which has as many as any
    const int64_t own = (slabs + 7) / 8, places = std::max<int64_t>(1, at_once / 32), turns = (m + 63) / 64 * (8 / rows), live = m / 64 * (8 / rows) + (std::min<int64_t>(m % 64, 8) + rows - 1) / rows;
    const int64_t wanted = (std::min<int64_t>(1024, (zeros + 4095) / 4096) + 7) / 8 * 8, alone = ((own + 3) / 4 + places - 1) / places;
    if (alone > 1 && at_once > compute_units()) return (int)wanted;
    for (int64_t zeroing = wanted; zeroing < wanted + 32; zeroing += 8) {
        int64_t most = 0;
        for (int64_t e = 0; e < 4; e++) most = std::max(most, (live - e + 3) / 4 + (own - ((e - turns - zeroing / 8) & 3) + 3) / 4);
        if ((most + places - 1) / places == alone) return (int)zeroing;
    }
    return -1;
}

hipError_t launch_gptq_order(const GptqOrder& order, int64_t n, int64_t k, int group, const void* a, int lhs_dtype, int64_t m, const DirectSpace& p, const DirectMats& zero,
                             int64_t zeros, bool& lhs_done, hipStream_t s) {
    const int groups = (int)(k / group);
    int bits = 0;
    while ((1 << bits) < groups) bits++;
    const size_t sort_lds = 2 * k + (2 * kWaves * groups + 3) / 4 * 4;
    auto words = [&](int cols) { return (size_t)(k / 2 * cols); };
    // The widest slab that fits a compute unit (a row of 32 words is a whole cache line), narrower ones where those still are no more than one for each.  us of the
    // whole call, 32 / 16 / 8 / 4 columns: 14336 x 4096 400 rows 123 / 126 / 133 / 152, 8192 x 8192 300 rows 125 / 131 / 133 / 151, 4096 x 14336 64 rows - / 64 / 75 / 99,
    // 4096 x 4096 64 rows 32.5 / 29.9 / 32.3 / 37.2, 1024 x 4096 20 rows 24.3 / 22.3 / 21.4 / 21.4; 12 rows 6144 x 8192 42.6 / 49.2 / 48.2, 2560 x 9088 - / 41.3 / 48.4.
    int cols = 32;
    while (cols > 8 && (words(cols) + sort_lds > kLdsPerCu || n <= (int64_t)cols / 2 * compute_units())) cols /= 2;
    // Several slabs for each compute unit, of which it holds one with the order: nothing is asked for while one is being sorted and permuted.  Without the order two
    // fit.  us, 12 rows, one launch / two: 28672 x 16384 393 / 261, 11008 x 18944 205 / 139, 14336 x 9088 97 / 81, 28672 x 8192 127 / 117, 14336 x 8192 72.5 / 73.4;
    // with one slab for each the other way round: 4096 x 14336 54 / 60 (and up to one and a half of 32 columns: 11008 x 5120 49.4 / 51.3).
    const bool sort_apart = words(cols) + sort_lds > kLdsPerCu ||
                            (2 * (words(cols) + sort_lds) > kLdsPerCu && n > (int64_t)(cols == 32 ? 48 : cols) * compute_units());
    if (sort_apart) cols = k <= 5120 ? 32 : k <= 20480 ? 16 : 8;  // (32 up to where two fit, 28672 x 5120 32 / 16 columns 78.5 / 80.4; 16 up to where one does, 14336 x 20480 16 / 8 165 / 175)
    const unsigned per_xcd = (unsigned)((n + 8 * cols - 1) / (8 * cols));
    // The lhs in the same launch where that takes no longer (order_lhs_room); otherwise the caller's preparation reads its rows in the order left in memory.
    const bool f32 = lhs_dtype == QMM_F32;
    const int64_t lds = words(cols) + (sort_apart ? 0 : sort_lds), at_once = compute_units() * (2 * lds <= kLdsPerCu && (sort_apart || k <= 8192) ? 2 : 1);
    const int rows = lhs_rows(cols, f32 ? 4 : 2), zeroing = order_lhs_room((n + cols - 1) / cols, at_once, m, rows, zeros);
    lhs_done = zeroing >= 0;
    const OrderLhs none{};
    const OrderLhs lhs{a, p.a16, p.inv, (int)m, (int)((m + 63) / 64 * 64 / rows), std::max(zeroing, 0), zero};
    int32_t* const source = sort_apart || !lhs_done ? order.space.source : nullptr;
    hipError_t e;
#define QMM_GO(AT, COLS, TURNS, WORDS, GRID, LDS, LHS)                                                                                                                  \
    do {                                                                                                                                                                \
        if ((e = allow_full_lds<gptq_order_kernel<AT, COLS, TURNS>>()) != hipSuccess) return e;                                                                         \
        gptq_order_kernel<AT, COLS, TURNS><<<dim3(GRID), dim3(kThreads), LDS, s>>>(WORDS, order.g_idx, (int)n, (int)k, group, bits, (int)per_xcd, source,               \
                                                                                   order.space.uneven, order.space.qweight, LHS);                                       \
    } while (0)
#define QMM_GO_WORDS(COLS, TURNS)                                                                                                          \
    do {                                                                                                                                   \
        const unsigned grid = 8 * per_xcd + (lhs_done ? (unsigned)(lhs.workgroups + lhs.zeroing) : 0u);                                    \
        if (!lhs_done) QMM_GO(uint16_t, COLS, TURNS, order.qweight, grid, lds, none);                                                      \
        else if (f32) QMM_GO(float, COLS, TURNS, order.qweight, grid, lds, lhs);                                                           \
        else QMM_GO(uint16_t, COLS, TURNS, order.qweight, grid, lds, lhs);                                                                 \
    } while (0)
    if (sort_apart) {
        QMM_GO(uint16_t, 8, 32, nullptr, 1, sort_lds, none);
        if (cols == 32) QMM_GO_WORDS(32, 0);
        else if (cols == 16) QMM_GO_WORDS(16, 0);
        else QMM_GO_WORDS(8, 0);
    } else if (cols == 32) {  // (fits up to K = 9100)
        if (k <= 4096) QMM_GO_WORDS(32, 4);
        else if (2 * (words(32) + sort_lds) <= kLdsPerCu) QMM_GO_WORDS(32, 8);
        else QMM_GO_WORDS(32, 16);
    } else if (cols == 16) {  // (up to K = 16380)
        if (k <= 4096) QMM_GO_WORDS(16, 4);
        else if (k <= 8192) QMM_GO_WORDS(16, 8);
        else QMM_GO_WORDS(16, 16);
    } else {
        if (k <= 4096) QMM_GO_WORDS(8, 4);
        else if (k <= 8192) QMM_GO_WORDS(8, 8);
        else if (k <= 16384) QMM_GO_WORDS(8, 16);
        else QMM_GO_WORDS(8, 32);
    }
#undef QMM_GO_WORDS
#undef QMM_GO
    return hipGetLastError();
}

}  // namespace qmm
