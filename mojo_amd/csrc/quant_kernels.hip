// Block unpack / dequantise kernels and the quantisers (fp32 -> packed blocks).
//
// Layouts are the on-disk GGUF ones (ggml-common.h) and AutoGPTQ v1 tensors.
// The quantisers are written as separate IEEE multiplies, adds and divides
// (this file is compiled with -ffp-contract=off) so that their packed output is
// bit-identical to a scalar CPU evaluation of the same formulas.
#include "qmm_internal.h"

namespace qmm {

// ---------------------------------------------------------------------------
// dequantise: bound by the stores (2 or 4 bytes out for 0.56 .. 0.82 in)
// ---------------------------------------------------------------------------
// A lane owns V consecutive elements (8 of a bf16 output, 4 of an fp32 one: 16 bytes), so that a wavefront stores 1 KB in one
// instruction, and always the same place of a block: the field offsets and shifts are set once per lane, and the lanes of a
// block read its header and codes from the same cache lines.  (One element per lane, byte loads and 2-byte stores: 14336 x 4096
// Q4_K to bf16 took 130 us.)  What four steps load is asked for before the first of them is used, behind no branch, and bf16 pairs are made by one instruction.  us, a wait behind each load and
// a branch for the NaN of each value / this way, 14336 x 4096 to fp32 and bf16: Q4_0 53.9 / 50.7 and 31.0 / 27.5, Q4_K 64.7 / 50.4 and 40.7 / 28.1, Q5_K 67.1 / 52.1 and 41.8 / 30.3, Q6_K 54.4 / 51.9 and
// 35.4 / 32.1; with the output where the last call left it, Q4_K to bf16 26.0 / 22.7 (6.6 TB/s).

typedef uint32_t dq_u4 __attribute__((ext_vector_type(4)));
typedef float dq_f4 __attribute__((ext_vector_type(4)));

// V bytes at an address of any alignment
template <int V>
struct Codes {
    uint32_t w[V / 4];
    __device__ __forceinline__ explicit Codes(const uint8_t* p) { __builtin_memcpy(w, p, V); }
};
__device__ __forceinline__ float code_f32(const uint32_t* w, int i) { return (float)byte_of(w[i >> 2], i & 3); }

__device__ __forceinline__ uint32_t bf16_pair(float x, float y) { return f2bf2(x, y); }

__device__ __forceinline__ void store_elems(float* out, const float (&v)[4]) { __builtin_nontemporal_store(dq_f4{v[0], v[1], v[2], v[3]}, (dq_f4*)out); }
__device__ __forceinline__ void store_elems(uint16_t* out, const float (&v)[8]) {
    __builtin_nontemporal_store(dq_u4{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]), bf16_pair(v[4], v[5]), bf16_pair(v[6], v[7])}, (dq_u4*)out);
}

// Elements pos .. pos + V - 1 of the block at b: what is loaded for them, and what it means.
template <int ENC, int V>
struct Elems {  // Q4_K, Q5_K (blocks are 16-byte aligned)
    dq_u4 hdr;
    Codes<V> c, fifth;
    __device__ __forceinline__ Elems(const uint8_t* b, int pos)
        : hdr(*(const dq_u4*)b), c(b + (ENC == QMM_Q4_K ? 16 : 48) + 32 * (pos >> 6) + (pos & 31)), fifth(b + (ENC == QMM_Q5_K ? 16 : 0) + (pos & 31)) {}
    __device__ __forceinline__ void values(int pos, float (&v)[V]) const {
        const int j = pos >> 5, shift = 8 * (j & 3);
        const uint32_t late = (uint32_t)((3 - j) >> 31);
        // (q4k_scale_min without a branch: half of a block's lanes are on either side of it)
        const uint32_t s0 = (hdr.y >> shift) & 255u, s1 = (hdr.z >> shift) & 255u, s2 = (hdr.w >> shift) & 255u;
        const uint32_t sc = (s0 & 63u & ~late) | (((s2 & 15u) | ((s0 >> 6) << 4)) & late),
                       mn = (s1 & 63u & ~late) | (((s2 >> 4) | ((s1 >> 6) << 4)) & late);
        const float ds = h2f((uint16_t)(hdr.x & 0xffffu)) * (float)sc, dm = h2f((uint16_t)(hdr.x >> 16)) * (float)mn;
#pragma unroll
        for (int i = 0; i < V / 4; i++) {
            uint32_t w[1] = {(c.w[i] >> (j & 1 ? 4 : 0)) & 0x0f0f0f0fu};
            if constexpr (ENC == QMM_Q5_K) w[0] |= ((fifth.w[i] >> j) & 0x01010101u) << 4;
#pragma unroll
            for (int e = 0; e < 4; e++) v[4 * i + e] = ds * code_f32(w, e) - dm;
        }
    }
};

template <int V>
struct Elems<QMM_Q4_0, V> {
    uint16_t d;
    Codes<V> c;
    __device__ __forceinline__ Elems(const uint8_t* b, int pos) : c(b + 2 + (pos & 15)) { __builtin_memcpy(&d, b, 2); }
    __device__ __forceinline__ void values(int pos, float (&v)[V]) const {
        const float df = h2f(d);
        const uint32_t shift = pos & 16 ? 4 : 0;
#pragma unroll
        for (int i = 0; i < V; i++) v[i] = ((float)((c.w[i >> 2] >> (shift + 8 * (i & 3))) & 15u) - 8.0f) * df;
    }
};

template <int V>
struct Elems<QMM_Q6_K, V> {
    uint16_t d;
    int8_t scale;
    Codes<V> lo, hi;
    __device__ __forceinline__ Elems(const uint8_t* b, int pos)
        : scale(((const int8_t*)b)[192 + (pos >> 4)]), lo(b + 64 * (pos >> 7) + 32 * ((pos >> 5) & 1) + (pos & 31)), hi(b + 128 + 32 * (pos >> 7) + (pos & 31)) {
        __builtin_memcpy(&d, b + 208, 2);
    }
    __device__ __forceinline__ void values(int pos, float (&v)[V]) const {
        const int quarter = (pos >> 5) & 3;
        const float ds = h2f(d) * (float)scale;
#pragma unroll
        for (int i = 0; i < V / 4; i++) {
            const uint32_t w[1] = {((lo.w[i] >> (quarter & 2 ? 4 : 0)) & 0x0f0f0f0fu) | (((hi.w[i] >> (2 * quarter)) & 0x03030303u) << 4)};
#pragma unroll
            for (int j = 0; j < 4; j++) v[4 * i + j] = ds * (code_f32(w, j) - 32.0f);
        }
    }
};

template <int ENC, typename OutT>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ w, int64_t total, OutT* __restrict__ out) {
    constexpr int EPB = ENC == QMM_Q4_0 ? Q4_0_EPB : 256;
    constexpr int BPB = ENC == QMM_Q4_0 ? Q4_0_BPB : (ENC == QMM_Q4_K ? Q4_K_BPB : (ENC == QMM_Q5_K ? Q5_K_BPB : Q6_K_BPB));
    constexpr int V = 16 / sizeof(OutT), kStep = 256 * V, kAhead = 4;  // (a workgroup walks kAhead steps: their loads are in flight together)
    const int pos = (int)(threadIdx.x * V) % EPB;
    const int64_t first = (int64_t)blockIdx.x * (kStep * kAhead) + threadIdx.x * V;
    auto convert = [&](const Elems<ENC, V>& x, int64_t e) __attribute__((always_inline)) {
        float v[V];
        x.values(pos, v);
        store_elems(out + e, v);
    };
    if ((int64_t)(blockIdx.x + 1) * (kStep * kAhead) <= total) {
        const uint8_t* const b = w + first / EPB * BPB;
        constexpr int kBytes = kStep / EPB * BPB;
        const Elems<ENC, V> x0(b, pos), x1(b + kBytes, pos), x2(b + 2 * kBytes, pos), x3(b + 3 * kBytes, pos);
        __builtin_amdgcn_sched_barrier(0);
        convert(x0, first);
        convert(x1, first + kStep);
        convert(x2, first + 2 * kStep);
        convert(x3, first + 3 * kStep);
    } else {
        for (int64_t e = first; e < total; e += kStep) convert(Elems<ENC, V>(w + e / EPB * BPB, pos), e);
    }
}

// GPTQ: the output is the transpose of the stored words, so a workgroup turns a tile of 64 columns x 128 of K through LDS.  A lane
// unpacks words of one column (256-byte rows of qweight, scale and zero rows of 64 neighbouring columns: with g_idx the group of an
// element is the same for all of them) and the tile leaves in runs of 128 elements of an output row.  LDS rows are 16 bytes longer
// than the run, which spreads the 16-byte writes of neighbouring columns over all banks.  (One element per lane along K read a 4-byte
// word of a row of qweight each: 14336 x 4096 to bf16 138 us, g_idx 258 us.)  What a wavefront loads is asked for before the first of it is used (scale and zeros once for its four words): from
// memory 58.1 / 50.9 to fp32, 37.0 / 33.7 to bf16, 4096 x 4096 18.9 / 17.3 and 9.5 / 8.9.
template <typename OutT>
__global__ __launch_bounds__(256) void dequant_gptq_kernel(const uint32_t* __restrict__ qweight, const uint16_t* __restrict__ scales,
                                                           const uint32_t* __restrict__ qzeros, const int32_t* __restrict__ g_idx, int64_t n, int64_t k,
                                                           int group, OutT* __restrict__ out) {
    constexpr int V = 16 / sizeof(OutT), kRun = 128, kLine = kRun / V + 1;  // 16-byte pieces of an LDS row
    __shared__ dq_u4 tile[64 * kLine];
    const int tid = threadIdx.x, c = tid & 63;
    const int64_t n0 = (int64_t)blockIdx.x * 64, r0 = (int64_t)blockIdx.y * (kRun / 8), rows = k >> 3;
    const int64_t col = n0 + c < n ? n0 + c : n - 1;  // (columns past the end repeat the last one and are not stored)
    const int first = __builtin_amdgcn_readfirstlane(tid >> 6) * 4;
    const int shift = 4 * (int)(col & 7);
    // (all loads before the first use of any, rows past the end repeat the last one; groups are multiples of 32: without g_idx the four words of a wavefront lie in one)
    uint32_t word[4];
#pragma unroll
    for (int i = 0; i < 4; i++) word[i] = qweight[min(r0 + first + i, rows - 1) * n + col];
    const int64_t group0 = (int64_t)((uint32_t)min(r0 + first, rows - 1) * 8u / (uint32_t)group);
    const uint32_t zeros0 = g_idx ? 0u : qzeros[group0 * (n >> 3) + (col >> 3)];
    const uint16_t scale0 = g_idx ? 0 : scales[group0 * n + col];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t row = r0 + first + i;
        if (row >= rows) break;
        float v[8];
        if (g_idx) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int64_t g = g_idx[row * 8 + e];
                const int z = (int)((qzeros[g * (n >> 3) + (col >> 3)] >> shift) & 0xFu) + 1;
                v[e] = h2f(scales[g * n + col]) * (float)((int)((word[i] >> (4 * e)) & 0xFu) - z);
            }
        } else {
            const int z = (int)((zeros0 >> shift) & 0xFu) + 1;
            const float s = h2f(scale0);
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = s * (float)((int)((word[i] >> (4 * e)) & 0xFu) - z);
        }
        dq_u4* t = tile + c * kLine + (first + i) * (8 / V);
        if constexpr (sizeof(OutT) == 2) {
            t[0] = dq_u4{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]), bf16_pair(v[4], v[5]), bf16_pair(v[6], v[7])};
        } else {
            t[0] = dq_u4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
            t[1] = dq_u4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])};
        }
    }
    __syncthreads();
    constexpr int kPieces = kRun / V;  // of a row
    const int piece = tid % kPieces;
    if ((r0 + piece * V / 8) >= rows) return;
#pragma unroll 4
    for (int r = tid / kPieces; r < 64; r += 256 / kPieces)
        if (n0 + r < n) __builtin_nontemporal_store(tile[r * kLine + piece], (dq_u4*)(out + (n0 + r) * k + r0 * 8) + piece);
}

// Plain read of a buffer: the yardstick for the streaming kernels.  The xor keeps the loads alive;
// the store never happens for real data.  The access pattern is the best plain one measured on this
// part: a workgroup takes contiguous chunks of U x 4 KB (U 16-byte loads per lane in flight), chunk
// index grid-strided, loads marked non-temporal (a 453 MB buffer: 7.0 TB/s; without the mark 6.3,
// with a lane-level grid stride instead of contiguous chunks 5.0 to 5.7).
typedef uint32_t probe_u4 __attribute__((ext_vector_type(4)));
template <int U>
__global__ __launch_bounds__(256) void read_probe_kernel(const probe_u4* __restrict__ p, int64_t n16,
                                                         uint32_t* __restrict__ sink) {
    const int64_t chunk16 = (int64_t)U * 256, nchunks = n16 / chunk16;
    probe_u4 acc = {0, 0, 0, 0};
    for (int64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const probe_u4* q = p + c * chunk16 + threadIdx.x;
        probe_u4 v[U];
#pragma unroll
        for (int j = 0; j < U; j++) v[j] = __builtin_nontemporal_load(q + j * 256);
#pragma unroll
        for (int j = 0; j < U; j++) acc ^= v[j];
    }
    // the rest (less than one chunk), by the first workgroup
    if (blockIdx.x == 0)
        for (int64_t i = nchunks * chunk16 + threadIdx.x; i < n16; i += 256) {
            acc ^= __builtin_nontemporal_load(p + i);
        }
    if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x9E3779B9u && sink) sink[0] = acc.x;
}

hipError_t launch_read_probe(const void* buf, int64_t bytes, hipStream_t s) {
    const int64_t n16 = bytes / 16;
    // enough chunks for a thousand workgroups where the buffer allows it; at most 2048 workgroups
    const int u = bytes >= (32ll << 20) ? 8 : bytes >= (16ll << 20) ? 4 : bytes >= (8ll << 20) ? 2 : 1;
    int64_t grid = n16 / (256 * u);
    if (grid > 2048) grid = 2048;
    if (grid < 1) grid = 1;
    const dim3 g((unsigned)grid), b(256);
    if (u == 8) read_probe_kernel<8><<<g, b, 0, s>>>((const probe_u4*)buf, n16, nullptr);
    else if (u == 4) read_probe_kernel<4><<<g, b, 0, s>>>((const probe_u4*)buf, n16, nullptr);
    else if (u == 2) read_probe_kernel<2><<<g, b, 0, s>>>((const probe_u4*)buf, n16, nullptr);
    else read_probe_kernel<1><<<g, b, 0, s>>>((const probe_u4*)buf, n16, nullptr);
    return hipGetLastError();
}

// Eight values a lane where both sides lie at multiples of 16 bytes, one by one otherwise and for what is left.  us, a value at a time / this way, product and narrowing: Q4_K 14336 x 4096 2048 rows
// 308.8 / 295.0, Q6_K 4104 x 4096 1000 rows 101.7 / 98.7; from 4096 x 4096 with 300 rows down the launch is all there is.
__global__ __launch_bounds__(256) void f32_to_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ out, int64_t count) {
    const int64_t step = (int64_t)gridDim.x * 256, first = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t pieces = (((uintptr_t)x | (uintptr_t)out) & 15) == 0 ? count >> 3 : 0;
    for (int64_t i = first; i < pieces; i += step) {
        const dq_f4 a = ((const dq_f4*)x)[2 * i], b = ((const dq_f4*)x)[2 * i + 1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        store_elems(out + 8 * i, v);
    }
    for (int64_t i = 8 * pieces + first; i < count; i += step) out[i] = f2bf(x[i]);
}

hipError_t launch_f32_to_bf16(const float* x, uint16_t* out, int64_t count, hipStream_t s) {
    int64_t g = (((uintptr_t)x | (uintptr_t)out) & 15) == 0 ? (count / 8 + 255) / 256 : (count + 255) / 256;
    if (g > 256 * 32) g = 256 * 32;
    f32_to_bf16_kernel<<<dim3((unsigned)(g > 0 ? g : 1)), dim3(256), 0, s>>>(x, out, count);
    return hipGetLastError();
}

// RMS normalisation of one row per workgroup: y = (x * rsqrt(mean(x^2) + eps)) * gamma in fp32, stored in the dtype of x.
// A thread holds every 256th value of the row, HELD of them at a time, all asked for (ONCE, a row no longer than that: gamma's too, and nothing is read twice) before the first is used; a load at a time, each
// pass was a chain of K / 256 latencies.  Few rows are bound by those, many by memory, and by the loads that a compute unit has in flight: buffer loads, whose addresses take one register where a
// pointer for each load took two and left room for one to three wavefronts a SIMD (16 / 32 / 64 values: 136 / 236 / 400 registers, now 40 / 72 / 136 with fp32 rows).  us, normalisation and a product with
// Q4_0 32 x K, a load at a time / pointers / this way: K = 14336 one bf16 row 23.0 / 13.2 / 10.2, 400 rows 56.0 / 41.3 / 34.4, 2000 121.5 / 131.9 / 99.3; 12288 2000 bf16 rows 105 / 119 / 88; 8448 2000 bf16 rows
// 78.8 / 98.6 / 69.9; 4096 400 bf16 rows 23.9 / 18.4 / 17.6; 2048 5000 bf16 rows 56.8 / 56.0 / 47.6; 1024 5000 fp32 rows 36.0 / 38.8 / 31.9.  The sums are the same.
template <typename T, int HELD, bool ONCE>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const T* __restrict__ x, const float* __restrict__ gamma, float eps, uint32_t k, T* __restrict__ y) {
    __shared__ float red[4];
    const T* const xr = x + (int64_t)blockIdx.x * k;
    T* const yr = y + (int64_t)blockIdx.x * k;
    // Values first .. first + 256 HELD - 1 of an array as a buffer: an offset beyond the row reads zero and stores nothing.
    auto part = [&](const auto* row, uint32_t first) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(row + first), 0, (int)(min(k - first, HELD * 256u) * (uint32_t)sizeof(*row)), 0x00020000);
    };
    // (made where it is used: with the offsets of every load in registers from one pass to the next, 16 values and their gammas took 81)
    auto mine = [&](uint32_t size) __attribute__((always_inline)) {
        uint32_t at = threadIdx.x * size;
        asm volatile("" : "+v"(at));
        return at;
    };
    T v[HELD];
    float g[HELD], ss = 0.0f;
    auto load = [&](uint32_t first) __attribute__((always_inline)) {
        const auto from = part(xr, first);
        const uint32_t at = mine(sizeof(T));
#pragma unroll
        for (int j = 0; j < HELD; j++) {
            if constexpr (sizeof(T) == 4) v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at + 1024u * j, 0, 0));
            else v[j] = __builtin_amdgcn_raw_buffer_load_b16(from, at + 512u * j, 0, 0);
        }
    };
    auto load_gamma = [&](uint32_t first) __attribute__((always_inline)) {
        const auto from = part(gamma, first);
        const uint32_t at = mine(4);
#pragma unroll
        for (int j = 0; j < HELD; j++) g[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at + 1024u * j, 0, 0));
    };
    for (uint32_t first = 0; first < (ONCE ? 1 : k); first += HELD * 256) {
        load(first);
        if constexpr (ONCE) load_gamma(first);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < HELD; j++) {
            const float z = load_f32(v, j);
            ss = fmaf(z, z, ss);  // (beyond the row: plus zero)
        }
    }
    ss = wave_sum_dpp(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float rs = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)k + eps);
    for (uint32_t first = 0; first < (ONCE ? 1 : k); first += HELD * 256) {
        if constexpr (!ONCE) {
            load(first);
            load_gamma(first);
            __builtin_amdgcn_sched_barrier(0);
        }
        const auto to = part(yr, first);
        const uint32_t at = mine(sizeof(T));
#pragma unroll
        for (int j = 0; j < HELD; j++) {
            const float z = (load_f32(v, j) * rs) * g[j];
            if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, z), to, at + 1024u * j, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16(f2bf(z), to, at + 512u * j, 0, 0);
        }
    }
}

hipError_t launch_rmsnorm(const void* x, int x_dtype, const float* gamma, float eps, int64_t rows, int64_t k, void* y, hipStream_t s) {
    const dim3 grid((unsigned)rows), block(256);
#define QMM_RMS(HELD, ONCE)                                                                                                                               \
    do {                                                                                                                                                  \
        if (x_dtype == QMM_F32) rmsnorm_kernel<float, HELD, ONCE><<<grid, block, 0, s>>>((const float*)x, gamma, eps, (uint32_t)k, (float*)y);            \
        else rmsnorm_kernel<uint16_t, HELD, ONCE><<<grid, block, 0, s>>>((const uint16_t*)x, gamma, eps, (uint32_t)k, (uint16_t*)y);                      \
    } while (0)
    // (no more loads than the row has values for: K = 512 5000 bf16 rows with 4 / 16 a thread 25.5 / 34.0 us.  Longer rows than 64 hold are read twice, with 32: 20480 one fp32 row 32 / 64 values 10.6 / 11.5,
    // 5000 bf16 rows 456 / 471; 28672 and 32768 within 2 % either way.)
    if (k <= 1024) QMM_RMS(4, true);
    else if (k <= 2048) QMM_RMS(8, true);
    else if (k <= 4096) QMM_RMS(16, true);
    else if (k <= 8192) QMM_RMS(32, true);
    else if (k <= 16384) QMM_RMS(64, true);
    else QMM_RMS(32, false);
#undef QMM_RMS
    return hipGetLastError();
}

hipError_t launch_dequant(int enc, const void* rhs, int64_t n, int64_t k, void* out, int out_dtype,
                          hipStream_t s) {
    const int64_t total = n * k;
    const int64_t per_group = 256 * 4 * (out_dtype == QMM_F32 ? 4 : 8);
    dim3 grid((unsigned)((total + per_group - 1) / per_group)), block(256);
    const uint8_t* w = (const uint8_t*)rhs;
#define QMM_DQ(E)                                                                              \
    if (out_dtype == QMM_F32) dequant_kernel<E, float><<<grid, block, 0, s>>>(w, total, (float*)out); \
    else dequant_kernel<E, uint16_t><<<grid, block, 0, s>>>(w, total, (uint16_t*)out)
    if (enc == QMM_Q4_0) { QMM_DQ(QMM_Q4_0); }
    else if (enc == QMM_Q4_K) { QMM_DQ(QMM_Q4_K); }
    else if (enc == QMM_Q5_K) { QMM_DQ(QMM_Q5_K); }
    else { QMM_DQ(QMM_Q6_K); }
#undef QMM_DQ
    return hipGetLastError();
}

hipError_t launch_dequant_gptq(const void* qweight, const void* scales, const void* qzeros,
                               const void* g_idx, int64_t n, int64_t k, int group, void* out,
                               int out_dtype, hipStream_t s) {
    dim3 grid((unsigned)((n + 63) / 64), (unsigned)((k + 127) / 128)), block(256);
    if (out_dtype == QMM_F32)
        dequant_gptq_kernel<float><<<grid, block, 0, s>>>((const uint32_t*)qweight, (const uint16_t*)scales,
                                                          (const uint32_t*)qzeros, (const int32_t*)g_idx, n, k,
                                                          group, (float*)out);
    else
        dequant_gptq_kernel<uint16_t><<<grid, block, 0, s>>>((const uint32_t*)qweight, (const uint16_t*)scales,
                                                             (const uint32_t*)qzeros, (const int32_t*)g_idx, n, k,
                                                             group, (uint16_t*)out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Q8_0 / Q4_0 quantisers: 32 lanes per block, two blocks per wavefront
// ---------------------------------------------------------------------------

// Writes GGUF Q8_0 blocks (blocks != null) and/or the planar form the Q4_0
// matmul kernels read: codes int8[rows, k], scales fp32[rows, k/32] (the fp16
// block scale widened) and code sums int32[rows, k/32].
template <typename InT>
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const InT* __restrict__ x, int64_t nblocks,
                                                            uint8_t* __restrict__ blocks,
                                                            int8_t* __restrict__ codes,
                                                            float* __restrict__ dscale,
                                                            int32_t* __restrict__ csum) {
    int64_t blk = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 5;
    int l = threadIdx.x & 31;
    if (blk >= nblocks) return;
    float v = load_f32(x, blk * 32 + l);
    float amax = fabsf(v);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 32));
    uint16_t dh;
    const float id = q8_0_block_rule(amax, dh);
    int q = q8_0_code(v, id);
    int sum = q;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 32);
    if (blocks) {
        uint8_t* ob = blocks + blk * Q8_0_BPB;
        if (l == 0) {
            ob[0] = (uint8_t)(dh & 0xff);
            ob[1] = (uint8_t)(dh >> 8);
        }
        ob[2 + l] = (uint8_t)(int8_t)q;
    }
    if (codes) {
        codes[blk * 32 + l] = (int8_t)q;
        if (l == 0) {
            dscale[blk] = h2f(dh);
            csum[blk] = sum;
        }
    }
}

// The weight quantisers are bound by the 4 bytes in per weight.  A wavefront takes 256 consecutive weights at a time, four per lane
// (one 16-byte load per lane, 1 KB per instruction), and finds the extremes of every block across its lanes; a lane rounds its own
// four weights and neighbouring lanes join their codes into the packed bytes.  Four such pieces are loaded ahead.  (One lane per
// 256-weight block, 32 lanes reading 32 cache lines an instruction: 14336 x 4096 to Q4_K took 1.1 ms.)
constexpr int kQuantAhead = 4;

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// the value of the lane OFF apart
template <int OFF>
__device__ __forceinline__ float lane_xor(float v) {
    if constexpr (OFF == 1) return dpp_move<0xB1>(v);
    else if constexpr (OFF == 2) return dpp_move<0x4E>(v);
    else return __shfl_xor(v, OFF, kWave);
}

// The element of largest magnitude over groups of lanes, with its sign; of equal magnitudes the one in the lowest lane (which takes
// the steps in rising order of OFF: what is compared then are neighbouring runs of lanes).
template <int OFF>
__device__ __forceinline__ void first_extreme_step(float& amax, float& mx, int lane) {
    const float oa = lane_xor<OFF>(amax), om = lane_xor<OFF>(mx);
    const bool lower = (lane & OFF) != 0;  // the other lane is the lower one
    if (oa > amax || (oa == amax && lower)) {
        amax = oa;
        mx = om;
    }
}
__device__ __forceinline__ void first_extreme4(const dq_f4& x, float& amax, float& mx) {
    amax = 0.0f;
    mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float v = x[i];
        if (amax < fabsf(v)) {
            amax = fabsf(v);
            mx = v;
        }
    }
}

// pieces of 256 weights: `piece` of this wavefront, then every `step`-th; f(piece, weights) for each of them
template <typename F>
__device__ __forceinline__ void for_pieces(const float* __restrict__ x, int64_t pieces, F f) {
    const int lane = threadIdx.x & 63;
    const int64_t step = (int64_t)gridDim.x * 4;
    int64_t piece = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    for (; piece < pieces; piece += step * kQuantAhead) {
        dq_f4 v[kQuantAhead];
#pragma unroll
        for (int u = 0; u < kQuantAhead; u++) {
            const int64_t q = piece + u * step;
            v[u] = q < pieces ? __builtin_nontemporal_load((const dq_f4*)(x + q * 256) + lane) : dq_f4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < kQuantAhead; u++)
            if (piece + u * step < pieces) f(piece + u * step, v[u]);
    }
}

// rint((v[e] + add) / d) for the four weights of a lane, as integers between low and high (low <= 0 <= high), to take(e, code); 0 where d is 0, infinite or undefined, as the quotient is then.
// d is otherwise the product of an fp16 number and an integer of up to eight bits.  One division instead of four: with y the reciprocal to nearest, q = a y, then q + (a - q d) y with fused
// multiply-adds is the quotient to nearest (Markstein, 1990; no step leaves fp32's normal range where the result is not rounded to zero anyway).  14336 x 4096, us, with the quotients of
// the whole block in one division too: Q4_K 99 -> 81, Q5_K 97 -> 80, Q6_K 75 -> 71 (some 170 vector instructions a block and chains from lane to lane keep it from the 50 that a copy takes;
// a branch to divisions for such a d, or for (hi - lo) / kQmax the same way with one, was slower: it keeps the pieces of a wavefront apart).
template <typename F>
__device__ __forceinline__ void quotient_codes(const dq_f4& v, float add, float d, int low, int high, F take) {
    const bool counts = d != 0.0f && fabsf(d) <= 3.402823466e38f;
    const float y = 1.0f / d;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float a = v[e] + add, q = __builtin_amdgcn_fmed3f(a * y, -1024.0f, 1024.0f), exact = fmaf(fmaf(-q, d, a), y, q);  // (beyond, and infinite, it ends at low or high in any case)
        take(e, counts ? clampi((int)rintf(exact), low, high) : 0);
    }
}

// Q4_0: 8 blocks of 32 per piece, 8 lanes each; a row whose block count is no multiple of 8 is no matter, since the packed blocks of
// a matrix are contiguous, but the last piece may be short.
__global__ __launch_bounds__(256) void quantize_q4_0_kernel(const float* __restrict__ x, int64_t nblocks, uint8_t* __restrict__ out) {
    __shared__ uint16_t packed[4][72];  // the 144 bytes of a piece: stored as whole dwords (blocks are 18 bytes long)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 7;
    auto piece = [&](int64_t p, const dq_f4& v, int blocks) {
        float amax, mx;
        first_extreme4(v, amax, mx);
        first_extreme_step<1>(amax, mx, lane);
        first_extreme_step<2>(amax, mx, lane);
        first_extreme_step<4>(amax, mx, lane);
        const float d = mx / -8.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        uint32_t codes = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float t = v[e] * id;
            t = t + 8.5f;
            int q = (int)t;
            if (q > 15) q = 15;
            codes |= (uint32_t)(uint8_t)q << (8 * e);
        }
        const uint32_t high = (uint32_t)__shfl_xor((int)codes, 4, kWave);  // positions 16 .. 31 of the block
        uint16_t* halves = packed[wave] + 9 * (lane >> 3);
        if (i < 4) {
            const uint32_t w = codes | (high << 4);
            halves[1 + 2 * i] = (uint16_t)w;
            halves[2 + 2 * i] = (uint16_t)(w >> 16);
        }
        if (i == 4) halves[0] = f2h(d);
        // (one wavefront writes and reads its own piece, in program order)
        if (blocks == 8) {
            if (lane < 36) ((uint32_t*)(out + p * 144))[lane] = (uint32_t)packed[wave][2 * lane] | ((uint32_t)packed[wave][2 * lane + 1] << 16);
        } else {
            for (int h = lane; h < blocks * 9; h += 64) ((uint16_t*)(out + p * 144))[h] = packed[wave][h];
        }
    };
    const int64_t whole = nblocks / 8;
    for_pieces(x, whole, [&](int64_t p, const dq_f4& v) { piece(p, v, 8); });
    const int rest = (int)(nblocks - whole * 8);
    if (rest && blockIdx.x == 0 && wave == 0) {
        dq_f4 v = {0, 0, 0, 0};
        if ((lane >> 3) < rest) v = ((const dq_f4*)(x + whole * 256))[lane];
        piece(whole, v, rest);
    }
}

// ---------------------------------------------------------------------------
// K-quant packers: direct min/max fit
// ---------------------------------------------------------------------------

// BITS = 4: Q4_K (codes at byte 16); BITS = 5: Q5_K (fifth bits in qh at byte 16, nibbles at byte 48).  Sub-block j of 32 weights:
// lanes 8 j .. 8 j + 7.
template <int BITS>
__global__ __launch_bounds__(256) void quantize_q4_k_kernel(const float* __restrict__ x, int64_t nblocks, uint8_t* __restrict__ out) {
    constexpr int kQmax = (1 << BITS) - 1;
    const int lane = threadIdx.x & 63, j = lane >> 3, i = lane & 7;
    for_pieces(x, nblocks, [&](int64_t blk, const dq_f4& v) {
        uint8_t* ob = out + blk * (BITS == 4 ? Q4_K_BPB : Q5_K_BPB);
        float lo = fminf(fminf(fminf(fminf(0.0f, v[0]), v[1]), v[2]), v[3]), hi = fmaxf(fmaxf(fmaxf(fmaxf(0.0f, v[0]), v[1]), v[2]), v[3]);
        lo = fminf(lo, dpp_move<0xB1>(lo));
        hi = fmaxf(hi, dpp_move<0xB1>(hi));
        lo = fminf(lo, dpp_move<0x4E>(lo));
        hi = fmaxf(hi, dpp_move<0x4E>(hi));
        lo = fminf(lo, dpp_move<0x141>(lo));
        hi = fmaxf(hi, dpp_move<0x141>(hi));
        const float scale = (hi - lo) / (float)kQmax, minv = 0.0f - lo;
        const float max_scale = __uint_as_float(wave_max_nonneg_bits(fmaxf(0.0f, scale))), max_min = __uint_as_float(wave_max_nonneg_bits(minv));
        // the four quotients of the whole block in one division: lanes of a four take one each
        const int which = lane & 3;
        const float extreme = which & 1 ? max_min : max_scale, quotient = (which < 2 ? 63.0f : extreme) / (which < 2 ? extreme : 63.0f);
        const float inv_scale = max_scale > 0.0f ? dpp_move<0x00>(quotient) : 0.0f;
        const float inv_min = max_min > 0.0f ? dpp_move<0x55>(quotient) : 0.0f;
        const uint32_t sc = (uint32_t)clampi((int)rintf(inv_scale * scale), 0, 63), mn = (uint32_t)clampi((int)rintf(inv_min * minv), 0, 63);
        const uint16_t dh = f2h(dpp_move<0xAA>(quotient)), mh = f2h(dpp_move<0xFF>(quotient));
        // the 6-bit fields of the eight sub-blocks, as bytes of a wave-uniform pair of dwords each
        uint32_t scs[2] = {0, 0}, mns[2] = {0, 0};
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t both = (uint32_t)__builtin_amdgcn_readlane((int)(sc | (mn << 8)), 8 * q);
            scs[q >> 2] |= (both & 63u) << (8 * (q & 3));
            mns[q >> 2] |= (both >> 8) << (8 * (q & 3));
        }
        if (lane == 0) {
            dq_u4 hdr;
            hdr.x = (uint32_t)dh | ((uint32_t)mh << 16);
            hdr.y = scs[0] | ((scs[1] & 0x30303030u) << 2);
            hdr.z = mns[0] | ((mns[1] & 0x30303030u) << 2);
            hdr.w = (scs[1] & 0x0f0f0f0fu) | ((mns[1] & 0x0f0f0f0fu) << 4);
            *(dq_u4*)ob = hdr;
        }
        const float dl = h2f(dh) * (float)sc, ml = h2f(mh) * (float)mn;
        uint32_t codes = 0;
        quotient_codes(v, ml, dl, 0, kQmax, [&](int e, int q) __attribute__((always_inline)) { codes |= (uint32_t)q << (8 * e); });
        const uint32_t nibbles = codes & 0x0f0f0f0fu, odd = (uint32_t)__shfl_xor((int)nibbles, 8, kWave);
        if ((j & 1) == 0) *(uint32_t*)(ob + (BITS == 4 ? 16 : 48) + 32 * (j >> 1) + 4 * i) = nibbles | (odd << 4);
        if constexpr (BITS == 5) {
            uint32_t fifth = ((codes >> 4) & 0x01010101u) << j;  // bit j of the four bytes
            fifth |= (uint32_t)__shfl_xor((int)fifth, 8, kWave);
            fifth |= (uint32_t)__shfl_xor((int)fifth, 16, kWave);
            fifth |= (uint32_t)__shfl_xor((int)fifth, 32, kWave);
            if (lane < 8) *(uint32_t*)(ob + 16 + 4 * i) = fifth;
        }
    });
}

// Sub-block j of 16 weights: lanes 4 j .. 4 j + 3.
__global__ __launch_bounds__(256) void quantize_q6_k_kernel(const float* __restrict__ x, int64_t nblocks, uint8_t* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    for_pieces(x, nblocks, [&](int64_t blk, const dq_f4& v) {
        uint8_t* ob = out + blk * Q6_K_BPB;
        float amax, mx;
        first_extreme4(v, amax, mx);
        first_extreme_step<1>(amax, mx, lane);
        first_extreme_step<2>(amax, mx, lane);
        const float scale = mx / -32.0f;
        float amax_scale = fabsf(scale), max_scale = scale;
        first_extreme_step<4>(amax_scale, max_scale, lane);
        first_extreme_step<8>(amax_scale, max_scale, lane);
        first_extreme_step<16>(amax_scale, max_scale, lane);
        first_extreme_step<32>(amax_scale, max_scale, lane);
        uint32_t codes = 0x20202020u;  // (an all-zero block: every code 32, scales and d zero)
        int s = 0;
        uint16_t dh = 0;
        if (amax_scale != 0.0f) {
            const float iscale = -128.0f / max_scale;
            dh = f2h(1.0f / iscale);
            s = clampi((int)rintf(iscale * scale), -128, 127);
            const float dd = h2f(dh) * (float)s;
            codes = 0;
            quotient_codes(v, 0.0f, dd, -32, 31, [&](int e, int q) __attribute__((always_inline)) { codes |= (uint32_t)(q + 32) << (8 * e); });
        }
        if ((lane & 3) == 0) ob[192 + (lane >> 2)] = (uint8_t)(int8_t)s;
        if (lane == 0) {
            ob[208] = (uint8_t)(dh & 0xff);
            ob[209] = (uint8_t)(dh >> 8);
        }
        // lane = 32 h + 8 quarter + i: ql of quarters 0 | 2 and 1 | 3, qh of all four
        const uint32_t low = codes & 0x0f0f0f0fu, low2 = (uint32_t)__shfl_xor((int)low, 16, kWave);
        const int h = lane >> 5, quarter = (lane >> 3) & 3, i = lane & 7;
        uint32_t high = ((codes >> 4) & 0x03030303u) << (2 * quarter);
        high |= (uint32_t)__shfl_xor((int)high, 8, kWave);
        high |= (uint32_t)__shfl_xor((int)high, 16, kWave);
        const uint32_t ql = low | (low2 << 4);
        uint8_t* at = quarter < 2 ? ob + 64 * h + 32 * quarter + 4 * i : ob + 128 + 32 * h + 4 * i;  // (blocks are 2-byte aligned)
        const uint32_t w = quarter < 2 ? ql : high;
        if (quarter < 3) {
            ((uint16_t*)at)[0] = (uint16_t)w;
            ((uint16_t*)at)[1] = (uint16_t)(w >> 16);
        }
    });
}

// GPTQ symmetric 4-bit: a workgroup takes one group of 64 output columns.  Lanes 4 c .. 4 c + 3 read 128 contiguous bytes of column
// c's row of w at a time; the words go through LDS so that qweight is written in 256-byte rows.  Groups of up to 128 stay in registers
// between the search for the extreme and the rounding.  (One thread per group and column, every lane on a row of its own: 14336 x 4096
// took 1.0 ms.)
__global__ __launch_bounds__(256) void quantize_gptq_kernel(const float* __restrict__ w, int64_t n, int64_t k,
                                                            int group, uint32_t* __restrict__ qweight,
                                                            uint16_t* __restrict__ scales,
                                                            uint32_t* __restrict__ qzeros,
                                                            int32_t* __restrict__ g_idx) {
    constexpr int kHeld = 4;
    __shared__ uint32_t words[4 * kHeld][65];
    const int tid = threadIdx.x, part = tid & 3;
    const unsigned tiles = (unsigned)((n + 63) / 64);
    const int64_t n0 = (int64_t)(blockIdx.x % tiles) * 64, g = blockIdx.x / tiles, col = n0 + (tid >> 2);
    const int steps = group / 32;
    if (n0 == 0)
        for (int i = tid; i < group; i += 256) g_idx[g * group + i] = (int32_t)g;
    if (tid < 8 && n0 + 8 * tid < n) qzeros[g * (n >> 3) + (n0 >> 3) + tid] = 0x77777777u;
    const float* wc = w + (col < n ? col : n - 1) * k + g * group + 8 * part;
    float held[kHeld][8];
    auto load = [&](int i, float (&v)[8]) __attribute__((always_inline)) {
        const dq_f4 a = *(const dq_f4*)(wc + 32 * i), b = *(const dq_f4*)(wc + 32 * i + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    };
    const bool hold = steps <= kHeld;
    float amax = 0.0f;
    if (hold) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i < steps) load(i, held[i]);
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i < steps)
#pragma unroll
                for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(held[i][e]));
    } else {
        for (int i = 0; i < steps; i++) {
            float v[8];
            load(i, v);
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
        }
    }
    amax = fmaxf(amax, dpp_move<0xB1>(amax));
    amax = fmaxf(amax, dpp_move<0x4E>(amax));
    const float scale = 2.0f * amax / 15.0f;
    if (part == 0 && col < n) scales[g * n + col] = f2h(scale);
    auto code = [&](const float (&v)[8]) __attribute__((always_inline)) {
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            int q = 8;
            if (scale != 0.0f) q = clampi((int)rintf(v[e] / scale) + 8, 0, 15);
            word |= (uint32_t)q << (4 * e);
        }
        return word;
    };
    for (int i0 = 0; i0 < steps; i0 += kHeld) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i0 + i < steps) {
                if (!hold) load(i0 + i, held[i]);
                words[4 * i + part][tid >> 2] = code(held[i]);
            }
        __syncthreads();
        const int rows = 4 * (steps - i0 < kHeld ? steps - i0 : kHeld);
        for (int r = tid >> 6; r < rows; r += 4)
            if (n0 + (tid & 63) < n) qweight[(g * (group / 8) + 4 * i0 + r) * n + n0 + (tid & 63)] = words[r][tid & 63];
        __syncthreads();
    }
}

hipError_t launch_quantize_q8_0(const void* x, int x_dtype, int64_t rows, int64_t k, void* blocks, void* codes,
                                void* dscale, void* csum, hipStream_t s) {
    int64_t nblocks = rows * (k / 32);
    dim3 block(256), grid((unsigned)((nblocks * 32 + 255) / 256));
    if (x_dtype == QMM_F32)
        quantize_q8_0_kernel<float><<<grid, block, 0, s>>>((const float*)x, nblocks, (uint8_t*)blocks,
                                                           (int8_t*)codes, (float*)dscale, (int32_t*)csum);
    else
        quantize_q8_0_kernel<uint16_t><<<grid, block, 0, s>>>((const uint16_t*)x, nblocks, (uint8_t*)blocks,
                                                              (int8_t*)codes, (float*)dscale, (int32_t*)csum);
    return hipGetLastError();
}

hipError_t launch_quantize(int enc, const float* x, int64_t rows, int64_t k, void* out, hipStream_t s) {
    if (enc == QMM_Q8_0) return launch_quantize_q8_0(x, QMM_F32, rows, k, out, nullptr, nullptr, nullptr, s);
    // four wavefronts per workgroup, kQuantAhead pieces of 256 weights each; at most eight workgroups per compute unit
    const int64_t pieces = (rows * k + 255) / 256;
    int64_t groups = (pieces + 4 * kQuantAhead - 1) / (4 * kQuantAhead);
    if (groups > 2048) groups = 2048;
    const dim3 grid((unsigned)groups), block(256);
    if (enc == QMM_Q4_0) quantize_q4_0_kernel<<<grid, block, 0, s>>>(x, rows * (k / 32), (uint8_t*)out);
    else if (enc == QMM_Q4_K) quantize_q4_k_kernel<4><<<grid, block, 0, s>>>(x, pieces, (uint8_t*)out);
    else if (enc == QMM_Q5_K) quantize_q4_k_kernel<5><<<grid, block, 0, s>>>(x, pieces, (uint8_t*)out);
    else quantize_q6_k_kernel<<<grid, block, 0, s>>>(x, pieces, (uint8_t*)out);
    return hipGetLastError();
}

hipError_t launch_quantize_gptq(const float* w, int64_t n, int64_t k, int group, void* qweight, void* scales,
                                void* qzeros, void* g_idx, hipStream_t s) {
    quantize_gptq_kernel<<<dim3((unsigned)((n + 63) / 64 * (k / group))), dim3(256), 0, s>>>(
        w, n, k, group, (uint32_t*)qweight, (uint16_t*)scales, (uint32_t*)qzeros, (int32_t*)g_idx);
    return hipGetLastError();
}

}  // namespace qmm
