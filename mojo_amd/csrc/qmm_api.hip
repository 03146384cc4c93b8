// C ABI of libqmm.so: argument validation and dispatch by encoding and shape.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <string>

#include "qmm_internal.h"

namespace qmm {

bool kernel_disabled(const char* family) {
    // (parsed on first use; a C++11 static initialiser runs once, also when two host threads get here together)
    static const std::string list = [] {
        const char* e = getenv("QMM_DISABLE");
        return std::string(",") + (e ? e : "") + ",";
    }();
    return list.size() > 2 && list.find(std::string(",") + family + ",") != std::string::npos;
}

}  // namespace qmm

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_status(hipError_t e, const char* what) {
    if (e == hipSuccess) return QMM_OK;
    return fail(QMM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

bool aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

// environment variables that send every shape that it takes to one kernel (tests), read once
bool is_one(const char* name) {
    const char* e = getenv(name);
    return e && e[0] == '1';
}
bool q4k_lanes_rows_forced() {
    static const bool set = is_one("QMM_Q4K_LANES_ROWS");
    return set;
}
bool q6k_mm_forced() {
    static const bool set = is_one("QMM_Q6K_MM");
    return set;
}
bool q5k_mm_forced() {
    static const bool set = is_one("QMM_Q5K_MM");
    return set;
}

// Q4_K with few lhs rows that no kernel before takes (9 .. 16 fp32 rows on 128 Mi weights and more with a workspace too small for the direct GEMM): the kernel that cuts K across
// workgroups, or the prefill kernel?
bool q4k_kc_wins(int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return m >= (lhs_dtype == QMM_F32 ? 9 : 5) && n <= 4096 && k > 4096;
}

static bool q4k_gemm_from_9_rows(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return encoding == QMM_Q4_K && lhs_dtype == QMM_F32 && m > 8 && m <= 16 && k > 4096 && k % 256 == 0 && n * k >= ((int64_t)128 << 20) &&
           !q4k_kc_wins(lhs_dtype, m, n, k);
}

// Q4_K with 2..4 lhs rows: the decode kernel with one sub-block per lane, or the small-batch matrix-core kernel?
bool q4k_lanes_rows_wins(int64_t n, int64_t k) {
    // The decode kernel pays per weight (its decode runs on the vector units once per row group), the matrix-core kernel
    // per K step and per launch.  Measured, 4 fp32 rows, decode kernel / matrix-core kernel: 512 x 4096 5.1 / 6.7 us,
    // 1024 x 4096 5.2 / 6.7, 2048 x 4096 6.3 / 6.8, 3072 x 4096 7.7 / 6.9, 4096 x 4096 8.9 / 7.0, 14336 x 4096 20.8 / 12.3,
    // 1024 x 8192 9.9 / 10.6, 1024 x 14336 16.2 / 17.5 (bf16 rows: 10.1 / 17.9), 4096 x 14336 42.9 / 18.0.
    return q4k_lanes_rows_forced() || n <= 1024 || n * k <= ((int64_t)8 << 20);
}

// Q6_K (K a multiple of 2048 up to 32768): the small-batch matrix-core kernel, or passes of the decode kernel (one or two
// lhs rows each)?
bool q6k_mm_wanted(int64_t m, int64_t n, int64_t k) {
    // Measured, small-batch kernel / decode-kernel passes, fp32 lhs: 128256 rows: 1 lhs row 87 / 78 us, 2 87 / 113, 4 95 / 225,
    // 8 98 / 449, 16 144 / 895; 14336 rows: 1 17.0 / 14.8, 2 17.5 / 20.6, 4 19.5 / 40.8, 8 21.6 / 81.7, 16 46.7 / 162;
    // 4096 rows: 2 10.3 / 9.6, 4 11.7 / 15.2, 8 13.8 / 32.9, 16 36 / 52; 1024 rows: 2 9.8 / 6.1, 4 11.2 / 7.7, 8 13.2 / 21.9,
    // 16 29 / 38; 4096 x 14336 (four rounds over K, side by side): 1 19.2 / 16.1, 2 20.0 / 22.4, 4 22.1 / 47.  (Its fixed cost is
    // the conversion of the lhs in every workgroup and round.)  QMM_Q6K_MM=1 sends every shape there.
    // (a K beyond 16384, which the decode kernel with the rows global -> LDS does not take: from one bf16 row on)
    return q6k_mm_forced() || m >= 5 || (m >= 3 && n >= 2048) || (m == 2 && (n >= 8192 || (k > 8192 && n >= 2048))) || (k > 16384 && n >= 2048);
}

// Q5_K: the small-batch matrix-core kernel, or passes of the decode kernel (up to four lhs rows each)?
bool q5k_mm_wanted(int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    // Measured, small-batch kernel / decode-kernel passes, fp32 lhs (bf16 lhs: the small-batch kernel is 10-20 % faster, and
    // sixteen bf16 rows cost what eight do): 14336 x 4096: 2 lhs rows 17.5 / 17.5 us, 4 19.2 / 27.2, 8 20.9 / 53.6, 16 41.5 / 106;
    // 4096 x 4096: 4 11.9 / 11.4, 8 14.3 / 22.1; 1024 x 4096: 4 11.6 / 7.8, 8 13.9 / 15.3; 4096 x 14336: 2 34.4 / 33.1, 4 40.4 / 65.4,
    // 8 50.2 / 130; with the rounds of a long K side by side: 2 19.9 / 32.1, 4 21.6 / 65.  QMM_Q5K_MM=1 sends every shape the kernel
    // takes there.
    // Other shapes: 5120 x 5120 with 4 rows 21 / 29.8; 32000 x 4096 with 2 rows 28 / 32.2; 8192 x 28672 with one row 50 / 61.
    // (three and four bf16 rows from 16 Mi weights on: 4096 x 4096 8.8 / 9.1 against 10.6 / 10.8)
    const int64_t min3 = lhs_dtype == QMM_BF16 ? ((int64_t)16 << 20) : ((int64_t)32 << 20);
    return q5k_mm_forced() || m >= 5 || (m >= 3 && (n * k >= min3 || (k > 4096 && n >= 2048))) ||
           (m >= 2 && ((k > 8192 && n >= 2048) || n * k >= ((int64_t)96 << 20))) || (k > 16384 && n >= 2048);
}

// GPTQ with more than 16 lhs rows: do passes of the small-batch kernel (16 rows each, bound by the bytes of the weights)
// beat the GEMM (128 x 256 output tiles, one workgroup each, bound by K per round of 256 tiles)?  Times in
// microseconds as measured on 14336 x 4096, 4096 x 14336 and 4096 x 4096 with 64 to 128 rows: a GEMM round costs
// 64 us per 4096 of K (bf16 lhs; 2.1 x that for an fp32 lhs, which runs two launches) whatever N is, so few column tiles
// (N = 4096: 16 of 256 compute units) and long K favour the passes: 4096 x 14336 with 128 bf16 rows 126 against 209 us.
bool gptq_small_batch_wins(int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    // Passes of the small-batch kernel (16 rows each) against the GEMM (128 x 256 tiles, cut into K shares when they are few, an
    // fp32 lhs of up to 256 rows as twice the rows), in microseconds as measured on this part: 4096 x 4096, bf16 / fp32 lhs: a
    // pass 10.2 / 15.9, the GEMM at 65 .. 256 rows 24 .. 28 / 23 .. 35; 14336 x 4096: a pass 13.0 / 19.6, the GEMM 30 .. 48 / 43 .. 77.
    const bool f32 = lhs_dtype == QMM_F32, twin = qmm::gemm_gptq_twin(lhs_dtype, m);
    const int64_t me = twin ? 2 * m : m;
    const int ks = qmm::gemm_gptq_k_shares(me, n, k);
    const double tiles = (double)((me + 127) / 128) * (double)((n + 255) / 256);
    const double rounds = (double)(int64_t)((tiles * ks + 255.0) / 256.0);
    const double gemm_us = rounds * ((double)k / 4096.0) * 64.0 / ks * (f32 && !twin ? 2.1 : 1.0) + (twin || ks > 1 ? 14.0 : 0.0);
    const double pass_us = (f32 ? 12.0 : 8.0) + (double)n * (double)k * 0.52 / (f32 ? 3.8e6 : 6.0e6) + (k > 4096 ? 2.0 : 0.0);
    return (double)((m + 15) / 16) * pass_us < gemm_us;
}

bool block_params(int enc, int64_t& epb, int64_t& bpb) {
    switch (enc) {
        case QMM_Q4_0: epb = 32; bpb = 18; return true;
        case QMM_Q8_0: epb = 32; bpb = 34; return true;
        case QMM_Q8_K: epb = 256; bpb = 292; return true;
        case QMM_Q4_K: epb = 256; bpb = 144; return true;
        case QMM_Q6_K: epb = 256; bpb = 210; return true;
        case QMM_Q5_K: epb = 256; bpb = 176; return true;
        default: return false;
    }
}

int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// sym = 0 (asymmetric checkpoints: zero points other than 8) is read like sym = 1: every kernel takes the zero
// point from qzeros (stored value + 1, the AutoGPTQ v1 convention); only the quantiser here is symmetric.
int check_gptq(const qmm_gptq_config* cfg, int64_t n, int64_t k, bool quantiser = false) {
    if (!cfg) return fail(QMM_ERR_INVALID, "GPTQ requires a config");
    if (cfg->bits != 4) return fail(QMM_ERR_UNSUPPORTED, "GPTQ bits=%d: only 4-bit is supported", cfg->bits);
    if (cfg->desc_act && quantiser) return fail(QMM_ERR_UNSUPPORTED, "GPTQ desc_act=True: the quantiser here writes plain groups only");
    if (!cfg->sym && quantiser) return fail(QMM_ERR_UNSUPPORTED, "GPTQ sym=False: the quantiser here is symmetric only");
    if (cfg->group_size <= 0 || cfg->group_size % 32 || k % cfg->group_size)
        return fail(QMM_ERR_INVALID, "GPTQ group_size=%d must be a multiple of 32 dividing K=%lld", cfg->group_size,
                    (long long)k);
    if (n % 8) return fail(QMM_ERR_INVALID, "GPTQ needs N %% 8 == 0 (N=%lld)", (long long)n);
    return QMM_OK;
}

// Workspace layout of the Q4_0 path: int8 codes [m,k], fp32 scales [m,k/32], int32 sums [m,k/32].
struct Q8Planes {
    int8_t* codes;
    float* scale;
    int32_t* sum;
    int64_t bytes;
};
Q8Planes q8_planes(void* ws, int64_t m, int64_t k) {
    Q8Planes p;
    int64_t codes = align_up(m * k, 256), sc = align_up(m * (k / 32) * 4, 256);
    p.codes = (int8_t*)ws;
    p.scale = (float*)((char*)ws + codes);
    p.sum = (int32_t*)((char*)ws + codes + sc);
    p.bytes = codes + 2 * sc;
    return p;
}

}  // namespace

// Scratch memory of qmm_matmul_static: device memory that belongs to the loaded library, one copy per GPU, held
// until the process ends.  In host code the array's name is only a handle for the runtime, not a device
// address; the address on each GPU comes from hipGetSymbolAddress with that GPU current, once, and only that
// pointer is ever handed to a kernel.  (No kernel names the array, so it is the host use in static_scratch() that
// makes the compiler emit it, with a symbol the runtime can look up; marking it `used` instead keeps that
// symbol local to the code object and the lookup then fails.)
static __device__ __align__(256) unsigned char scratch[QMM_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

int static_scratch(void** ws) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_status(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul_static: device ordinal %d out of range", dev);
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        // (two threads that get here together read the same address for this device)
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_status(e, "hipGetSymbolAddress(scratch)");
        if (!p || !aligned(p, 256)) return fail(QMM_ERR_HIP, "qmm_matmul_static: the static scratch buffer has no usable device address");
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *ws = p;
    return QMM_OK;
}

}  // namespace

extern "C" {

int qmm_version(void) { return 106; }

const char* qmm_last_error(void) { return g_err; }

int qmm_block_params(int encoding, int64_t* elements_per_block, int64_t* bytes_per_block) {
    int64_t e, b;
    if (!elements_per_block || !bytes_per_block) return fail(QMM_ERR_INVALID, "null output pointer");
    if (!block_params(encoding, e, b)) return fail(QMM_ERR_INVALID, "encoding %d has no block layout", encoding);
    *elements_per_block = e;
    *bytes_per_block = b;
    return QMM_OK;
}

int qmm_device_info(int32_t* compute_units, int32_t* clock_khz) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_status(e, "hipGetDevice");
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) return hip_status(e, "hipGetDeviceProperties");
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (clock_khz) *clock_khz = prop.clockRate;
    return QMM_OK;
}

int qmm_read_probe(const void* buf, int64_t bytes, void* stream) {
    if (!buf || bytes < 16) return fail(QMM_ERR_INVALID, "qmm_read_probe: needs a buffer of at least 16 bytes");
    if (!aligned(buf, 16)) return fail(QMM_ERR_INVALID, "qmm_read_probe: buffer must be 16-byte aligned");
    return hip_status(qmm::launch_read_probe(buf, bytes, (hipStream_t)stream), "qmm_read_probe");
}

int qmm_mfma_probe(void* out, int64_t out_bytes, int kind, int iters, int64_t* flops, void* stream) {
    if (!out || !flops) return fail(QMM_ERR_INVALID, "qmm_mfma_probe: null pointer");
    if (kind < 0 || kind > 6 || iters < 1 || iters > (1 << 24)) return fail(QMM_ERR_INVALID, "qmm_mfma_probe: kind 0..6, iters 1..2^24");
    int32_t cus = 0;
    if (int rc = qmm_device_info(&cus, nullptr)) return rc;
    if (!aligned(out, 4) || out_bytes < (int64_t)cus * 512 * 4)
        return fail(QMM_ERR_INVALID, "qmm_mfma_probe: out must hold 512 floats per compute unit (%lld bytes)", (long long)cus * 512 * 4);
    *flops = (int64_t)cus * 8 * iters * 16 * (kind == 4 || kind == 5 ? 2ll * 16 * 16 * 32 : 2ll * 32 * 32 * 16);
    return hip_status(qmm::launch_mfma_probe((float*)out, cus, kind, iters, (hipStream_t)stream), "qmm_mfma_probe");
}

int qmm_dequantize(int encoding, const void* rhs, int64_t n, int64_t k, void* out, int out_dtype, void* stream) {
    int64_t epb, bpb;
    if (encoding == QMM_Q8_0 || encoding == QMM_Q8_K || !block_params(encoding, epb, bpb))
        return fail(QMM_ERR_INVALID, "qmm_dequantize: encoding %d is not a GGUF weight encoding", encoding);
    if (!rhs || !out) return fail(QMM_ERR_INVALID, "qmm_dequantize: null pointer");
    if (n <= 0 || k <= 0 || k % epb)
        return fail(QMM_ERR_INVALID, "qmm_dequantize: N=%lld, K=%lld; K must be a positive multiple of %lld",
                    (long long)n, (long long)k, (long long)epb);
    if (out_dtype != QMM_F32 && out_dtype != QMM_BF16)
        return fail(QMM_ERR_INVALID, "qmm_dequantize: out_dtype must be f32 or bf16");
    if ((encoding == QMM_Q4_K || encoding == QMM_Q5_K) && !aligned(rhs, 16))
        return fail(QMM_ERR_INVALID, "qmm_dequantize: Q4_K / Q5_K rhs must be 16-byte aligned");
    return hip_status(qmm::launch_dequant(encoding, rhs, n, k, out, out_dtype, (hipStream_t)stream),
                      "qmm_dequantize");
}

int qmm_dequantize_gptq(const qmm_gptq_config* cfg, const void* qweight, const void* scales, const void* qzeros,
                        const void* g_idx, int64_t n, int64_t k, void* out, int out_dtype, void* stream) {
    if (!qweight || !scales || !qzeros || !out) return fail(QMM_ERR_INVALID, "qmm_dequantize_gptq: null pointer");
    if (n <= 0 || k <= 0) return fail(QMM_ERR_INVALID, "qmm_dequantize_gptq: empty shape");
    if (int rc = check_gptq(cfg, n, k)) return rc;
    if (cfg->desc_act && !g_idx) return fail(QMM_ERR_INVALID, "qmm_dequantize_gptq: desc_act=True needs g_idx");
    if (out_dtype != QMM_F32 && out_dtype != QMM_BF16)
        return fail(QMM_ERR_INVALID, "qmm_dequantize_gptq: out_dtype must be f32 or bf16");
    // desc_act = 0: the groups are k / group_size whatever g_idx says (it is not read)
    return hip_status(qmm::launch_dequant_gptq(qweight, scales, qzeros, cfg->desc_act ? g_idx : nullptr, n, k, cfg->group_size, out, out_dtype,
                                               (hipStream_t)stream),
                      "qmm_dequantize_gptq");
}

int qmm_quantize(int encoding, const float* x, int64_t rows, int64_t k, void* out, void* stream) {
    int64_t epb, bpb;
    if (!block_params(encoding, epb, bpb)) return fail(QMM_ERR_INVALID, "qmm_quantize: unknown encoding %d", encoding);
    if (!x || !out) return fail(QMM_ERR_INVALID, "qmm_quantize: null pointer");
    if (rows <= 0 || k <= 0 || k % epb)
        return fail(QMM_ERR_INVALID, "qmm_quantize: rows=%lld, K=%lld; K must be a positive multiple of %lld",
                    (long long)rows, (long long)k, (long long)epb);
    if (encoding == QMM_Q8_K)
        return hip_status(qmm::launch_quantize_q8_k(x, QMM_F32, rows, k, out, (hipStream_t)stream), "qmm_quantize(Q8_K)");
    return hip_status(qmm::launch_quantize(encoding, x, rows, k, out, (hipStream_t)stream), "qmm_quantize");
}

int qmm_quantize_gptq(const qmm_gptq_config* cfg, const float* w, int64_t n, int64_t k, void* qweight, void* scales,
                      void* qzeros, void* g_idx, void* stream) {
    if (!w || !qweight || !scales || !qzeros || !g_idx) return fail(QMM_ERR_INVALID, "qmm_quantize_gptq: null pointer");
    if (n <= 0 || k <= 0) return fail(QMM_ERR_INVALID, "qmm_quantize_gptq: empty shape");
    if (int rc = check_gptq(cfg, n, k, true)) return rc;
    return hip_status(
        qmm::launch_quantize_gptq(w, n, k, cfg->group_size, qweight, scales, qzeros, g_idx, (hipStream_t)stream),
        "qmm_quantize_gptq");
}

// Q4_K and GPTQ have prefill kernels that need no weight planes: the plane GEMM serves them only when the caller's
// workspace holds the planes (what qmm_matmul_workspace_bytes reports); a smaller workspace gets the other kernel.  The
// switch is per call and thread: set at the top of qmm_matmul, read by the dispatch and by the size queries under it.
static thread_local bool g_skip_twin_rows = false;
struct TwinRowsScope {
    bool prev;
    explicit TwinRowsScope(bool skip) : prev(g_skip_twin_rows) { g_skip_twin_rows = skip; }
    ~TwinRowsScope() { g_skip_twin_rows = prev; }
};
extern "C++" {
namespace qmm {
bool twin_rows_allowed() { return !g_skip_twin_rows; }
}  // namespace qmm
}
static thread_local bool g_skip_optional_planes = false;
struct OptionalPlanesScope {
    bool prev;
    explicit OptionalPlanesScope(bool skip) : prev(g_skip_optional_planes) { g_skip_optional_planes = skip; }
    ~OptionalPlanesScope() { g_skip_optional_planes = prev; }
};
static bool kquant_planes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return qmm::gemm_planes_wanted(encoding, lhs_dtype, m, n, k) && !(encoding == QMM_Q4_K && g_skip_optional_planes);
}
static bool gptq_planes(int64_t m, int64_t n, int64_t k, int group) {
    return !g_skip_optional_planes && qmm::gemm_gptq_planes_wanted(m, n, k, group);
}

// what a call cannot do without
static int64_t required_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    if (m <= 0 || k <= 0) return 0;
    if (kquant_planes(encoding, lhs_dtype, m, n, k)) return qmm::gemm_planes_workspace_bytes(encoding, lhs_dtype, m, n, k);
    if (encoding == QMM_Q4_0) {
        const int64_t a = q8_planes(nullptr, m, k).bytes, b = (m >= 5 || k > 4096) && k % 32 == 0 ? qmm::gemm_q4_0_workspace_bytes(m, k) : 0;
        const int64_t c = qmm::gemm_q4_0_planes_wanted(m, n, k) ? qmm::gemm_q4_0_planes_workspace_bytes(m, n, k) : 0;
        return std::max(std::max(a, b), c);
    }
    if (encoding == QMM_Q4_K && m <= 16 && k % 256 == 0) {  // partial sums of K chunks; from 9 rows on the lhs planes of the prefill kernel, whether it serves the call or not
        const int64_t a = m <= 8 ? 0 : qmm::gemm_q4_k_lhs_bytes(lhs_dtype, m, k), b = m >= 2 ? qmm::gemv_q4_k_kc_workspace_bytes(m, n, k) : 0;
        const int64_t c = q4k_gemm_from_9_rows(encoding, lhs_dtype, m, n, k) ? qmm::gemm_q4_k_workspace_bytes(lhs_dtype, m, n, k) : 0;
        return std::max(std::max(a, b), c);
    }
    if (encoding == QMM_Q4_K && m > 16 && k % 256 == 0) return qmm::gemm_q4_k_workspace_bytes(lhs_dtype, m, n, k);
    // (the small-batch kernels with the rounds of a long K side by side; the decode kernels need nothing)
    if (encoding == QMM_Q5_K) return q5k_mm_wanted(lhs_dtype, m, n, k) && k % 512 == 0 ? qmm::gemv_kquant_mm_workspace_bytes(m, n, k) : 0;
    if (encoding == QMM_Q6_K) return q6k_mm_wanted(m, n, k) && k % 2048 == 0 ? qmm::gemv_kquant_mm_workspace_bytes(m, n, k) : 0;
    if (encoding == QMM_GPTQ && k % 256 == 0) {  // small-batch kernel: partial sums of the K chunks; GEMM: lhs planes
        const int64_t a = qmm::gemv_gptq_mm_workspace_bytes(m, n, k), b = m > 16 ? qmm::gemm_gptq_workspace_bytes(lhs_dtype, m, n, k) : 0;
        const int64_t c = gptq_planes(m, n, k, 128) ? qmm::gemm_gptq_planes_workspace_bytes(lhs_dtype, m, n, k) : 0;  // (the group size is not known here)
        return std::max(std::max(a, b), c);
    }
    return 0;
}

static int64_t up256(int64_t v) { return (v + 255) / 256 * 256; }

// Q6_K with five and six fp32 rows on a short K that is no multiple of 2048: the kernel behind sums weight by weight in fp32, the matrix cores, with four
// products a value, a bit less exactly.  Relative error / us against the direct GEMM, 6400 x 1024: 1.0e-7 / 10.9, 12.0 and 1.55e-7 / 9.7 (with four
// rows the decode kernel has 2.5e-7, from seven on the next one 1.9e-7).
static bool decode_sums_more_exactly(int encoding, int lhs_dtype, int64_t m, int64_t k) {
    return encoding == QMM_Q6_K && lhs_dtype == QMM_F32 && (m == 5 || m == 6) && k % 2048 != 0 && k < 4096;
}

// The direct GEMM serves a problem when the caller's workspace holds its operands (qmm_preferred_workspace_bytes); with the smaller one
// the other kernels do.
static int direct_group(const qmm_gptq_config* cfg) { return cfg ? cfg->group_size : 0; }
static bool direct_wanted(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, const void* w = nullptr) {
    return qmm::gemm_direct_wanted(encoding, lhs_dtype, m, n, k, direct_group(cfg), w) && !decode_sums_more_exactly(encoding, lhs_dtype, m, k);
}
static bool direct_serves(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, const void* w, const void* workspace,
                          int64_t workspace_bytes) {
    if (encoding == QMM_GPTQ && (!cfg || cfg->desc_act)) return false;
    return workspace && aligned(workspace, 256) && m > 0 && n > 0 && k > 0 && direct_wanted(encoding, cfg, lhs_dtype, m, n, k, w) &&
           workspace_bytes >= qmm::gemm_direct_workspace_bytes(encoding, lhs_dtype, m, k);
}

// Block encodings with a few lhs rows: the kernel with a super-block per wavefront, unless one of the others is faster.
// us, that other / here (weights from memory), over 42 matrices of 256 .. 128256 rows and K of 512 .. 28672 with 2 .. 16 rows:
// - Q4_K, two to four rows, few long rows (the decode kernel with a sub-block per lane): 1024 x 4096 2 rows 4.0 / 4.7, 4 fp32 rows 5.2 / 5.5 (bf16 4.95 / 4.97), 2048 x 4096 2 rows 4.9 / 5.1,
//   1024 x 8192 2 rows 4.9 / 7.1, 4 bf16 rows 6.5 / 7.4 (fp32 10.1 / 7.9); but 1024 x 2048 4 rows 4.9 / 4.3, 1024 x 11008 4 rows 13.7 / 6.9.
//   Slower here and left so for the relative error: 2 fp32 rows 1024 x 2048 3.44 / 3.75 (2.6e-7 / 1.1e-7), 4 bf16 rows 1024 x 4096 4.8 / 5.2 (2.6e-7 / 0.8e-7), one fp32 row of Q6_K 14336 x 4096 13.5 / 14.1 (3.3e-7 / 1.0e-7).
// - Q5_K, two fp32 rows on few columns (its decode kernel): 512 x 4096 5.0 / 5.2; 2048 x 4096 5.7 / 5.1.
// - 9 .. 16 bf16 rows on large matrices with several groups of K, where few results fit LDS next to the ring: Q6_K 28672 x 8192 51 / 66, 4096 x 14336 9 rows 22.2 / 23.3 (16 rows 25.0 / 22.7), Q5_K 8192 x 28672
//   47 / 51; but Q6_K 8192 x 8192 24 / 21, 5120 x 13824 38 / 24.
// - One row (the decode kernels; 72 matrices of 256 .. 128256 rows and K of 512 .. 28672).  They stream a row per wavefront, and a short one leaves their lanes idle; those of Q5_K and Q6_K hold their loads in registers
//   (Q6_K: unless K is a multiple of 2048).  Q4_K 32000 x 1024 11.9 / 6.4, 14336 x 2048 6.5 / 6.3, but 5632 x 2048 4.4 / 4.9, 14336 x 4096 7.4 / 8.9; Q5_K 4096 x 4096 7.1 / 5.6, 14336 x 4096 12.1 / 10.2, 4096 x 14336 16.7 / 12.4,
//   but 1024 x 4096 4.3 / 5.0, 2048 x 8192 7.0 / 7.9; Q6_K 4096 x 4096 7.2 / 5.7, 4096 x 11008 16.4 / 11.9, 8192 x 28672 53 / 44, but 1024 x 4096 4.6 / 5.0, 128256 x 4096 77 / 86, 4096 x 14336 13.9 / 14.6.
//   Relative error, fp32 row, K = 4096: 2.5e-7 / 1.1e-7, 1.9e-7 / 1.2e-7, 3.3e-7 / 1.0e-7.
// - Q4_0 against its decode kernel (one and two rows; three and four up to K = 4096) and the lhs quantised by a launch of its own (21 matrices): 1 row 8192 x 28672 42 / 31, 32000 x 512 11.6 / 4.6, but 4096 x 4096 4.4 / 4.7; 2 rows
//   4096 x 4096 5.5 / 4.9, 4096 x 14336 16.7 / 10.9, but 2048 x 5632 6.0 / 7.2, 28672 x 8192 25 / 27; 4 rows 4096 x 4096 7.4 / 5.4, 14336 x 4096 12.7 / 9.5; 8 rows 8.7 / 6.7, 13.4 / 10.4, 4096 x 14336 16.7 / 12.6;
//   16 bf16 rows 32000 x 512 13.0 / 10.5, 1024 x 14336 14.7 / 12.4, but 4096 x 4096 8.7 / 10.2.
// - Q6_K, five and six fp32 rows, K = 256 or 512: more exact weight by weight (decode_sums_more_exactly), 0.85e-7 against 0.88e-7.
// More rows than one workgroup takes (fp32: 8, bf16: 16), GPTQ too: two to four workgroups side by side, each of which streams the weights itself, against the lhs prepared by a launch of its own and the direct, shared or older
// small-batch GEMM.  us, those / here (45 matrices of 128 .. 38000 rows and K of 512 .. 28672, and groups of two to sixteen; weights from memory):
// - 9 .. 16 fp32 rows: Q4_K 4096 x 4096 11.7 / 9.2, 14336 x 4096 21.7 / 15.5, 4096 x 14336 25.5 / 19.1, 1024 x 14336 23.9 / 11.4, 65536 x 4096 68 / 60, 262144 x 1024 75 / 63, but 8192 x 28672 61 / 100; GPTQ 4096 x 4096 12.0 / 8.9, but 8192 x 8192 21.7 / 28.8;
//   Q4_0 5856 x 4096 10.0 / 8.6, 39368 x 512 16.2 / 9.2, but 14336 x 4096 13.5 / 13.7, 3144 x 8192 11.1 / 12.3.
// - 17 .. 32 fp32 rows: Q4_K 912 x 1024 7.9 / 4.3, 1024 x 14336 24.6 / 13.5; 4096 x 4096 11.9 / 11.4, but 4096, 1024 and 1024 x 4096 in one call 12.9 / 15; GPTQ (never in groups) 4096 x 4096 12.3 / 11.5;
//   Q4_0 4096, 1024 and 1024 x 4096 15.2 / 11.0.
// - 17 .. 32 bf16 rows: Q4_K 4096 x 4096 10.5 / 9.8, 14336 x 4096 19.6 / 17.4, 1024 x 14336 19.9 / 11.8, but 32000 x 4096 31 / 34, 8192 x 8192 20.6 / 22, Q5_K 5120 x 5120 17.8 / 15.3, but with two of 1024 x 5120
//   15.9 / 19.9; Q4_0 600 x 2048 7.9 / 6.9, 21848 x 2560 27 / 20, but 2520 x 2048 20 % longer.
// - 33 .. 64 bf16 rows: Q4_K 912 x 1024 7.9 / 4.8, 512 x 28672 31 / 15, but two of 1024 x 14336 18.8 / 26; 1520 x 3072 5 % less, 2048 x 5632 12.2 / 13.0; GPTQ 4096 x 4096 12.7 / 11.6.
// - Q4_0, 9 .. 16 fp32 rows: the other kernel has a tile of 16 weight rows a compute unit at a time, and is ahead where they fill its rounds: 11008 x 4096 11.9 / 12.8, 4096 x 14336 17.3 / 18.4, but 4560 x 14336 21.1 / 18.0.
// - Short K: a workgroup has few wavefronts, and what counts is how many the fullest compute unit gets.  Q4_0 33 .. 64 bf16 rows 3072 x 768 with 9 of them 7.4 / 8.4, 2048 x 1536 with 12 8.7 / 9.6, 1280 x 2048 with 16 8.2 / 9.7,
//   but 1024 x 1536 with 6 8.0 / 6.8; 9 .. 16 bf16 rows 14336 x 1024 with 16 9.2 / 9.8, but 11976 x 1024 with 12 9.7 / 8.6.  Five wavefronts (K = 1280) do not divide among four SIMDs either: 17 .. 32 bf16 rows with three
//   workgroups of them Q4_K 5688 x 1280 10.1 / 10.5, Q6_K 5096 x 1280 9.9 / 10.7, 12648 x 1280 14.1 / 18.0, but with two Q4_K 7168 x 1280 10.4 / 9.3.
// - 17 .. 32 bf16 rows Q6_K 14336 x 4096 24.2 / 24.5, 14528 x 4096 26.3 / 28.7, but 11008 x 4096 23.7 / 22.
// Over 3000 random calls (128 .. 48000 rows, K of 256 .. 28672, 9 .. 64 rows; the other side forced each time): 0.2 % take more than 4 % longer here than there.  Weights in the last-level cache, which a program's layers do not
// stay in: the others read them again at little cost, and 4 % take more than 4 % longer here, 17 bf16 rows Q4_K 4096 x 4096 8.9 / 9.5, 14336 x 4096 15.3 / 17.2, Q5_K 4096 x 4096 9.3 / 10.4, Q6_K 11008 x 4096 20.6 / 21.5,
// Q4_0 14336 x 4096 16.9 / 19.2 (from memory 10.3 / 9.9, 19.4 / 17.5, 11.1 / 10.4, 25.2 / 22.1, 21.1 / 19.4).
// The lines follow K more than the number of weight rows: a call with several matrices sends each where a call of its own would, and two ways for one call cost more than either.
// (Asked once the kernel is known to take the call.)
static bool small_tiles_wanted(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const int64_t million = (int64_t)1 << 20, weights = n * k;
    const bool f32 = lhs_dtype == QMM_F32, q6 = encoding == QMM_Q6_K;
    const qmm::SmallLoad load = qmm::small_load(lhs_dtype, m, n, k);
    const bool five = k > 1024 && k <= 1280 && load.wavefronts > 12;
    if (encoding == QMM_GPTQ) {
        if (f32 && m <= 16) return k <= 4096 || weights < (k <= 8192 ? 60 : 80) * million;
        if (f32) return m <= 32 && weights < (k <= 4096 ? 17 : k <= 8192 ? 24 : 40) * million;
        if (m <= 32) return weights < (k <= 2048 ? 16 : k <= 4096 ? 80 : k <= 8192 ? 40 : 45) * million;
        return m <= 64 && weights < (k <= 2048 ? 5 : k <= 4096 ? 20 : k <= 8192 ? 4 : 16) * million;
    }
    if (encoding == QMM_Q4_0) {
        if (f32 && m <= 16) return weights < (k <= 3072 ? 128 : k <= 4096 ? 40 : k <= 8192 ? 24 : n > 3584 && n <= 4096 ? 30 : 70) * million;
        if (f32) return m <= 32 && weights < (k <= 4096 ? 45 : k <= 8192 ? 28 : 40) * million;
        if (k > 8192) return n <= (m <= 32 ? 2048 : m <= 64 ? 512 : 0);
        if (k <= 2048 && weights < 3 * million) return m <= 32 || (m <= 64 && load.wavefronts <= 8 && load.workgroups <= (k <= 256 ? 4 : 3));
        return m <= 32 && k <= 4096 && !five && weights >= 18 * million && weights < 110 * million;
    }
    if (f32 && m <= 16) return (encoding == QMM_Q4_K && k <= 4096) || weights < (k <= 8192 ? 256 : 128) * million;
    if (k > 8192) return n <= (f32 ? (m > 32 ? 0 : q6 ? 768 : 1024) : m <= 32 ? (q6 ? 768 : 2048) : m <= 64 ? 512 : 0);
    if (!f32 && m <= 32) return k <= 4096 && !five && weights < (k <= 2048 ? 16 : q6 && k > 3072 ? 50 : 64) * million;
    return m <= (f32 ? 32 : 64) && k <= 1024 && weights < 5 * million;
}

static bool small_wanted(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, const void* w) {
    if (m < 1 || (m == 1 && (encoding == QMM_Q4_K || encoding == QMM_Q4_0) && k <= 14528 && (k > 2048 || n < 8192)) || (m == 1 && encoding == QMM_Q4_K && k > 2048) || !qmm::gemv_kquant_small_supported(encoding, lhs_dtype, m, n, k, w)) return false;
    const bool f32 = lhs_dtype == QMM_F32;
    if (m > qmm::small_most_rows(lhs_dtype)) return !(encoding == QMM_Q5_K && q5k_mm_forced()) && !(encoding == QMM_Q6_K && q6k_mm_forced()) && small_tiles_wanted(encoding, lhs_dtype, m, n, k);
    if (m == 1) {
        if (encoding == QMM_Q4_K) return true;
        if (encoding == QMM_Q5_K) return !q5k_mm_forced() && (k <= 2048 || k > 8192 || n > 2048);
        if (encoding == QMM_Q4_0) return k > 14528 || (k <= 1536 && n >= 8192);
        if (q6k_mm_forced()) return false;
        return n <= 1024 ? k > 8192 : k <= 2048 || k % 2048 != 0 || k > 16384 || (k == 4096 && n > 2048 && n <= 14336);
    }
    if (encoding == QMM_Q4_K) {
        if (m <= 4 && q4k_lanes_rows_forced()) return false;
        return qmm::kernel_disabled("q4k_lanes_rows") || k <= 2304 || k > 8192 ||
               !((m == 2 && (n <= 1024 || (k <= 4096 && n * k <= ((int64_t)8 << 20)))) || (m <= 4 && n <= 1024 && f32 == (k <= 4096)));
    }
    if (encoding == QMM_Q4_0)
        return m == 2 ? k > 8192 || ((n > 2048 || k <= 2048) && n * k <= (int64_t)64 << 20) : m <= 8 || (k <= 1024 && !(k > 512 && n > 12288 && n <= 16384)) || (n <= 2048 && k <= 2048) || (n <= 1024 && k > 8192);
    const bool large = m > 8 && k > 4096;
    if (encoding == QMM_Q5_K) return !q5k_mm_forced() && !(f32 && m == 2 && n <= 1024 && k > 2304 && k <= 4096) && !(large && n * k >= ((int64_t)190 << 20));
    if (f32 && (m == 5 || m == 6) && k <= 512) return false;
    return !q6k_mm_forced() && !(large && (n * k >= ((int64_t)96 << 20) || (m < 12 && k > 8192 && k % 2048 == 0 && n * k >= ((int64_t)54 << 20))));
}

// GPTQ with groups in their order, up to 16 lhs rows (fp32: 8).  us, the kernels before (decode, small batch, direct GEMM) / here, weights from memory: one bf16 row 4096 x 4096 6.5 / 4.9, 14336 x 4096 10.2 / 8.9,
// 4096 x 14336 15.6 / 11.6, one fp32 row 6.6 / 5.1, 10.4 / 9.4, 15.7 / 11.4 (weights in the last-level cache 4.5 / 4.8, 7.5 / 8.4, 10.3 / 10.8: the decode kernel has less to do before its first product); four bf16 rows 9.4 / 5.5, 12.4 / 9.0, 15.2 / 11.3; eight fp32 rows 13.6 / 7.7, 18.3 / 12.6, 20.9 / 12.9; 16 bf16 rows 11.1 / 8.9, 14.3 / 13.5, 16.8 / 14.6.  Relative error, K = 4096: 4.2e-7 /
// 0.8e-7 (fp32 rows), 2.2e-7 and 1.2e-7 / 0.65e-7 (one and four bf16 rows).
static bool gptq_small_wanted(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return encoding == QMM_GPTQ && cfg && !cfg->desc_act && qmm::gemv_gptq_small_supported(lhs_dtype, m, n, k, cfg->group_size) &&
           (m <= qmm::small_most_rows(lhs_dtype) || small_tiles_wanted(encoding, lhs_dtype, m, n, k));
}

// Does the kernel that serves this problem store bf16 itself?  (The Q4_K decode kernel does; everything else goes
// through an fp32 result in the workspace and a narrowing pass.)
static bool stores_bf16_itself(int encoding, int64_t m, int64_t k, int flags) {
    return encoding == QMM_Q4_K && m == 1 && k % 256 == 0 && k <= 16384 && !(flags & QMM_FLAG_ACT_Q8K) && !qmm::kernel_disabled("q4k_lanes");
}

// Q8_K activations: up to 16 lhs rows go through kernels that take the integer sub-block dots themselves, in passes of four
// rows (Q4_K: the lhs quantised inside the kernel, K <= 16384; Q5_K and Q6_K: quantised once per call into planes in the
// workspace).  More rows: the lhs is quantised, d8 * code written as fp32 rows into the workspace, and the floating-point
// path runs on those (the products of the integer treatment, summed in fp32).
constexpr int64_t kQ8kIntegerMaxRows = 16;
static bool q8k_integer_kernel(int encoding, int64_t m, int64_t k) {
    if (m > kQ8kIntegerMaxRows || k % 256) return false;
    return encoding == QMM_Q4_K ? k <= 16384 : (encoding == QMM_Q5_K || encoding == QMM_Q6_K);
}
static int64_t q8k_integer_workspace(int encoding, int64_t m, int64_t k) { return encoding == QMM_Q4_K ? 0 : qmm::q8k_planes_bytes(m, k); }

static int64_t required_bytes_flags(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    int64_t base = required_bytes(encoding, lhs_dtype, m, n, k);
    if ((flags & QMM_FLAG_ACT_Q8K) && m > 0 && k > 0)
        base = q8k_integer_kernel(encoding, m, k) ? q8k_integer_workspace(encoding, m, k)
                                                  : up256(m * k * 4) + required_bytes(encoding, QMM_F32, m, n, k);
    if (!(flags & QMM_FLAG_OUT_BF16) || m <= 0 || n <= 0 || stores_bf16_itself(encoding, m, k, flags)) return base;
    return up256(base) + up256(m * n * 4);
}

static int64_t preferred_matmul(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags);

// Act-order GPTQ by sorted columns: the sorted tensors, then what the plain product on them needs.  0: not this way.
// The sorted columns go to the direct GEMM whatever the number of rows: the small-batch kernel and the GEMM that unpacks tiles drop low bits of their
// products.  Relative errors, look-up / small batch / tile GEMM / direct: 6400 x 1024 with 5 fp32 rows 1.6e-7 / 4.0e-7 / - / 1.1e-7, 14336 x 4096 with
// 400 bf16 rows 2e-7 / - / 3e-6 / 7e-8 (the call takes 10 us less with the tile GEMM).  Matrices beyond what that
// takes (2^32 weights) stay with the look-up kernel.
static int64_t order_bytes(const qmm_gptq_config& cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    if (!cfg.desc_act || cfg.group_size <= 0 || k % cfg.group_size || (flags & ~QMM_FLAG_OUT_BF16) || qmm::kernel_disabled("direct") ||
        !qmm::gptq_order_wanted(lhs_dtype, m, n, k, cfg.group_size) || n * k >= ((int64_t)1 << 32))
        return 0;
    return qmm::gptq_order_space(nullptr, n, k).bytes + up256(qmm::gemm_direct_workspace_bytes(QMM_GPTQ, lhs_dtype, m, k));
}
static bool order_serves(const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags, const void* workspace, int64_t workspace_bytes) {
    const int64_t need = order_bytes(*cfg, lhs_dtype, m, n, k, flags);
    return need > 0 && workspace && aligned(workspace, 256) && workspace_bytes >= need;
}

static int64_t preferred_matmul(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    const int64_t need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    if (m <= 0 || n <= 0 || k <= 0 || (encoding == QMM_GPTQ && (!cfg || cfg->group_size <= 0))) return need;
    if (encoding == QMM_GPTQ && cfg->desc_act) {
        const int64_t order = order_bytes(*cfg, lhs_dtype, m, n, k, flags);
        return order ? std::max(need, order + ((flags & QMM_FLAG_OUT_BF16) ? up256(m * n * 4) : 0)) : need;
    }
    int64_t ahead = 0;
    // the kernels for a few rows; from where others served the call, also what those need (the weights' alignment is not known here)
    int64_t few = -1;
    if (!(flags & QMM_FLAG_ACT_Q8K) && gptq_small_wanted(encoding, cfg, lhs_dtype, m, n, k)) few = qmm::gemv_gptq_small_workspace_bytes(lhs_dtype, m, n, k, cfg->group_size);
    else if (!(flags & QMM_FLAG_ACT_Q8K) && small_wanted(encoding, lhs_dtype, m, n, k, nullptr)) few = qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, n, k);
    if (few >= 0) {
        const int64_t direct = m > qmm::small_most_rows(lhs_dtype) && direct_wanted(encoding, cfg, lhs_dtype, m, n, k) ? qmm::gemm_direct_workspace_bytes(encoding, lhs_dtype, m, k) : 0;
        return std::max(std::max(need, direct), up256(few) + (flags & QMM_FLAG_OUT_BF16 ? up256(m * n * 4) : 0));
    }
    if (flags & QMM_FLAG_ACT_Q8K) {  // (the lhs as fp32 rows in front, where the integer kernels do not serve the call)
        if (q8k_integer_kernel(encoding, m, k) || (flags & QMM_FLAG_OUT_BF16)) return need;
        ahead = up256(m * k * 4);
        lhs_dtype = QMM_F32;
        if (small_wanted(encoding, lhs_dtype, m, n, k, nullptr)) few = qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, n, k);
    }
    if (!direct_wanted(encoding, cfg, lhs_dtype, m, n, k)) return few > 0 ? std::max(need, ahead + up256(few)) : need;
    return std::max(need, ahead + std::max(few > 0 ? up256(few) : 0, qmm::gemm_direct_workspace_bytes(encoding, lhs_dtype, m, k)));
}

// Where a call takes a workspace at all, the figure holds what the direct GEMM needs too (up to a size that the static buffer also has).
int64_t qmm_matmul_workspace_bytes_flags(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    const int64_t need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    if (need <= 0) return need;
    qmm_gptq_config cfg{4, 128, 0, 1};
    int64_t more = preferred_matmul(encoding, &cfg, lhs_dtype, m, n, k, flags);
    if (encoding == QMM_GPTQ) {  // (the group size is not known here)
        cfg.group_size = 32;
        more = std::max(more, preferred_matmul(encoding, &cfg, lhs_dtype, m, n, k, flags));
    }
    return more <= (int64_t)QMM_STATIC_SCRATCH_BYTES ? more : need;
}
int64_t qmm_matmul_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return qmm_matmul_workspace_bytes_flags(encoding, lhs_dtype, m, n, k, 0);
}

static int matmul_f32(int encoding, const qmm_gptq_config* cfg, const void* lhs, int lhs_dtype, int64_t m, int64_t k,
                      const void* const* rhs, int n_rhs, int64_t n, float* out, void* workspace, int64_t workspace_bytes,
                      int flags, void* stream, uint16_t* out16 = nullptr);

int qmm_matmul(int encoding, const qmm_gptq_config* cfg, const void* lhs, int lhs_dtype, int64_t m, int64_t k,
               const void* const* rhs, int n_rhs, int64_t n, float* out, void* workspace, int64_t workspace_bytes,
               int flags, void* stream) {
    // the plane GEMM for Q4_K / GPTQ only with a workspace that holds the planes
    const bool optional = (encoding == QMM_Q4_K || encoding == QMM_GPTQ) && m > 0 && n > 0 && k > 0 && !g_skip_optional_planes;
    const OptionalPlanesScope scope(g_skip_optional_planes ||
                                    (optional && (!workspace || workspace_bytes < required_bytes_flags(encoding, lhs_dtype, m, n, k, flags))));
    if (!(flags & QMM_FLAG_OUT_BF16) || (flags & ~(QMM_FLAG_W_BF16 | QMM_FLAG_ACT_Q8K | QMM_FLAG_OUT_BF16)))
        return matmul_f32(encoding, cfg, lhs, lhs_dtype, m, k, rhs, n_rhs, n, out, workspace, workspace_bytes, flags, stream);
    // bf16 output
    const int inner = flags & ~QMM_FLAG_OUT_BF16;
    if (!lhs || !rhs || !out) return fail(QMM_ERR_INVALID, "qmm_matmul: null pointer");
    if (!aligned(out, 2)) return fail(QMM_ERR_INVALID, "qmm_matmul: bf16 out must be 2-byte aligned");
    if (m > 0 && n > 0 && k > 0 && m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX && n_rhs == 1 && rhs[0] &&
        (lhs_dtype == QMM_F32 || lhs_dtype == QMM_BF16) && aligned(lhs, 16) && aligned(rhs[0], 16) && !(inner & QMM_FLAG_W_BF16) &&
        stores_bf16_itself(encoding, m, k, inner)) {
        if (small_wanted(encoding, lhs_dtype, m, n, k, rhs[0])) {  // (one group of K: no workspace)
            const hipError_t e = qmm::launch_gemv_kquant_small(encoding, lhs, lhs_dtype, 1, rhs, &n, &out, m, k, false, true, nullptr, (hipStream_t)stream);
            return hip_status(e, "qmm_matmul(Q4_K, few columns, bf16 out)");
        }
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_k_lanes(lhs, lhs_dtype, (const uint8_t*)rhs[0], (int)m, n, k, out, n, (hipStream_t)stream, &handled, true);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_K decode, bf16 out)");
        if (handled) return QMM_OK;
    }
    if (m <= 0 || n <= 0) return fail(QMM_ERR_INVALID, "qmm_matmul: M=%lld N=%lld must be positive", (long long)m, (long long)n);
    const void* const w = n_rhs > 0 ? rhs[0] : nullptr;
    const bool few = encoding == QMM_GPTQ ? (n_rhs == 3 || n_rhs == 4) && cfg && cfg->group_size > 0 && gptq_small_wanted(encoding, cfg, lhs_dtype, m, n, k)
                                          : n_rhs == 1 && w && small_wanted(encoding, lhs_dtype, m, n, k, w);
    const bool small = few && k > 0 && (lhs_dtype == QMM_F32 || lhs_dtype == QMM_BF16) &&
                       workspace && aligned(workspace, 256) && workspace_bytes >= required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    if (!(inner & QMM_FLAG_ACT_Q8K) && (small || direct_serves(encoding, cfg, lhs_dtype, m, n, k, w, workspace, workspace_bytes)))
        return matmul_f32(encoding, cfg, lhs, lhs_dtype, m, k, rhs, n_rhs, n, out, workspace, workspace_bytes, inner, stream, (uint16_t*)out);
    // (the fp32 result sits behind everything the inner call needs, the Q8_K round trip of the lhs included)
    int64_t base = up256(required_bytes_flags(encoding, lhs_dtype, m, n, k, inner));
    if (encoding == QMM_GPTQ && cfg) {
        const int64_t order = std::max(base, order_bytes(*cfg, lhs_dtype, m, n, k, inner));
        if (workspace_bytes >= order + up256(m * n * 4)) base = order;
    }
    const int64_t need = base + up256(m * n * 4);
    if (!workspace || workspace_bytes < need)
        return fail(QMM_ERR_WORKSPACE, "qmm_matmul: bf16 output of this problem goes through an fp32 result in the workspace: %lld bytes required "
                                       "(qmm_matmul_workspace_bytes_flags), %lld given", (long long)need, (long long)workspace_bytes);
    if (!aligned(workspace, 256)) return fail(QMM_ERR_INVALID, "qmm_matmul: workspace must be 256-byte aligned");
    float* tmp = (float*)((char*)workspace + base);
    if (int rc = matmul_f32(encoding, cfg, lhs, lhs_dtype, m, k, rhs, n_rhs, n, tmp, workspace, base, inner, stream)) return rc;
    return hip_status(qmm::launch_f32_to_bf16(tmp, (uint16_t*)out, m * n, (hipStream_t)stream), "qmm_matmul(narrow to bf16)");
}

static int matmul_f32(int encoding, const qmm_gptq_config* cfg, const void* lhs, int lhs_dtype, int64_t m, int64_t k,
                      const void* const* rhs, int n_rhs, int64_t n, float* out, void* workspace, int64_t workspace_bytes,
                      int flags, void* stream, uint16_t* out16) {
    // (out16 != null: a call that the direct GEMM serves, with the bf16 form of the result stored there instead of `out`)
    hipStream_t s = (hipStream_t)stream;
    if (!lhs || !rhs || !out) return fail(QMM_ERR_INVALID, "qmm_matmul: null pointer");
    if (flags & ~(QMM_FLAG_W_BF16 | QMM_FLAG_ACT_Q8K)) return fail(QMM_ERR_INVALID, "qmm_matmul: unknown flag bits 0x%x", flags);
    if (flags & QMM_FLAG_W_BF16)
        return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul: QMM_FLAG_W_BF16 (weights rounded to bf16 before the product) has no kernel in this build");
    if (m <= 0 || n <= 0 || k <= 0)
        return fail(QMM_ERR_INVALID, "qmm_matmul: M=%lld N=%lld K=%lld must all be positive", (long long)m,
                    (long long)n, (long long)k);
    if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return fail(QMM_ERR_INVALID, "qmm_matmul: dimension too large");
    if (lhs_dtype != QMM_F32 && lhs_dtype != QMM_BF16)
        return fail(QMM_ERR_INVALID, "qmm_matmul: lhs dtype must be f32 or bf16");
    if (!aligned(lhs, 16) || !aligned(out, (void*)out == (void*)out16 ? 2 : 4)) return fail(QMM_ERR_INVALID, "qmm_matmul: lhs must be 16-byte aligned");
    int64_t esz = lhs_dtype == QMM_F32 ? 4 : 2;
    int64_t need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags & QMM_FLAG_ACT_Q8K);
    if (need > 0 && (!workspace || workspace_bytes < need))
        return fail(QMM_ERR_WORKSPACE, "qmm_matmul: workspace of %lld bytes required, %lld given", (long long)need,
                    (long long)workspace_bytes);
    if (need > 0 && !aligned(workspace, 256)) return fail(QMM_ERR_INVALID, "qmm_matmul: workspace must be 256-byte aligned");

    if (encoding == QMM_GPTQ) {
        if (n_rhs != 3 && n_rhs != 4)
            return fail(QMM_ERR_INVALID, "qmm_matmul: GPTQ takes rhs = (qweight, scales, qzeros[, g_idx]), got %d", n_rhs);
        if (int rc = check_gptq(cfg, n, k)) return rc;
        for (int i = 0; i < 3; i++)
            if (!rhs[i] || !aligned(rhs[i], 4)) return fail(QMM_ERR_INVALID, "qmm_matmul: GPTQ rhs[%d] null or misaligned", i);
        if (cfg->desc_act) {
            // act-order checkpoints: the columns sorted by group, then the kernels for plain groups; the decode kernel that looks the group of
            // every k up, four lhs rows per pass, for few rows and with a workspace too small for the sorted matrix
            if (n_rhs != 4 || !rhs[3] || !aligned(rhs[3], 4))
                return fail(QMM_ERR_INVALID, "qmm_matmul: GPTQ desc_act=True needs rhs[3] = g_idx int32[K]");
            const int32_t* only_if = nullptr;
            if (order_serves(cfg, lhs_dtype, m, n, k, flags, workspace, workspace_bytes)) {
                const qmm::GptqOrder order{(const uint32_t*)rhs[0], (const int32_t*)rhs[3], qmm::gptq_order_space(workspace, n, k)};
                const void* sorted[1] = {order.space.qweight};
                const hipError_t e = qmm::launch_gemm_direct(encoding, lhs, lhs_dtype, 1, sorted, &n, &out, (const uint16_t*)rhs[1], (const uint32_t*)rhs[2], cfg->group_size, m, k,
                                                             nullptr, (char*)workspace + order.space.bytes, s, true, &order);
                if (e != hipSuccess) return hip_status(e, "qmm_matmul(GPTQ act-order, direct GEMM)");
                only_if = order.space.uneven;
            }
            hipError_t e = qmm::launch_gemv_gptq_act_order(lhs, lhs_dtype, (const uint32_t*)rhs[0], (const uint16_t*)rhs[1], (const uint32_t*)rhs[2],
                                                           (const int32_t*)rhs[3], (int)m, n, k, cfg->group_size, out, n, s, only_if);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul(GPTQ act-order)");
            return QMM_OK;
        }
        if (gptq_small_wanted(encoding, cfg, lhs_dtype, m, n, k)) {
            const bool parts = workspace && aligned(workspace, 256) && workspace_bytes >= qmm::gemv_gptq_small_workspace_bytes(lhs_dtype, m, n, k, cfg->group_size);
            return hip_status(qmm::launch_gemv_gptq_small(lhs, lhs_dtype, (const uint32_t*)rhs[0], (const uint16_t*)rhs[1], (const uint32_t*)rhs[2], m, n, k, cfg->group_size, out,
                                                          out16 != nullptr, parts ? workspace : nullptr, s), "qmm_matmul(GPTQ, few rows)");
        }
        if (direct_serves(encoding, cfg, lhs_dtype, m, n, k, rhs[0], workspace, workspace_bytes))
            return hip_status(qmm::launch_gemm_direct(encoding, lhs, lhs_dtype, 1, rhs, &n, &out, (const uint16_t*)rhs[1], (const uint32_t*)rhs[2],
                                                      cfg->group_size, m, k, out16, workspace, s),
                              "qmm_matmul(direct GEMM)");
        // GEMM (128 x 256 tiles) or passes of the small-batch kernel (16 rows each)?
        if (gptq_planes(m, n, k, cfg->group_size))
            return hip_status(qmm::launch_gemm_gptq_planes(lhs, lhs_dtype, (const uint32_t*)rhs[0], (const uint16_t*)rhs[1], (const uint32_t*)rhs[2],
                                                           m, n, k, cfg->group_size, out, workspace, s),
                              "qmm_matmul(GPTQ planes GEMM)");
        const bool gemm_wins = !gptq_small_batch_wins(lhs_dtype, m, n, k);
        if (m > 16 && qmm::gemm_gptq_supported(k, cfg->group_size) &&
            (gemm_wins || !qmm::gemv_gptq_mm_supported(rhs[0], n, k, cfg->group_size)))
            return hip_status(qmm::launch_gemm_gptq(lhs, lhs_dtype, (const uint32_t*)rhs[0], (const uint16_t*)rhs[1],
                                                    (const uint32_t*)rhs[2], m, n, k, cfg->group_size, out, workspace, s),
                              "qmm_matmul(GPTQ GEMM)");
        // One pass of the matrix-core small-batch kernel per 16 lhs rows; the fewest rows go to the column kernels (weights from the
        // last-level cache, us).  More than 4096 columns, 64 per workgroup: one row, and two fp32 rows (14336 x 4096 with two rows:
        // 12.3 bf16 / 16 fp32 in the small-batch kernel, 16.5 in the column kernel); on a K past 8192 not even one (that kernel walks
        // K with one workgroup per 64 columns, the small-batch kernel splits it: 8192 x 28672 30 against 37).  Up to 4096 columns,
        // 16 per workgroup: one and two rows at any K (4096 x 4096: 4.2 / 5.9 against 6.7 / 8.0; 4096 x 14336: 9.0 / 14.2 against
        // 13.0 / 17.0), three and four fp32 rows up to K = 4096 (9.1 / 9.7 against 11.1 / 11.5).
        const bool long_k = k > 8192 && !qmm::kernel_disabled("gptq_long_k_mm");
        const bool cols16 = qmm::gemv_gptq_cols16_wanted(n, cfg->group_size) && !qmm::kernel_disabled("gptq_cols");
        const int mm_min = cols16 ? (lhs_dtype == QMM_F32 && k <= 4096 ? 5 : 3) : long_k ? 1 : (lhs_dtype == QMM_F32 ? 3 : 2);
        for (int64_t m0 = 0; m0 < m; m0 += 16) {
            int mt = (int)(m - m0 < 16 ? m - m0 : 16);
            bool handled = false;
            if (m >= mm_min) {
                hipError_t e = qmm::launch_gemv_gptq_mm((const char*)lhs + m0 * k * esz, lhs_dtype, (const uint32_t*)rhs[0],
                                                        (const uint16_t*)rhs[1], (const uint32_t*)rhs[2], mt, n, k,
                                                        cfg->group_size, out + m0 * n, n, workspace, s, &handled);
                if (e != hipSuccess) return hip_status(e, "qmm_matmul(GPTQ small batch)");
            }
            if (handled) continue;
            hipError_t e = qmm::launch_gemv_gptq((const char*)lhs + m0 * k * esz, lhs_dtype, (const uint32_t*)rhs[0],
                                                 (const uint16_t*)rhs[1], (const uint32_t*)rhs[2], mt, n, k,
                                                 cfg->group_size, out + m0 * n, n, s);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul(GPTQ)");
        }
        return QMM_OK;
    }

    int64_t epb, bpb;
    if (encoding == QMM_Q8_0 || encoding == QMM_Q8_K || !block_params(encoding, epb, bpb))
        return fail(QMM_ERR_INVALID, "qmm_matmul: unknown encoding %d", encoding);
    if (n_rhs != 1 || !rhs[0]) return fail(QMM_ERR_INVALID, "qmm_matmul: GGUF encodings take exactly one rhs tensor");
    if (k % epb)
        return fail(QMM_ERR_INVALID, "qmm_matmul: K=%lld is not a multiple of the block size %lld", (long long)k,
                    (long long)epb);
    const uint8_t* w = (const uint8_t*)rhs[0];
    if ((encoding == QMM_Q4_K || encoding == QMM_Q5_K) && !aligned(w, 16))
        return fail(QMM_ERR_INVALID, "qmm_matmul: Q4_K / Q5_K rhs must be 16-byte aligned");
    if (!aligned(w, 2)) return fail(QMM_ERR_INVALID, "qmm_matmul: rhs must be 2-byte aligned");

    if (flags & QMM_FLAG_ACT_Q8K) {
        if (encoding != QMM_Q4_K && encoding != QMM_Q5_K && encoding != QMM_Q6_K)
            return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul: Q8_K activations go with Q4_K, Q5_K and Q6_K weights");
        if (q8k_integer_kernel(encoding, m, k) && encoding == QMM_Q4_K) {
            for (int64_t m0 = 0; m0 < m; m0 += 4) {
                bool handled = false;
                hipError_t e = qmm::launch_gemv_q4_k_q8k((const char*)lhs + m0 * k * esz, lhs_dtype, w, (int)std::min<int64_t>(4, m - m0), n, k,
                                                         out + m0 * n, n, s, &handled);
                if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_K x Q8_K)");
                if (!handled) return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul: Q4_K x Q8_K shape not taken (M=%lld K=%lld)", (long long)m, (long long)k);
            }
            return QMM_OK;
        }
        if (q8k_integer_kernel(encoding, m, k)) {
            if (encoding == QMM_Q5_K && !aligned(w, 16)) return fail(QMM_ERR_INVALID, "qmm_matmul: Q5_K rhs must be 16-byte aligned");
            const qmm::Q8KPlanes p = qmm::q8k_planes(workspace, m, k);
            hipError_t e = qmm::launch_quantize_q8_k_planes(lhs, lhs_dtype, m, k, p, s);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q8_K planes)");
            for (int64_t m0 = 0; m0 < m; m0 += 4) {
                e = qmm::launch_gemv_kquant_q8k(encoding, p, m0, (int)std::min<int64_t>(4, m - m0), w, n, k, out + m0 * n, n, s);
                if (e != hipSuccess) return hip_status(e, "qmm_matmul(K-quant x Q8_K)");
            }
            return QMM_OK;
        }
        // the quantised activations as fp32 rows (d8 * code), then the floating-point path on them: the products are those of
        // the integer treatment, summed in fp32
        const int64_t ybytes = up256(m * k * 4);
        float* y = (float*)workspace;
        hipError_t e = qmm::launch_q8k_round_trip(lhs, lhs_dtype, m, k, y, s);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q8_K round trip)");
        return matmul_f32(encoding, cfg, y, QMM_F32, m, k, rhs, n_rhs, n, out, (char*)workspace + ybytes, workspace_bytes - ybytes, 0, stream);
    }
    // a few lhs rows
    if (small_wanted(encoding, lhs_dtype, m, n, k, w)) {
        const bool parts = workspace && aligned(workspace, 256) && workspace_bytes >= qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, n, k);
        return hip_status(qmm::launch_gemv_kquant_small(encoding, lhs, lhs_dtype, 1, rhs, &n, &out, m, k, false, out16 != nullptr, parts ? workspace : nullptr, s),
                          "qmm_matmul(K-quant small batch)");
    }
    // from a few to a few hundred lhs rows
    if (direct_serves(encoding, cfg, lhs_dtype, m, n, k, w, workspace, workspace_bytes))
        return hip_status(qmm::launch_gemm_direct(encoding, lhs, lhs_dtype, 1, rhs, &n, &out, nullptr, nullptr, 0, m, k, out16, workspace, s), "qmm_matmul(direct GEMM)");
    // Q5_K and Q6_K with many lhs rows, Q4_K with more than 512 on large matrices: weights to fp16 integer planes in the workspace,
    // then the matrix cores
    if (kquant_planes(encoding, lhs_dtype, m, n, k))
        return hip_status(qmm::launch_gemm_planes(encoding, lhs, lhs_dtype, w, m, n, k, out, workspace, s), "qmm_matmul(K-quant planes GEMM)");
    // Q5_K with several lhs rows: the small-batch matrix-core kernel (passes of 16 or 8 rows)
    if (encoding == QMM_Q5_K && q5k_mm_wanted(lhs_dtype, m, n, k) && qmm::gemv_q5_k_mm_supported(w, m, n, k))
        return hip_status(qmm::launch_gemv_q5_k_mm(lhs, lhs_dtype, w, (int)m, n, k, out, n, workspace, s), "qmm_matmul(Q5_K small batch)");
    if (encoding == QMM_Q5_K) {
        // a decode-shaped kernel; a pass takes as many lhs rows as fit its LDS copy of the lhs
        const int64_t ngroups = (k / 256 + 15) / 16;
        const int64_t pass = ngroups <= 2 ? 4 : ngroups <= 4 ? 2 : 1;
        if (ngroups > 8) return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul: Q5_K takes K <= 32768 (K = %lld)", (long long)k);
        for (int64_t m0 = 0; m0 < m; m0 += pass) {
            bool handled = false;
            hipError_t e = qmm::launch_gemv_q5_k((const char*)lhs + m0 * k * esz, lhs_dtype, w, (int)std::min<int64_t>(pass, m - m0), n, k,
                                                 out + m0 * n, n, s, &handled);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q5_K)");
            if (!handled) return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul: Q5_K shape not taken (M=%lld K=%lld)", (long long)m, (long long)k);
        }
        return QMM_OK;
    }
    if (encoding == QMM_Q4_0 && qmm::gemm_q4_0_planes_wanted(m, n, k))
        return hip_status(qmm::launch_gemm_q4_0_planes(lhs, lhs_dtype, w, m, n, k, out, workspace, s), "qmm_matmul(Q4_0 plane GEMM)");
    // (two rows and more on a K beyond what the decode kernel takes: the matrix-core kernel too, 4096 x 14336 with 4 rows 32 -> 16 us)
    // (three and four rows on a K beyond 4096 as well: 8192 x 8192 with 4 rows 34.8 -> 14.4 us, 5120 x 5120 18.1 -> 12.2)
    if (encoding == QMM_Q4_0 && (m >= 5 || (m >= 2 && k > 8192 && k % 256 == 0) || (m >= 3 && k > 4096 && k % 256 == 0)) && !qmm::kernel_disabled("q4_0_mfma"))
        return hip_status(qmm::launch_gemm_q4_0(lhs, lhs_dtype, w, m, n, k, out, workspace, s), "qmm_matmul(Q4_0 int8 MFMA)");
    if (encoding == QMM_Q4_0 && m <= 4) {
        // decode: the kernel that quantises the lhs itself (takes K <= 8192)
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_0_stream(lhs, lhs_dtype, w, (int)m, n, k, out, n, s, &handled);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_0 decode)");
        if (handled) return QMM_OK;
    }
    if (encoding == QMM_Q4_0) {
        Q8Planes p = q8_planes(workspace, m, k);
        hipError_t e = qmm::launch_quantize_q8_0(lhs, lhs_dtype, m, k, nullptr, p.codes, p.scale, p.sum, s);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q8_0 quantise)");
        for (int64_t m0 = 0; m0 < m; m0 += 16) {
            int mt = (int)(m - m0 < 16 ? m - m0 : 16);
            e = qmm::launch_gemv_q4_0(p.codes + m0 * k, p.scale + m0 * (k / 32), p.sum + m0 * (k / 32), w, mt, n, k,
                                      out + m0 * n, n, s);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_0)");
        }
        return QMM_OK;
    }

    // 2..4 lhs rows on a small matrix: the decode kernel with one sub-block per lane (the activations of four rows fit a
    // lane's registers)
    if (encoding == QMM_Q4_K && m >= 2 && m <= 4 && q4k_lanes_rows_wins(n, k)) {
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_k_lanes_rows(lhs, lhs_dtype, w, (int)m, n, k, out, n, s, &handled);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_K decode, 2..4 rows)");
        if (handled) return QMM_OK;
    }
    // 2..16 lhs rows on few weight rows and long K: the small-batch kernel that cuts K across workgroups
    if (encoding == QMM_Q4_K && m >= 2 && m <= 16 && q4k_kc_wins(lhs_dtype, m, n, k) && qmm::gemv_q4_k_kc_supported(w, k)) {
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_k_kc(lhs, lhs_dtype, w, (int)m, n, k, out, n, workspace, s, &handled);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul(Q4_K small batch, K chunks)");
        if (handled) return QMM_OK;
    }
    // more than 16 lhs rows, and 9..16 fp32 rows on a large matrix with a long K: the prefill kernel
    if (q4k_gemm_from_9_rows(encoding, lhs_dtype, m, n, k))
        return hip_status(qmm::launch_gemm_q4_k(lhs, lhs_dtype, w, m, n, k, out, workspace, s), "qmm_matmul(Q4_K GEMM)");
    if (encoding == QMM_Q4_K && m > 16)
        return hip_status(qmm::launch_gemm_q4_k(lhs, lhs_dtype, w, m, n, k, out, workspace, s), "qmm_matmul(Q4_K GEMM)");

    // Q6_K with 2..64 lhs rows: the small-batch matrix-core kernel (passes of 16 or 8 rows)
    if (encoding == QMM_Q6_K && q6k_mm_wanted(m, n, k) && qmm::gemv_q6_k_mm_supported(w, m, n, k))
        return hip_status(qmm::launch_gemv_q6_k_mm(lhs, lhs_dtype, w, (int)m, n, k, out, n, workspace, s), "qmm_matmul(Q6_K small batch)");

    // (Q6_K with more than four rows on a long K that is no multiple of 2048: passes of four rows through the kernel that stages
    // the lhs, not the first-version kernel on all of them: 4096 x 11008 with 8 rows 102 -> 73 us)
    const int64_t pass = encoding == QMM_Q6_K && m > 4 && k % 2048 != 0 && k > 8192 ? 4 : 16;
    for (int64_t m0 = 0; m0 < m; m0 += pass) {
        int mt = (int)(m - m0 < pass ? m - m0 : pass);
        const void* a = (const char*)lhs + m0 * k * esz;
        hipError_t e = encoding == QMM_Q4_K ? qmm::launch_gemv_q4_k(a, lhs_dtype, w, mt, n, k, out + m0 * n, n, s)
                                            : qmm::launch_gemv_q6_k(a, lhs_dtype, w, mt, n, k, out + m0 * n, n, s);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul");
    }
    return QMM_OK;
}

int64_t qmm_matmul_rmsnorm_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    if (m <= 0 || k <= 0) return 0;
    return up256(m * k * (lhs_dtype == QMM_F32 ? 4 : 2)) + required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
}

int qmm_matmul_rmsnorm(int encoding, const qmm_gptq_config* cfg, const void* x, int x_dtype, const float* gamma, float eps, int64_t m,
                       int64_t k, const void* const* rhs, int n_rhs, int64_t n, float* out, void* workspace, int64_t workspace_bytes,
                       int flags, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (!x || !gamma || !rhs || !out) return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: null pointer");
    if (m <= 0 || n <= 0 || k <= 0 || m > INT32_MAX || n > INT32_MAX || k > INT32_MAX)
        return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: M=%lld N=%lld K=%lld out of range", (long long)m, (long long)n, (long long)k);
    if (x_dtype != QMM_F32 && x_dtype != QMM_BF16) return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: x dtype must be f32 or bf16");
    if (!aligned(x, 16) || !aligned(gamma, 4)) return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: x must be 16-byte aligned, gamma 4-byte aligned");
    if (!(eps >= 0.0f)) return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: eps must be non-negative");
    // One launch: the Q4_0 decode kernel normalises the rows it quantises anyway.
    if (encoding == QMM_Q4_0 && m <= 4 && flags == 0 && n_rhs == 1 && rhs[0] && k % 32 == 0 && aligned(rhs[0], 2)) {
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_0_stream(x, x_dtype, (const uint8_t*)rhs[0], (int)m, n, k, out, n, s, &handled, gamma, eps);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul_rmsnorm(Q4_0 decode)");
        if (handled) return QMM_OK;
    }
    // Otherwise: normalised rows into the workspace, then the matmul on them.
    const int64_t ybytes = up256(m * k * (x_dtype == QMM_F32 ? 4 : 2));
    const int64_t need = ybytes + required_bytes_flags(encoding, x_dtype, m, n, k, flags);
    if (!workspace || workspace_bytes < need)
        return fail(QMM_ERR_WORKSPACE, "qmm_matmul_rmsnorm: workspace of %lld bytes required (qmm_matmul_rmsnorm_workspace_bytes), %lld given",
                    (long long)need, (long long)workspace_bytes);
    if (!aligned(workspace, 256)) return fail(QMM_ERR_INVALID, "qmm_matmul_rmsnorm: workspace must be 256-byte aligned");
    hipError_t e = qmm::launch_rmsnorm(x, x_dtype, gamma, eps, m, k, workspace, s);
    if (e != hipSuccess) return hip_status(e, "qmm_matmul_rmsnorm(normalise)");
    return qmm_matmul(encoding, cfg, workspace, x_dtype, m, k, rhs, n_rhs, n, out, (char*)workspace + ybytes, workspace_bytes - ybytes, flags, stream);
}

int qmm_matmul_static(int encoding, const qmm_gptq_config* cfg, const void* lhs, int lhs_dtype, int64_t m, int64_t k,
                      const void* const* rhs, int n_rhs, int64_t n, float* out, int flags, void* stream) {
    int64_t need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    const TwinRowsScope twin(need > (int64_t)QMM_STATIC_SCRATCH_BYTES);  // (the two-pass treatment of an fp32 lhs needs less)
    if (need > (int64_t)QMM_STATIC_SCRATCH_BYTES) need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    if (need > (int64_t)QMM_STATIC_SCRATCH_BYTES && (encoding == QMM_Q4_K || encoding == QMM_GPTQ)) {
        const OptionalPlanesScope no_planes(true);  // the kernels that need no weight planes
        need = required_bytes_flags(encoding, lhs_dtype, m, n, k, flags);
    }
    if (need > (int64_t)QMM_STATIC_SCRATCH_BYTES)
        return fail(QMM_ERR_WORKSPACE,
                    "qmm_matmul_static: this problem needs %lld bytes of scratch and the static buffer holds %lld; "
                    "use qmm_matmul with a workspace of the caller's",
                    (long long)need, (long long)QMM_STATIC_SCRATCH_BYTES);
    void* ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    return qmm_matmul(encoding, cfg, lhs, lhs_dtype, m, k, rhs, n_rhs, n, out, ws, (int64_t)QMM_STATIC_SCRATCH_BYTES, flags, stream);
}

// Weight planes kept across calls.  The buffer starts with a 256-byte record of what it was made for; the planes follow.
namespace {
constexpr int64_t kPackHeaderBytes = 256;
constexpr uint32_t kPackMagic = 0x504D4D51u;  // "QMMP"
constexpr uint32_t kPackLayout = 1;           // bumped whenever the plane layouts change
struct PackHeader {
    uint32_t magic, layout;
    int32_t encoding, group;
    int64_t n, k, bytes;
};
static_assert(sizeof(PackHeader) <= kPackHeaderBytes, "header fits its 256 bytes");
__host__ __device__ inline bool same_header(const PackHeader& a, const PackHeader& b) {
    return a.magic == b.magic && a.layout == b.layout && a.encoding == b.encoding && a.group == b.group && a.n == b.n && a.k == b.k &&
           a.bytes == b.bytes;
}
PackHeader make_header(int encoding, const qmm_gptq_config* cfg, int64_t n, int64_t k, int64_t bytes) {
    PackHeader h;
    h.magic = kPackMagic;
    h.layout = kPackLayout;
    h.encoding = encoding;
    h.group = encoding == QMM_GPTQ && cfg ? cfg->group_size : 0;
    h.n = n;
    h.k = k;
    h.bytes = bytes;
    return h;
}
__global__ void pack_header_write_kernel(PackHeader* at, const PackHeader h) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *at = h;
}
// Runs behind the kernels of a qmm_matmul_repacked call.  A buffer whose record says another encoding, shape or group than the
// call (planes of the same size made for something else pass every host-side check) turns the whole result into NaN: a
// wrong buffer cannot pass for a right one.
__global__ __launch_bounds__(256) void pack_header_check_kernel(const PackHeader* at, const PackHeader want, float* out, int64_t count) {
    const PackHeader have = *at;
    if (same_header(have, want)) return;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) out[i] = __uint_as_float(0x7fc00000u);
}
}  // namespace

static bool repackable(int encoding, const qmm_gptq_config* cfg, int64_t n, int64_t k) {
    if (n <= 0 || k < 256 || k % 256 || n > INT32_MAX || k > INT32_MAX) return false;
    if (encoding == QMM_GPTQ) return cfg && cfg->bits == 4 && !cfg->desc_act && qmm::gptq_planes_supported(n, k, cfg->group_size);
    return encoding == QMM_Q4_K || encoding == QMM_Q5_K || encoding == QMM_Q6_K || encoding == QMM_Q4_0;
}

static int64_t repack_plane_bytes(int encoding, int64_t n, int64_t k) {
    if (encoding == QMM_Q4_0) return qmm::repacked_q4_0_bytes(n, k);
    return encoding == QMM_GPTQ ? qmm::repacked_gptq_bytes(n, k) : qmm::repacked_planes_bytes(encoding, n, k);
}

int64_t qmm_repack_bytes(int encoding, const qmm_gptq_config* cfg, int64_t n, int64_t k) {
    if (!repackable(encoding, cfg, n, k)) return 0;
    return kPackHeaderBytes + repack_plane_bytes(encoding, n, k);
}

int qmm_repack_check(int encoding, const qmm_gptq_config* cfg, int64_t n, int64_t k, const void* packed, int64_t packed_bytes,
                     void* stream) {
    if (!packed) return fail(QMM_ERR_INVALID, "qmm_repack_check: null pointer");
    if (!repackable(encoding, cfg, n, k))
        return fail(QMM_ERR_UNSUPPORTED, "qmm_repack_check: no weight planes for encoding %d with N=%lld K=%lld", encoding, (long long)n, (long long)k);
    const int64_t need = qmm_repack_bytes(encoding, cfg, n, k);
    if (packed_bytes < need || !aligned(packed, 256))
        return fail(QMM_ERR_INVALID, "qmm_repack_check: the packed buffer must be 256-byte aligned and hold qmm_repack_bytes = %lld bytes (%lld given)",
                    (long long)need, (long long)packed_bytes);
    PackHeader have;
    hipError_t e = hipMemcpyAsync(&have, packed, sizeof(have), hipMemcpyDeviceToHost, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return hip_status(e, "qmm_repack_check");
    const PackHeader want = make_header(encoding, cfg, n, k, need);
    if (have.magic != kPackMagic) return fail(QMM_ERR_INVALID, "qmm_repack_check: the buffer does not start with the record qmm_repack writes");
    if (!same_header(have, want))
        return fail(QMM_ERR_INVALID, "qmm_repack_check: the buffer holds planes of encoding %d, N=%lld, K=%lld, group %d, layout %u; the call names "
                                     "encoding %d, N=%lld, K=%lld, group %d, layout %u", have.encoding, (long long)have.n, (long long)have.k, have.group,
                    have.layout, want.encoding, (long long)want.n, (long long)want.k, want.group, want.layout);
    return QMM_OK;
}

int qmm_repack(int encoding, const qmm_gptq_config* cfg, const void* const* rhs, int n_rhs, int64_t n, int64_t k, void* packed,
               int64_t packed_bytes, void* stream) {
    if (!rhs || !packed) return fail(QMM_ERR_INVALID, "qmm_repack: null pointer");
    if (!repackable(encoding, cfg, n, k))
        return fail(QMM_ERR_UNSUPPORTED, "qmm_repack: no weight planes for encoding %d with N=%lld K=%lld (Q4_0, Q4_K, Q5_K, Q6_K, and 4-bit GPTQ with "
                                         "plain groups of 128 or 256; K a multiple of 256)", encoding, (long long)n, (long long)k);
    const int64_t need = qmm_repack_bytes(encoding, cfg, n, k);
    if (packed_bytes < need) return fail(QMM_ERR_WORKSPACE, "qmm_repack: %lld bytes required (qmm_repack_bytes), %lld given", (long long)need, (long long)packed_bytes);
    if (!aligned(packed, 256)) return fail(QMM_ERR_INVALID, "qmm_repack: the buffer must be 256-byte aligned");
    void* const planes = (char*)packed + kPackHeaderBytes;
    auto finish = [&](hipError_t e, const char* what) {
        if (e != hipSuccess) return hip_status(e, what);
        pack_header_write_kernel<<<dim3(1), dim3(64), 0, (hipStream_t)stream>>>((PackHeader*)packed, make_header(encoding, cfg, n, k, need));
        return hip_status(hipGetLastError(), "qmm_repack(record)");
    };
    if (encoding == QMM_GPTQ) {
        if (n_rhs != 3 && n_rhs != 4) return fail(QMM_ERR_INVALID, "qmm_repack: GPTQ takes rhs = (qweight, scales, qzeros[, g_idx]), got %d", n_rhs);
        if (int rc = check_gptq(cfg, n, k)) return rc;
        for (int i = 0; i < 3; i++)
            if (!rhs[i] || !aligned(rhs[i], 4)) return fail(QMM_ERR_INVALID, "qmm_repack: GPTQ rhs[%d] null or misaligned", i);
        return finish(qmm::launch_repack_gptq((const uint32_t*)rhs[0], (const uint16_t*)rhs[1], (const uint32_t*)rhs[2], n, k, cfg->group_size,
                                              planes, (hipStream_t)stream), "qmm_repack(GPTQ)");
    }
    if (n_rhs != 1 || !rhs[0]) return fail(QMM_ERR_INVALID, "qmm_repack: GGUF encodings take exactly one rhs tensor");
    if (!aligned(rhs[0], encoding == QMM_Q6_K || encoding == QMM_Q4_0 ? 2 : 16))
        return fail(QMM_ERR_INVALID, "qmm_repack: rhs misaligned (Q4_K / Q5_K 16 bytes, Q4_0 / Q6_K 2)");
    if (encoding == QMM_Q4_0)
        return finish(qmm::launch_repack_q4_0((const uint8_t*)rhs[0], n, k, planes, (hipStream_t)stream), "qmm_repack(Q4_0)");
    return finish(qmm::launch_repack_planes(encoding, (const uint8_t*)rhs[0], n, k, planes, (hipStream_t)stream), "qmm_repack");
}

// Does a call with these rows go through the planes?  Without the packed tensors every row count does.
// Q4_0: passes of the 16-row int8 kernel against the kept planes.  4096 x 4096: 28 us against 35 at 64 rows, 41 against 37 at 96;
// 4096 x 14336: 57 against 83 at 64 rows, 84 against 84 at 96.
static int64_t q4_0_repacked_min_rows(int64_t k) { return k > 4096 ? 96 : 80; }
// With the planes at hand the direct GEMM on the packed tensors still wins while the weights are most of the traffic (the planes are 2 or 4
// bytes a weight against 0.6 .. 0.8), and with fp32 rows, for which the planes are walked twice.  us, planes / direct:
// - up to 150 bf16 rows, or few results: Q5_K 4096 x 4096 128 rows 33 / 20; Q4_0 14336 x 4096 128 rows 60 / 42, 450 rows 94 / 138.
// - bf16 rows beyond: Q5_K 4096 x 4096 512 rows 54 / 37, 14336 x 4096 200 rows 75 / 49, 700 121 / 119, 1000 130 / 149; Q4_K 14336 x 4096 700 rows 121 / 108, 1000 128 / 134.
//   From some 256 rows on only for the staged kernel (Q6_K 14336 x 4096 400 rows 119 / 154 in the direct one, Q5_K 2560 x 14336 700 rows 105 / 196), and but for Q4_K
//   not on 100 M weights and more (Q5_K 28672 x 4096 512 rows 143 / 167, Q6_K 400 rows 224 / 298, GPTQ 28672 x 8192 512 rows 233 / 245).
// - fp32 rows: GPTQ 14336 x 4096 700 rows 260 / 173, 3000 rows 0.78 times as long; Q5_K 14336 x 4096 1400 rows 0.78, 3000 rows 0.87; on a longer K not
//   beyond 2048 rows (Q4_K 4096 x 14336 2048 rows 0.94, 2560 x 14336 3000 rows 1.13, 5120 x 8192 3000 rows 1.09).  Where planes served before the staged kernel and
//   are the more exact ones they still do: relative error, planes / direct, GPTQ 30424 x 512 700 rows 0.92e-7 / 1.07e-7, Q6_K 2056 x 256 2048 rows 1.38e-7 / 1.98e-7,
//   1536 x 1024 2048 rows 1.92e-7 / 2.00e-7 (but 14336 x 1024 2.6e-7 / 2.0e-7, K = 4096 5.5e-7 / 2.1e-7).
static bool direct_over_planes(int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    const bool narrow = m * n <= (int64_t)1300 << 10, q40 = encoding == QMM_Q4_0, f32 = lhs_dtype == QMM_F32 && !q40;
    if ((encoding == QMM_GPTQ && cfg->desc_act) || !direct_wanted(encoding, cfg, lhs_dtype, m, n, k)) return false;
    if (narrow || m <= (!f32 ? 150 : encoding == QMM_GPTQ ? 400 : 1400)) return true;
    if (q40) return false;
    if (f32) {
        if (encoding == QMM_GPTQ && k < 768) return false;
        if (encoding == QMM_Q6_K && (k < 768 || (k <= 1024 && m * n <= (int64_t)4 << 20))) return false;
        return k <= 4096 || m <= 2048;
    }
    if (m <= 256) return true;
    return m <= 768 && (encoding == QMM_Q4_K || n * k <= (int64_t)100 << 20) && qmm::gemm_direct_takes_staged(encoding, lhs_dtype, m, n, k, direct_group(cfg));
}
static bool repacked_path(int encoding, int64_t m, int64_t n, int64_t k, bool have_rhs) {
    if (!have_rhs) return true;
    if (encoding == QMM_Q4_0) return m > q4_0_repacked_min_rows(k);
    return encoding == QMM_GPTQ ? qmm::repacked_gptq_wanted(m, n) : qmm::repacked_planes_wanted(encoding, m, n, k);
}

int64_t qmm_matmul_repacked_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    if (m <= 0 || n <= 0 || k < 256 || k % 256) return 0;
    const int64_t planes = encoding == QMM_Q4_0 ? qmm::repacked_q4_0_workspace_bytes(m, n, k)
                           : encoding == QMM_GPTQ ? qmm::repacked_gptq_workspace_bytes(lhs_dtype, m, k)
                                                  : qmm::repacked_planes_workspace_bytes(encoding, lhs_dtype, m, n, k);
    if (repacked_path(encoding, m, n, k, true)) return planes;
    const OptionalPlanesScope no_planes(true);  // the other route: qmm_matmul's kernels on the packed tensors (or, without those, the planes)
    return std::max(planes, required_bytes(encoding, lhs_dtype, m, n, k));
}

int qmm_matmul_repacked(int encoding, const qmm_gptq_config* cfg, const void* lhs, int lhs_dtype, int64_t m, int64_t k,
                        const void* const* rhs, int n_rhs, const void* packed, int64_t packed_bytes, int64_t n, float* out,
                        void* workspace, int64_t workspace_bytes, int flags, void* stream) {
    if (!lhs || !packed || !out) return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: null pointer");
    if (flags) return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul_repacked: flags must be 0 (0x%x given)", flags);
    if (m <= 0 || m > INT32_MAX) return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: M=%lld", (long long)m);
    if (!repackable(encoding, cfg, n, k))
        return fail(QMM_ERR_UNSUPPORTED, "qmm_matmul_repacked: no weight planes for encoding %d with N=%lld K=%lld", encoding, (long long)n, (long long)k);
    if (packed_bytes < qmm_repack_bytes(encoding, cfg, n, k) || !aligned(packed, 256))
        return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: the packed buffer must be 256-byte aligned and hold qmm_repack_bytes = %lld bytes (%lld given)",
                    (long long)qmm_repack_bytes(encoding, cfg, n, k), (long long)packed_bytes);
    if (!repacked_path(encoding, m, n, k, rhs != nullptr) ||
        (rhs && direct_over_planes(encoding, cfg, lhs_dtype, m, n, k) && direct_serves(encoding, cfg, lhs_dtype, m, n, k, n_rhs > 0 ? rhs[0] : nullptr, workspace, workspace_bytes))) {
        const OptionalPlanesScope no_planes(true);
        return qmm_matmul(encoding, cfg, lhs, lhs_dtype, m, k, rhs, n_rhs, n, out, workspace, workspace_bytes, 0, stream);
    }
    if (lhs_dtype != QMM_F32 && lhs_dtype != QMM_BF16) return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: lhs dtype must be f32 or bf16");
    if (!aligned(lhs, 16) || !aligned(out, 4)) return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: lhs must be 16-byte aligned");
    const int64_t need = encoding == QMM_Q4_0 ? qmm::repacked_q4_0_workspace_bytes(m, n, k)
                         : encoding == QMM_GPTQ ? qmm::repacked_gptq_workspace_bytes(lhs_dtype, m, k)
                                                : qmm::repacked_planes_workspace_bytes(encoding, lhs_dtype, m, n, k);
    if (!workspace || workspace_bytes < need)
        return fail(QMM_ERR_WORKSPACE, "qmm_matmul_repacked: workspace of %lld bytes required, %lld given", (long long)need, (long long)workspace_bytes);
    if (!aligned(workspace, 256)) return fail(QMM_ERR_INVALID, "qmm_matmul_repacked: workspace must be 256-byte aligned");
    const void* const planes = (const char*)packed + kPackHeaderBytes;
    hipError_t e;
    if (encoding == QMM_Q4_0) e = qmm::launch_gemm_q4_0_repacked(lhs, lhs_dtype, planes, m, n, k, out, workspace, (hipStream_t)stream);
    else if (encoding == QMM_GPTQ) e = qmm::launch_gemm_gptq_repacked(lhs, lhs_dtype, planes, m, n, k, cfg->group_size, out, workspace, (hipStream_t)stream);
    else e = qmm::launch_gemm_planes_repacked(encoding, lhs, lhs_dtype, planes, m, n, k, out, workspace, (hipStream_t)stream);
    if (e != hipSuccess) return hip_status(e, "qmm_matmul_repacked");
    // the record at the head of the buffer against this call, on the device (the host never reads the buffer here)
    const int64_t count = m * n;
    pack_header_check_kernel<<<dim3((unsigned)std::min<int64_t>((count + 255) / 256, 1024)), dim3(256), 0, (hipStream_t)stream>>>(
        (const PackHeader*)packed, make_header(encoding, cfg, n, k, qmm_repack_bytes(encoding, cfg, n, k)), out, count);
    return hip_status(hipGetLastError(), "qmm_matmul_repacked(record check)");
}

int qmm_matmul_grouped(int encoding, const void* lhs, int lhs_dtype, int64_t m, int64_t k, int count,
                       const void* const* rhs, const int64_t* n, float* const* out, void* workspace,
                       int64_t workspace_bytes, void* stream) {
    if (!lhs || !rhs || !n || !out) return fail(QMM_ERR_INVALID, "qmm_matmul_grouped: null pointer");
    if (count < 1 || count > 64) return fail(QMM_ERR_INVALID, "qmm_matmul_grouped: count %d out of range (1..64)", count);
    int64_t epb, bpb;
    if (encoding == QMM_Q8_0 || encoding == QMM_Q8_K || encoding == QMM_GPTQ || !block_params(encoding, epb, bpb))
        return fail(QMM_ERR_INVALID, "qmm_matmul_grouped: encoding %d is not a GGUF weight encoding", encoding);
    for (int j = 0; j < count; j++)
        if (!rhs[j] || !out[j] || n[j] <= 0) return fail(QMM_ERR_INVALID, "qmm_matmul_grouped: matrix %d: null pointer or N <= 0", j);
    // Matrices that a call of their own would give to the small-batch kernel or to the direct GEMM go there together; the others, if any, then form their own group.
    if (m > 0 && m <= INT32_MAX && k > 0 && k <= INT32_MAX && (lhs_dtype == QMM_F32 || lhs_dtype == QMM_BF16) && aligned(lhs, 16)) {
        const void *direct_w[64], *rest_w[64];
        int64_t direct_n[64], rest_n[64];
        float *direct_out[64], *rest_out[64];
        int directs = 0, rest = 0;
        for (int j = 0; j < count; j++) {
            if (aligned(out[j], 4) && small_wanted(encoding, lhs_dtype, m, n[j], k, rhs[j])) direct_w[directs] = rhs[j], direct_n[directs] = n[j], direct_out[directs++] = out[j];
            else rest_w[rest] = rhs[j], rest_n[rest] = n[j], rest_out[rest++] = out[j];
        }
        for (int j = 0, take; j < directs; j += take) {
            take = std::min(qmm::kLanesMaxMats, directs - j);
            int64_t all = 0;
            for (int i = 0; i < take; i++) all += direct_n[j + i];
            const int64_t share = qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, all, k);  // (of groups of K side by side; the same sums without)
            void* const parts = share > 0 && workspace && aligned(workspace, 256) && workspace_bytes >= share ? workspace : nullptr;
            const hipError_t e = qmm::launch_gemv_kquant_small(encoding, lhs, lhs_dtype, take, direct_w + j, direct_n + j, direct_out + j, m, k, false, false, parts, (hipStream_t)stream);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul_grouped(K-quant small batch)");
        }
        if (directs > 0)
            return rest == 0 ? QMM_OK
                             : qmm_matmul_grouped(encoding, lhs, lhs_dtype, m, k, rest, rest_w, rest_n, rest_out, workspace, workspace_bytes, stream);
        rest = 0;
        for (int j = 0; j < count; j++) {
            if (aligned(rhs[j], 16) && aligned(out[j], 4) && n[j] <= INT32_MAX && direct_serves(encoding, nullptr, lhs_dtype, m, n[j], k, rhs[j], workspace, workspace_bytes))
                direct_w[directs] = rhs[j], direct_n[directs] = n[j], direct_out[directs++] = out[j];
            else rest_w[rest] = rhs[j], rest_n[rest] = n[j], rest_out[rest++] = out[j];
        }
        for (int j = 0; j < directs; j += qmm::kDirectMaxMats) {
            const hipError_t e = qmm::launch_gemm_direct(encoding, lhs, lhs_dtype, std::min(qmm::kDirectMaxMats, directs - j), direct_w + j, direct_n + j,
                                                         direct_out + j, nullptr, nullptr, 0, m, k, nullptr, workspace, (hipStream_t)stream);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul_grouped(direct GEMM)");
        }
        if (directs > 0)
            return rest == 0 ? QMM_OK
                             : qmm_matmul_grouped(encoding, lhs, lhs_dtype, m, k, rest, rest_w, rest_n, rest_out, workspace, workspace_bytes, stream);
    }
    if (encoding == QMM_Q4_K && m >= 1 && m <= 4 && k > 0 && k % 256 == 0 && count <= qmm::kLanesMaxMats &&
        (lhs_dtype == QMM_F32 || lhs_dtype == QMM_BF16) && aligned(lhs, 16)) {
        bool ok = true;
        int64_t total = 0;
        const uint8_t* ws[qmm::kLanesMaxMats];
        for (int j = 0; j < count; j++) {
            ok = ok && aligned(rhs[j], 16) && aligned(out[j], 4);
            total += n[j];
            ws[j] = (const uint8_t*)rhs[j];
        }
        if (ok && total <= INT32_MAX && m == 1) {
            bool handled = false;
            hipError_t e = qmm::launch_gemv_q4_k_lanes_grouped(lhs, lhs_dtype, count, ws, n, out, 1, k, 0, (hipStream_t)stream, &handled);
            if (e != hipSuccess) return hip_status(e, "qmm_matmul_grouped(Q4_K decode)");
            if (handled) return QMM_OK;
        }
        if (ok && total <= INT32_MAX && m >= 2 && m <= 4) {
            // Each matrix goes to the kernel qmm_matmul would give it, so a group and separate calls agree bit for bit:
            // the small ones as one launch of the decode kernel, the others (below) one by one.
            const uint8_t* small_w[qmm::kLanesMaxMats];
            int64_t small_n[qmm::kLanesMaxMats];
            float* small_out[qmm::kLanesMaxMats];
            int small = 0;
            for (int j = 0; j < count; j++)
                if (q4k_lanes_rows_wins(n[j], k)) small_w[small] = ws[j], small_n[small] = n[j], small_out[small++] = out[j];
            bool handled = false;
            if (small > 0) {
                hipError_t e = qmm::launch_gemv_q4_k_lanes_rows_grouped(lhs, lhs_dtype, small, small_w, small_n, small_out, (int)m, k, 0,
                                                                        (hipStream_t)stream, &handled);
                if (e != hipSuccess) return hip_status(e, "qmm_matmul_grouped(Q4_K decode, 2..4 rows)");
            }
            if (handled) {
                if (small == count) return QMM_OK;
                int rest = 0;
                const void* rest_w[qmm::kLanesMaxMats];
                int64_t rest_n[qmm::kLanesMaxMats];
                float* rest_out[qmm::kLanesMaxMats];
                for (int j = 0; j < count; j++)
                    if (!q4k_lanes_rows_wins(n[j], k)) rest_w[rest] = rhs[j], rest_n[rest] = n[j], rest_out[rest++] = out[j];
                return qmm_matmul_grouped(encoding, lhs, lhs_dtype, m, k, rest, rest_w, rest_n, rest_out, workspace, workspace_bytes, stream);
            }
        }
    }
    for (int j = 0; j < count; j++) {
        const void* one[1] = {rhs[j]};
        if (int rc = qmm_matmul(encoding, nullptr, lhs, lhs_dtype, m, k, one, 1, n[j], out[j], workspace, workspace_bytes, 0, stream))
            return rc;
    }
    return QMM_OK;
}

// What separate calls need at most, and what matrices that share a launch of the kernel for few rows need for their groups of K next to each other.
int64_t qmm_matmul_grouped_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t k, int count, const int64_t* n) {
    if (!n || count < 1 || count > 64) return 0;
    int64_t need = 0, all = 0;
    int taken = 0;
    for (int j = 0; j < count; j++) {
        need = std::max(need, qmm_preferred_workspace_bytes(QMM_OP_MATMUL, encoding, nullptr, lhs_dtype, m, n[j], k, 0));
        if (m <= 0 || n[j] <= 0 || k <= 0 || !small_wanted(encoding, lhs_dtype, m, n[j], k, nullptr)) continue;  // (the weights' alignment is not known here)
        all += n[j];
        need = std::max(need, qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, all, k));
        if (++taken % qmm::kLanesMaxMats == 0) all = 0;
    }
    return need;
}

int64_t qmm_matmul_swiglu_workspace_bytes(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    // one lhs row of Q4_K goes through the decode kernel with the combination as its epilogue: nothing to keep
    if (encoding == QMM_Q4_K && m == 1 && k % 256 == 0 && k <= 16384) return 0;
    return align_up(required_bytes(encoding, lhs_dtype, m, n, k), 256) + 2 * align_up(m * n * 4, 256);
}

// What gate and up side by side take for their groups of K (0: not so, or one group).
static int64_t swiglu_share(int encoding, int lhs_dtype, int64_t m, int64_t n, int64_t k) {
    return small_wanted(encoding, lhs_dtype, m, n, k, nullptr) ? qmm::gemv_kquant_small_workspace_bytes(encoding, lhs_dtype, m, 2 * n, k) : 0;
}

int qmm_matmul_swiglu(int encoding, const void* lhs, int lhs_dtype, int64_t m, int64_t k, const void* gate, const void* up,
                      int64_t n, float* out, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!lhs || !gate || !up || !out) return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: null pointer");
    int64_t epb, bpb;
    if (encoding == QMM_Q8_0 || encoding == QMM_Q8_K || encoding == QMM_GPTQ || !block_params(encoding, epb, bpb))
        return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: encoding %d is not a GGUF weight encoding", encoding);
    if (m <= 0 || n <= 0 || k <= 0 || k % epb || m > INT32_MAX || n > INT32_MAX / 2 || k > INT32_MAX)
        return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: M=%lld N=%lld K=%lld (K a positive multiple of %lld)", (long long)m,
                    (long long)n, (long long)k, (long long)epb);
    if (lhs_dtype != QMM_F32 && lhs_dtype != QMM_BF16) return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: lhs dtype must be f32 or bf16");
    if (!aligned(lhs, 16) || !aligned(out, 4)) return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: lhs must be 16-byte aligned");
    if (encoding == QMM_Q4_K && m == 1 && k % 256 == 0 && aligned(gate, 16) && aligned(up, 16)) {
        const uint8_t* ws[2] = {(const uint8_t*)gate, (const uint8_t*)up};
        const int64_t ns[2] = {n, n};
        float* outs[2] = {out, out};
        bool handled = false;
        hipError_t e = qmm::launch_gemv_q4_k_lanes_grouped(lhs, lhs_dtype, 2, ws, ns, outs, 1, k, 0, (hipStream_t)stream, &handled, true);
        if (e != hipSuccess) return hip_status(e, "qmm_matmul_swiglu(Q4_K decode)");
        if (handled) return QMM_OK;
    }
    // two products into the workspace, then the combination (all that the caller gave beyond the products is the matmuls' workspace)
    int64_t mm_ws = align_up(required_bytes(encoding, lhs_dtype, m, n, k), 256);
    const int64_t plane = align_up(m * n * 4, 256);
    if (workspace_bytes > mm_ws + 2 * plane) mm_ws = (workspace_bytes - 2 * plane) / 256 * 256;
    if (!workspace || workspace_bytes < mm_ws + 2 * plane)
        return fail(QMM_ERR_WORKSPACE, "qmm_matmul_swiglu: workspace of %lld bytes required, %lld given", (long long)(mm_ws + 2 * plane),
                    (long long)workspace_bytes);
    if (!aligned(workspace, 256)) return fail(QMM_ERR_INVALID, "qmm_matmul_swiglu: workspace must be 256-byte aligned");
    // where the small-batch kernel would serve both products (but for groups of K side by side: 1024 x 14336 16 bf16 rows 32 us here, 18 as two products)
    if (small_wanted(encoding, lhs_dtype, m, n, k, gate) && small_wanted(encoding, lhs_dtype, m, n, k, up) && (swiglu_share(encoding, lhs_dtype, m, n, k) == 0 || swiglu_share(encoding, lhs_dtype, m, n, k) > mm_ws)) {
        const void* const both[2] = {gate, up};
        const int64_t ns[2] = {n, n};
        float* const outs[2] = {out, out};
        return hip_status(qmm::launch_gemv_kquant_small(encoding, lhs, lhs_dtype, 2, both, ns, outs, m, k, true, false, nullptr, (hipStream_t)stream), "qmm_matmul_swiglu(K-quant small batch)");
    }
    float* g = (float*)((char*)workspace + mm_ws);
    float* u = (float*)((char*)workspace + mm_ws + plane);
    // (one launch for both products where a kernel takes matrices that share their lhs: Q4_K with 2..16 rows)
    const void* both[2] = {gate, up};
    const int64_t ns[2] = {n, n};
    float* outs[2] = {g, u};
    if (int rc = qmm_matmul_grouped(encoding, lhs, lhs_dtype, m, k, 2, both, ns, outs, workspace, mm_ws, stream)) return rc;
    return hip_status(qmm::launch_swiglu(g, u, out, m * n, (hipStream_t)stream), "qmm_matmul_swiglu(combine)");
}

int qmm_block_dots_q4_0(const void* lhs_q8_0, const void* rhs_q4_0, int64_t m, int64_t n, int64_t k, int32_t* out,
                        void* stream) {
    if (!lhs_q8_0 || !rhs_q4_0 || !out) return fail(QMM_ERR_INVALID, "qmm_block_dots_q4_0: null pointer");
    if (m <= 0 || n <= 0 || k <= 0 || k % 32) return fail(QMM_ERR_INVALID, "qmm_block_dots_q4_0: bad shape");
    return hip_status(qmm::launch_block_dots_q4_0((const uint8_t*)lhs_q8_0, (const uint8_t*)rhs_q4_0, m, n, k, out,
                                                  (hipStream_t)stream),
                      "qmm_block_dots_q4_0");
}

int64_t qmm_preferred_workspace_bytes(int op, int encoding, const qmm_gptq_config* cfg, int lhs_dtype, int64_t m, int64_t n, int64_t k, int flags) {
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    switch (op) {
        case QMM_OP_MATMUL: return preferred_matmul(encoding, cfg, lhs_dtype, m, n, k, flags);
        case QMM_OP_RMSNORM: return up256(m * k * (lhs_dtype == QMM_F32 ? 4 : 2)) + preferred_matmul(encoding, cfg, lhs_dtype, m, n, k, flags);
        case QMM_OP_SWIGLU: {
            const int64_t need = qmm_matmul_swiglu_workspace_bytes(encoding, lhs_dtype, m, n, k);
            return need ? std::max(need, std::max(up256(preferred_matmul(encoding, cfg, lhs_dtype, m, n, k, 0)), up256(swiglu_share(encoding, lhs_dtype, m, n, k))) + 2 * up256(m * n * 4)) : 0;
        }
        case QMM_OP_REPACKED: {
            const int64_t need = qmm_matmul_repacked_workspace_bytes(encoding, lhs_dtype, m, n, k);
            return repacked_path(encoding, m, n, k, true) && !direct_over_planes(encoding, cfg, lhs_dtype, m, n, k) ? need : std::max(need, preferred_matmul(encoding, cfg, lhs_dtype, m, n, k, 0));
        }
        default: return 0;
    }
}

}  // extern "C"
