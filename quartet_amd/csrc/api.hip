// C ABI of libquartet_hip.so: argument validation + dispatch to the kernels.
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <mutex>

#include "../../include/quartet_hip.h"
#include "qm_kernels.h"
#include "qm_math.h"
#include "shape_table.h"

namespace {

thread_local char g_last_error[256] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
    va_end(ap);
    return code;
}

int from_hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return 0;
    snprintf(g_last_error, sizeof(g_last_error), "%s: %s", what, hipGetErrorString(e));
    return (int)e;
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
bool valid_hd(int hd) { return hd == 32 || hd == 64 || hd == 128; }
bool valid_dtype(int d) { return d == QM_BF16 || d == QM_F32; }
bool valid_mode(int m) { return m >= QM_QUEST_RTN && m <= QM_QUEST_SR; }
bool valid_layout(int l) { return l == QM_LAYOUT_ROWMAJOR || l == QM_LAYOUT_TILED; }
bool valid_layer_layout(int l) { return valid_layout(l) || l == QM_LAYOUT_PADDED; }

qm::SignBits make_signs(const uint32_t* sign_bits, int hd) {
    qm::SignBits sb{{0u, 0u, 0u, 0u}};
    if (sign_bits)
        for (int i = 0; i < (hd + 31) / 32; ++i) sb.w[i] = sign_bits[i];
    return sb;
}

}  // namespace

extern "C" {

int qm_version(void) { return 16; }

const char* qm_last_error(void) { return g_last_error; }

int qm_quantize_mxfp4(const void* x, int x_dtype, int64_t rows, int64_t cols, int hadamard_dim,
                      const uint32_t* sign_bits, int mode, int transposed_in, const float* u, uint64_t seed,
                      uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant, int codes_layout, void* stream) {
    if (!valid_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: unknown codes_layout %d", codes_layout);
    if (!valid_dtype(x_dtype)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: x_dtype %d is not QM_BF16/QM_F32", x_dtype);
    if (!valid_hd(hadamard_dim) && hadamard_dim != 1)
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: hadamard_dim %d not in {1,32,64,128}", hadamard_dim);
    if (hadamard_dim == 1 && (transposed_in || u || sign_bits || codes_layout != QM_LAYOUT_ROWMAJOR || cols % 32 ||
                              !aligned(codes, 16) || !aligned(maskbits, 4)))
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: hadamard_dim 1 (input already rotated) needs row-major input and codes, "
                                    "cols %% 32 == 0, no sign bits, no explicit uniforms, 16-byte aligned codes");
    if (!valid_mode(mode)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: unknown mode %d", mode);
    if (rows < 0 || cols < 0) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: negative shape [%lld, %lld]", (long long)rows, (long long)cols);
    if (cols % hadamard_dim) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: cols %lld not a multiple of hadamard_dim %d", (long long)cols, hadamard_dim);
    if (rows == 0 || cols == 0) return 0;
    if (!x || !codes || !scales) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: x, codes and scales must be non-null");
    if (transposed_in && rows % 8) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: transposed input needs rows %% 8 == 0 (got %lld)", (long long)rows);
    if (!aligned(x, 16) || !aligned(codes, 4) || (dequant && !aligned(dequant, 16)) || (u && !aligned(u, 16)))
        return fail(QM_ERR_UNALIGNED, "qm_quantize_mxfp4: x/dequant/u need 16-byte and codes 4-byte alignment");
    if (codes_layout == QM_LAYOUT_TILED &&
        (!qm::quantize_supports_tiled(rows, cols, hadamard_dim, mode, transposed_in != 0, u, maskbits) || !aligned(codes, 16) ||
         !aligned(scales, 4) || !aligned(maskbits, 4)))
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4: tiled codes need hadamard_dim 32, rows %% 16 == 0, cols %% 128 == 0, "
                                    "no explicit uniforms, no mask with transposed input, 16-byte aligned codes (rows=%lld cols=%lld)",
                    (long long)rows, (long long)cols);
    return from_hip(qm::quantize_mxfp4(x, x_dtype, rows, cols, hadamard_dim, make_signs(sign_bits, hadamard_dim), mode,
                                       transposed_in != 0, u, seed, codes, scales, maskbits, dequant, codes_layout,
                                       reinterpret_cast<hipStream_t>(stream)),
                    "qm_quantize_mxfp4");
}

int qm_pseudo_quantize_mxfp4(const void* x, int x_dtype, int64_t rows, int64_t cols, int hadamard_dim, const uint32_t* sign_bits, int mode,
                             uint64_t seed, uint8_t* maskbits, void* dequant, void* stream) {
    if (!valid_dtype(x_dtype)) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: x_dtype %d is not QM_BF16/QM_F32", x_dtype);
    if (!valid_hd(hadamard_dim)) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: hadamard_dim %d not in {32,64,128}", hadamard_dim);
    if (!valid_mode(mode)) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: unknown mode %d", mode);
    if (rows < 0 || cols < 0) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: negative shape [%lld, %lld]", (long long)rows, (long long)cols);
    if (cols % hadamard_dim) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: cols %lld not a multiple of hadamard_dim %d", (long long)cols, hadamard_dim);
    if (rows == 0 || cols == 0) return 0;
    if (!x || !dequant) return fail(QM_ERR_INVALID, "qm_pseudo_quantize_mxfp4: x and dequant must be non-null");
    if (!aligned(x, 16) || !aligned(dequant, 16) || !aligned(maskbits, 4))
        return fail(QM_ERR_UNALIGNED, "qm_pseudo_quantize_mxfp4: x and dequant need 16-byte, maskbits 4-byte alignment");
    return from_hip(qm::quantize_values(x, x_dtype, rows, cols, hadamard_dim, make_signs(sign_bits, hadamard_dim), mode, seed, maskbits, dequant,
                                        reinterpret_cast<hipStream_t>(stream)),
                    "qm_pseudo_quantize_mxfp4");
}

int qm_requantize_transposed_mxfp4(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                   int val_dtype, int hadamard_dim, const uint32_t* sign_bits, int mode,
                                   const float* u, uint64_t seed, uint8_t* codes_out, uint8_t* scales_out,
                                   void* dequant, int in_layout, int out_layout, void* stream) {
    if (!valid_layout(in_layout) || !valid_layout(out_layout))
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: unknown layout %d / %d", in_layout, out_layout);
    if (!valid_dtype(val_dtype)) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: val_dtype %d", val_dtype);
    if (!valid_hd(hadamard_dim)) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: hadamard_dim %d not in {32,64,128}", hadamard_dim);
    if (!valid_mode(mode)) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: unknown mode %d", mode);
    if (R < 0 || C < 0 || C % 32 || R % hadamard_dim)
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: need C %% 32 == 0 and R %% hadamard_dim == 0 (R=%lld C=%lld hd=%d)", (long long)R, (long long)C, hadamard_dim);
    if (R == 0 || C == 0) return 0;
    if (!codes_in || !scales_in || !codes_out || !scales_out) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: null tensor");
    if (!aligned(codes_in, 16) || !aligned(codes_out, 4) || (dequant && !aligned(dequant, 16)) || (u && !aligned(u, 16)))
        return fail(QM_ERR_UNALIGNED, "qm_requantize_transposed_mxfp4: codes_in/dequant/u need 16-byte and codes_out 4-byte alignment");
    if ((in_layout == QM_LAYOUT_TILED || out_layout == QM_LAYOUT_TILED) &&
        (!qm::requantize_supports_tiled(R, C, hadamard_dim, mode, u) || !aligned(codes_out, 16) || !aligned(scales_out, 4)))
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4: tiled codes need hadamard_dim 32, R %% 128 == 0, C %% 128 == 0, "
                                    "no explicit uniforms, 16-byte aligned codes_out (R=%lld C=%lld)", (long long)R, (long long)C);
    return from_hip(qm::requantize_transposed_mxfp4(codes_in, scales_in, R, C, post, val_dtype, hadamard_dim,
                                                    make_signs(sign_bits, hadamard_dim), mode, u, seed, codes_out,
                                                    scales_out, dequant, in_layout, out_layout,
                                                    reinterpret_cast<hipStream_t>(stream)),
                    "qm_requantize_transposed_mxfp4");
}

int qm_quantize_mxfp4_dense(const void* x, int x_dtype, int64_t rows, int64_t cols, const float* matrix, int mode,
                            int transposed_in, uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant,
                            int codes_layout, void* stream) {
    if (!valid_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: unknown codes_layout %d", codes_layout);
    if (!valid_dtype(x_dtype)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: x_dtype %d is not QM_BF16/QM_F32", x_dtype);
    if (!valid_mode(mode)) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: unknown mode %d", mode);
    if (rows < 0 || cols < 0 || cols % 32)
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: cols %lld not a multiple of 32", (long long)cols);
    if (rows == 0 || cols == 0) return 0;
    if (!x || !codes || !scales || !matrix) return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: x, matrix, codes and scales must be non-null");
    if (!aligned(x, 16) || !aligned(codes, 16) || !aligned(matrix, 4) || !aligned(maskbits, 4) || (dequant && !aligned(dequant, 16)))
        return fail(QM_ERR_UNALIGNED, "qm_quantize_mxfp4_dense: x/codes/dequant need 16-byte, matrix and maskbits 4-byte alignment");
    if (transposed_in && (maskbits || cols % 128 || rows % 8 || !aligned(scales, 4)))
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: transposed input needs cols %% 128 == 0, rows %% 8 == 0, no clip mask, "
                                    "4-byte aligned scales (rows=%lld cols=%lld)", (long long)rows, (long long)cols);
    if (codes_layout == QM_LAYOUT_TILED && (rows % 16 || cols % 128))
        return fail(QM_ERR_INVALID, "qm_quantize_mxfp4_dense: tiled codes need rows %% 16 == 0 and cols %% 128 == 0 (rows=%lld cols=%lld)",
                    (long long)rows, (long long)cols);
    return from_hip(qm::quantize_mxfp4_dense(x, x_dtype, rows, cols, matrix, mode, transposed_in != 0, seed, codes, scales, maskbits,
                                             dequant, codes_layout, reinterpret_cast<hipStream_t>(stream)),
                    "qm_quantize_mxfp4_dense");
}

int qm_requantize_transposed_mxfp4_dense(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                         int val_dtype, const float* matrix, int mode, uint64_t seed, uint8_t* codes_out,
                                         uint8_t* scales_out, void* dequant, int in_layout, int out_layout, void* stream) {
    if (!valid_layout(in_layout) || !valid_layout(out_layout))
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: unknown layout %d / %d", in_layout, out_layout);
    if (!valid_dtype(val_dtype)) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: val_dtype %d", val_dtype);
    if (!valid_mode(mode)) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: unknown mode %d", mode);
    if (R < 0 || C < 0 || C % 32 || R % 128)
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: need C %% 32 == 0 and R %% 128 == 0 (R=%lld C=%lld)", (long long)R, (long long)C);
    if (R == 0 || C == 0) return 0;
    if (!codes_in || !scales_in || !codes_out || !scales_out || !matrix) return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: null tensor");
    if (!aligned(codes_in, 16) || !aligned(codes_out, 16) || !aligned(scales_out, 4) || !aligned(matrix, 4) || (dequant && !aligned(dequant, 16)))
        return fail(QM_ERR_UNALIGNED, "qm_requantize_transposed_mxfp4_dense: codes and dequant need 16-byte, scales_out and matrix 4-byte alignment");
    if ((in_layout == QM_LAYOUT_TILED || out_layout == QM_LAYOUT_TILED) && C % 128)
        return fail(QM_ERR_INVALID, "qm_requantize_transposed_mxfp4_dense: tiled codes need C %% 128 == 0 (C=%lld)", (long long)C);
    return from_hip(qm::requantize_transposed_mxfp4_dense(codes_in, scales_in, R, C, post, val_dtype, matrix, mode, seed, codes_out,
                                                          scales_out, dequant, in_layout, out_layout,
                                                          reinterpret_cast<hipStream_t>(stream)),
                    "qm_requantize_transposed_mxfp4_dense");
}

int qm_gemm_mxfp4_tn(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                     int64_t M, int64_t N, int64_t K, float alpha, void* c, int c_dtype, int a_layout, int b_layout,
                     void* workspace, size_t workspace_bytes, void* stream) {
    if (!valid_layout(a_layout) || !valid_layout(b_layout))
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn: unknown layout %d / %d", a_layout, b_layout);
    if (!valid_dtype(c_dtype)) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn: c_dtype %d", c_dtype);
    if (M < 0 || N < 0 || K < 0 || K % 32) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn: need K %% 32 == 0 (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    if (M == 0 || N == 0) return 0;
    if (!c || (K > 0 && (!a_codes || !a_scales || !b_codes || !b_scales))) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn: null tensor");
    // the 256 x 256 tile kernels store c in 16-byte pieces; the generic kernel (any M, N) stores single elements
    const uintptr_t c_align = qm::gemm_supports_tiled(M, N, K) ? 16 : 4;
    if (!aligned(a_codes, 16) || !aligned(b_codes, 16) || !aligned(a_scales, 4) || !aligned(b_scales, 4) || !aligned(c, c_align))
        return fail(QM_ERR_UNALIGNED, "qm_gemm_mxfp4_tn: codes need 16-byte, scales 4-byte alignment, c 16-byte (4-byte for shapes "
                                      "outside the tile kernels: M or N not a multiple of 64 or below 256, K %% 128 != 0)");
    if ((a_layout == QM_LAYOUT_TILED || b_layout == QM_LAYOUT_TILED) && !qm::gemm_supports_tiled(M, N, K))
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn: tiled operands need M, N multiples of 64 and >= 256, K %% 128 == 0 (M=%lld N=%lld K=%lld)",
                    (long long)M, (long long)N, (long long)K);
    return from_hip(qm::gemm_mxfp4_tn(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, c_dtype, a_layout, b_layout,
                                      workspace, workspace_bytes, reinterpret_cast<hipStream_t>(stream)),
                    "qm_gemm_mxfp4_tn");
}

int qm_diag_gemm_tile_phases(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                             int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_layout, int b_layout,
                             const uint8_t* maskbits, uint64_t* stamps, size_t stamps_bytes, void* stream) {
    if (!a_codes || !a_scales || !b_codes || !b_scales || !c || !stamps || !aligned(a_codes, 16) || !aligned(b_codes, 16) ||
        !aligned(c, 16) || !aligned(stamps, 8) || !aligned(maskbits, 4) || !valid_layout(a_layout) || !valid_layout(b_layout))
        return fail(QM_ERR_INVALID, "qm_diag_gemm_tile_phases: null, misaligned or ill-typed arguments");
    int grid = 0;
    const hipError_t e = qm::gemm_tile_phases(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_layout, b_layout, maskbits,
                                              reinterpret_cast<unsigned long long*>(stamps), stamps_bytes, &grid,
                                              reinterpret_cast<hipStream_t>(stream));
    if (e == hipErrorInvalidValue && grid == 0)
        return fail(QM_ERR_INVALID, "qm_diag_gemm_tile_phases: serves M, N multiples of 64 and >= 256, K %% 512 == 0, 16-byte aligned scales, "
                                    "and needs %d 64-bit values per workgroup in stamps", qm::gemm_phase_stamps_per_group());
    if (int rc = from_hip(e, "qm_diag_gemm_tile_phases")) return rc > 0 ? -rc : rc;
    return grid;
}

int64_t qm_diag_mfma_only(const uint8_t* operands, size_t operand_bytes, float* sink, size_t sink_bytes, int iters, void* stream) {
    const int blocks = qm::mfma_only_blocks();
    if (!operands || !sink || iters < 0 || operand_bytes < (size_t)blocks * 32768 || sink_bytes < (size_t)blocks * 1024 ||
        !aligned(operands, 16) || !aligned(sink, 4))
        return fail(QM_ERR_INVALID, "qm_diag_mfma_only: needs %zu bytes of operands (16-byte aligned) and %zu bytes of sink",
                    (size_t)blocks * 32768, (size_t)blocks * 1024);
    if (int rc = from_hip(qm::mfma_only(operands, sink, iters, reinterpret_cast<hipStream_t>(stream)), "qm_diag_mfma_only")) return -(int64_t)(rc > 0 ? rc : -rc);
    return (int64_t)blocks * 4 * (int64_t)iters * 16;
}

int qm_gemm_mxfp4_bf16_nn(const uint8_t* a_codes, const uint8_t* a_scales, const void* b, int64_t M, int64_t N, int64_t K,
                          float alpha, void* c, int c_dtype, void* stream) {
    if (!valid_dtype(c_dtype)) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_bf16_nn: c_dtype %d", c_dtype);
    if (M < 0 || N < 0 || K < 0) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_bf16_nn: negative extent");
    if (M == 0 || N == 0) return 0;
    if (!qm::gemm_fp4_bf16_nn_supported(M, N, K))
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_bf16_nn: need K a positive multiple of 64 and N a multiple of 8 (M=%lld N=%lld K=%lld)",
                    (long long)M, (long long)N, (long long)K);
    if (!a_codes || !a_scales || !b || !c) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_bf16_nn: null tensor");
    if (!aligned(a_codes, 16) || !aligned(a_scales, 2) || !aligned(b, 16) || !aligned(c, 16))
        return fail(QM_ERR_UNALIGNED, "qm_gemm_mxfp4_bf16_nn: a_codes, b and c need 16-byte, a_scales 2-byte alignment");
    return from_hip(qm::gemm_fp4_bf16_nn(a_codes, a_scales, b, M, N, K, alpha, c, c_dtype, reinterpret_cast<hipStream_t>(stream)),
                    "qm_gemm_mxfp4_bf16_nn");
}

size_t qm_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32) return 0;
    return qm::gemm_workspace_bytes(M, N, K);
}

}  // extern "C"

// ---- the product without any allocation: split-K partial sums live in a file-scope device array ---------------
namespace {
constexpr size_t kNoAllocScratchBytes = QM_GEMM_NOALLOC_SCRATCH_BYTES;
// One copy per GPU the library is loaded on, held until the process ends.  In host code this name is only a handle for
// hipGetSymbolAddress: the device address of each GPU's copy is looked up once per device and used from then on.
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// device address of the current device's scratch array (nullptr + error code on failure)
int scratch_of_current_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return from_hip(e, "qm_gemm_mxfp4_tn_noalloc: hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_noalloc: device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return from_hip(e == hipSuccess ? hipErrorInvalidSymbol : e, "qm_gemm_mxfp4_tn_noalloc: hipGetSymbolAddress");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace

extern "C" {

size_t qm_gemm_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

int qm_gemm_noalloc_prepare(void) {
    void* ws = nullptr;
    return scratch_of_current_device(&ws);
}

int qm_gemm_mxfp4_tn_noalloc(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                             int64_t M, int64_t N, int64_t K, float alpha, void* c, int c_dtype, int a_layout, int b_layout,
                             void* stream) {
    if (M < 0 || N < 0 || K < 0 || K % 32)
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_noalloc: need K %% 32 == 0 (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    if (M == 0 || N == 0) return 0;
    // refused: few tiles and a K so long that the ranges filling the CUs do not fit.  Every other product runs, in the cut that
    // qm_gemm_mxfp4_tn makes of it where that fits and whole where it does not (2176 x 8192 x 28672: two ranges, 136 MiB).
    const size_t need = qm::gemm_few_tiles_bytes(M, N, K);
    if (need > kNoAllocScratchBytes)
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_noalloc: this shape's split-K partial sums need %zu bytes, the built-in scratch "
                                    "holds %zu (M=%lld N=%lld K=%lld); use qm_gemm_mxfp4_tn with a caller-provided workspace",
                    need, kNoAllocScratchBytes, (long long)M, (long long)N, (long long)K);
    // resolved on every path, so that the first call on a device is the only one that can make the runtime load this
    // library's device image (qm_gemm_noalloc_prepare() does the same ahead of time)
    void* ws = nullptr;
    if (int rc = scratch_of_current_device(&ws)) return rc;
    return qm_gemm_mxfp4_tn(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, c_dtype, a_layout, b_layout, ws, kNoAllocScratchBytes, stream);
}

int qm_masked_hadamard_bwd(const void* g, int g_dtype, int64_t rows, int64_t cols, int hadamard_dim, int scale_dtype,
                           const uint32_t* sign_bits, const uint8_t* maskbits, void* out, int out_dtype, void* stream) {
    if (!valid_dtype(g_dtype) || !valid_dtype(out_dtype) || !valid_dtype(scale_dtype))
        return fail(QM_ERR_INVALID, "qm_masked_hadamard_bwd: dtypes must be QM_BF16/QM_F32");
    if (!valid_hd(hadamard_dim)) return fail(QM_ERR_INVALID, "qm_masked_hadamard_bwd: hadamard_dim %d not in {32,64,128}", hadamard_dim);
    if (rows < 0 || cols < 0 || cols % hadamard_dim)
        return fail(QM_ERR_INVALID, "qm_masked_hadamard_bwd: cols %lld not a multiple of hadamard_dim %d", (long long)cols, hadamard_dim);
    if (rows == 0 || cols == 0) return 0;
    if (!g || !out) return fail(QM_ERR_INVALID, "qm_masked_hadamard_bwd: null tensor");
    if (!aligned(g, 16) || !aligned(out, 16)) return fail(QM_ERR_UNALIGNED, "qm_masked_hadamard_bwd: g and out need 16-byte alignment");
    return from_hip(qm::masked_hadamard_bwd(g, g_dtype, rows, cols, hadamard_dim, scale_dtype,
                                            make_signs(sign_bits, hadamard_dim), maskbits, out, out_dtype, false,
                                            reinterpret_cast<hipStream_t>(stream)),
                    "qm_masked_hadamard_bwd");
}

int qm_gemm_fuses_rotation(const uint8_t* a_scales, const uint8_t* b_scales, int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32) return 0;
    // not where the persistent kernel's few tiles leave CUs idle and K ranges would fill them; whether smaller tiles, or a cut
    // on them, would be cheaper is the caller's business (qm_linear_backward weighs that by itself)
    return qm::gemm_few_tiles_bytes(M, N, K) == 0 && qm::gemm_persistent_rotates(a_scales, b_scales, M, N, K) ? 1 : 0;
}

int qm_gemm_mxfp4_tn_rotated(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                             int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_layout, int b_layout,
                             const uint8_t* maskbits, const uint32_t* sign_bits, int scale_dtype, void* stream) {
    if (!valid_layout(a_layout) || !valid_layout(b_layout))
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_rotated: unknown layout %d / %d", a_layout, b_layout);
    if (!valid_dtype(scale_dtype)) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_rotated: scale_dtype %d", scale_dtype);
    if (M < 0 || N < 0 || K < 0) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_rotated: negative extent");
    if (M == 0 || N == 0) return 0;
    if (!c || !a_codes || !a_scales || !b_codes || !b_scales || !maskbits) return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_rotated: null tensor");
    if (!qm_gemm_fuses_rotation(a_scales, b_scales, M, N, K))
        return fail(QM_ERR_INVALID, "qm_gemm_mxfp4_tn_rotated: shape M=%lld N=%lld K=%lld is not served with the rotation fused "
                                    "(see qm_gemm_fuses_rotation); call qm_gemm_mxfp4_tn and qm_masked_hadamard_bwd",
                    (long long)M, (long long)N, (long long)K);
    if (!aligned(a_codes, 16) || !aligned(b_codes, 16) || !aligned(a_scales, 4) || !aligned(b_scales, 4) || !aligned(c, 16) || !aligned(maskbits, 4))
        return fail(QM_ERR_UNALIGNED, "qm_gemm_mxfp4_tn_rotated: codes and c need 16-byte, scales and mask bits 4-byte alignment");
    qm::TileProduct p = qm::make_product(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_layout, b_layout);
    p.mask = maskbits;
    p.signs = make_signs(sign_bits, 32);
    p.rot_c = qm::hadamard_scale(32, scale_dtype);
    return from_hip(qm::gemm_persistent_rotated(p, reinterpret_cast<hipStream_t>(stream)), "qm_gemm_mxfp4_tn_rotated");
}

int qm_dequantize_mxfp4(const uint8_t* codes, const uint8_t* scales, int64_t R, int64_t C, float post, void* out,
                        int out_dtype, void* stream) {
    if (!valid_dtype(out_dtype)) return fail(QM_ERR_INVALID, "qm_dequantize_mxfp4: out_dtype %d", out_dtype);
    if (R < 0 || C < 0 || C % 32) return fail(QM_ERR_INVALID, "qm_dequantize_mxfp4: need C %% 32 == 0 (R=%lld C=%lld)", (long long)R, (long long)C);
    if (R == 0 || C == 0) return 0;
    if (!codes || !scales || !out) return fail(QM_ERR_INVALID, "qm_dequantize_mxfp4: null tensor");
    if (!aligned(codes, 4) || !aligned(out, 16)) return fail(QM_ERR_UNALIGNED, "qm_dequantize_mxfp4: codes need 4-byte and out 16-byte alignment");
    return from_hip(qm::dequantize_mxfp4(codes, scales, R, C, post, out, out_dtype, reinterpret_cast<hipStream_t>(stream)),
                    "qm_dequantize_mxfp4");
}


// ---- whole-layer entry points: one call issues every launch of the forward / backward pass -------------------

namespace {
size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }
size_t esize(int dtype) { return dtype == QM_BF16 ? 2 : 4; }

// one packed operand: codes, scales, mask bits, each region 256-byte aligned.  The code and scale regions hold the tiled
// layout with its rows padded to 16 and its columns to 128; a row-major operand occupies the front of each region.
size_t code_bytes(int64_t rows, int64_t cols) { return up256((size_t)qm::padded_rows(rows) * qm::padded_cols(cols) / 2); }
size_t scale_bytes(int64_t rows, int64_t cols) { return up256((size_t)qm::padded_rows(rows) * qm::padded_cols(cols) / 32); }
struct PackedLayout {
    size_t c, s, m, total;
};
PackedLayout packed_layout(int64_t rows, int64_t cols) {
    PackedLayout l;
    size_t o = 0;
    l.c = o; o += code_bytes(rows, cols);
    l.s = o; o += scale_bytes(rows, cols);
    l.m = o; o += up256((size_t)rows * cols / 8);
    l.total = o;
    return l;
}
struct WorkLayout {
    size_t ec, es, wtc, wts, gxq, etc, ets, xtc, xts, gwq, gemm_ws, gemm_ws_bytes, total;
};
WorkLayout work_layout(int64_t T, int64_t I, int64_t O, int mid_dtype) {
    WorkLayout l;
    size_t o = 0;
    l.ec = o; o += code_bytes(T, O);
    l.es = o; o += scale_bytes(T, O);
    l.wtc = o; o += code_bytes(I, O);
    l.wts = o; o += scale_bytes(I, O);
    l.gxq = o; o += up256((size_t)T * I * esize(mid_dtype));
    l.etc = o; o += code_bytes(O, T);
    l.ets = o; o += scale_bytes(O, T);
    l.xtc = o; o += code_bytes(I, T);
    l.xts = o; o += scale_bytes(I, T);
    l.gwq = o; o += up256((size_t)O * I * esize(mid_dtype));
    // split-K scratch, shared by the two products (they run one after the other), for either layout's contraction length
    const int64_t Op = qm::padded_cols(O), Tp = qm::padded_cols(T);
    const size_t need[] = {qm::gemm_workspace_bytes(T, I, O), qm::gemm_workspace_bytes(O, I, T), qm::gemm_workspace_bytes(T, I, Op),
                           qm::gemm_workspace_bytes(O, I, Tp)};
    l.gemm_ws_bytes = 0;
    for (size_t n : need) l.gemm_ws_bytes = n > l.gemm_ws_bytes ? n : l.gemm_ws_bytes;
    l.gemm_ws = o; o += up256(l.gemm_ws_bytes);
    l.total = o;
    return l;
}
// the error-only scheme: Q(e), Q(e^T), the packed operands as eight-bit ones, a product before its rotation (one at a time)
struct ErrorLayout {
    size_t ec, es, etc, ets, wv, ws, wl, wf, xv, xs, xl, xf, plain, gemm_ws, gemm_ws_bytes, total;
};
ErrorLayout error_layout(int64_t T, int64_t I, int64_t O) {
    ErrorLayout l;
    size_t o = 0;
    const auto take = [&](size_t& at, size_t n) { at = o; o += up256(n); };
    const int64_t Tp = qm::padded_cols(T), Op = qm::padded_cols(O);
    take(l.ec, code_bytes(T, O)); take(l.es, scale_bytes(T, O));
    take(l.etc, code_bytes(O, T)); take(l.ets, scale_bytes(O, T));
    take(l.wv, (size_t)I * Op); take(l.ws, (size_t)I * Op / 32); take(l.wl, (size_t)((I + 127) / 128) * (Op / 128)); take(l.wf, (size_t)qm::six_bit_flags(O, I));
    take(l.xv, (size_t)I * Tp); take(l.xs, (size_t)I * Tp / 32); take(l.xl, (size_t)((I + 127) / 128) * (Tp / 128)); take(l.xf, (size_t)qm::six_bit_flags(T, I));
    take(l.plain, (size_t)(T > O ? T : O) * I * 2);
    const size_t need_x = qm::gemm_e5m2_workspace_bytes(T, I, Op), need_w = qm::gemm_e5m2_workspace_bytes(O, I, Tp);
    l.gemm_ws_bytes = need_x > need_w ? need_x : need_w;
    take(l.gemm_ws, l.gemm_ws_bytes);
    l.total = o;
    return l;
}
bool tiled_layout(int codes_layout) { return codes_layout != QM_LAYOUT_ROWMAJOR; }
// the layout the kernels of a single operation are told
int kernel_layout(int codes_layout) { return tiled_layout(codes_layout) ? QM_LAYOUT_TILED : QM_LAYOUT_ROWMAJOR; }
// a device seed base is read by the kernels of the tiled layer path, and offered for the extents the interface promises it for
bool seed_base_served(int codes_layout, int64_t T, int64_t I, int64_t O, int hd_a, int hd_b, int hd_c) {
    return tiled_layout(codes_layout) && hd_a == 32 && hd_b == 32 && hd_c == 32 && T % 128 == 0 && I % 128 == 0 &&
           O % 128 == 0;
}
extern "C++" {
// Both products of the error-only scheme on whole 256 x 256 tiles: one grid for them.  us per step, two launches against one: 4096^3 174 -> 169.6,
// 2048 x 8192 x 4096 218.8 -> 215; what is gained is one start and one last wave of tiles.
bool wide_pair(const qm::TileProduct& x, const qm::ProductChoice& cx, const qm::TileProduct& w, const qm::ProductChoice& cw) {
    const auto whole = [](const qm::ProductChoice& c) { return c.path == qm::ProductChoice::TILE && c.kind == qm::WIDE_256x256 && c.splits == 1 && c.rotates; };
    return whole(cx) && whole(cw) && qm::gemm_wide_pair_serves(x, w);
}
// The masked inverse rotation of the forward quantizer in a gradient product, into dst
qm::TileProduct with_rotation(qm::TileProduct p, void* dst, int hd, const uint8_t* mask, const uint32_t* signs, int scale_dtype) {
    p.c = dst;
    p.mask = mask;
    p.hd = hd;
    p.signs = make_signs(signs, hd);
    p.rot_c = qm::hadamard_scale(hd, scale_dtype);
    return p;
}
// A gradient product of the backward pass and the kernel that serves it by itself: with that rotation where that kernel applies it,
// otherwise without (into plain.c)
struct GradProduct {
    qm::TileProduct p;
    qm::ProductChoice choice;
    int out_dtype;
};
GradProduct plan_gradient(const qm::TileProduct& plain, void* final_dst, bool want_rotation, int hd, int mid_dtype, int final_dtype, const uint8_t* mask,
                          const uint32_t* signs, int scale_dtype, void* ws, size_t ws_bytes) {
    if (want_rotation && final_dst && aligned(final_dst, 16) && valid_dtype(scale_dtype) && valid_hd(hd) && plain.N % hd == 0) {
        const qm::TileProduct r = with_rotation(plain, final_dst, hd, mask, signs, scale_dtype);
        const qm::ProductChoice c = qm::choose_product(r, mid_dtype, final_dtype, ws, ws_bytes);
        if (c.rotates) return {r, c, final_dtype};
    }
    return {plain, qm::choose_product(plain, mid_dtype, mid_dtype, ws, ws_bytes), mid_dtype};
}
// How the two gradient products of a layer on tiled operands share a launch, of bf16 results.  One launch adds a whole contraction up
// in one chain, launched apart a product may be cut into K ranges, which rounds differently: so a layer's gradients must not change with
// the form of its call (gx left rotated for the fused kernel behind it, an fp32 or a bf16 weight).  It is decided from what all forms have in
// common, the extents, the Hadamard blocks and the kind of column signs, with the figures of the form that rotates both into bf16; the
// weight gradient's type counts where neither product would be cut, whose sums are then the same either way.  With gx left rotated the estimate is
// up to 0.07 nearer to two launches', and 40 such steps that share a launch are 0.96 to 1.09 times as fast for it, all but two 0.99 and more.
qm::PairChoice choose_gradient_pair(int64_t T, int64_t I, int64_t O, int hd_x, int hd_w, const uint32_t* signs_x, const uint32_t* signs_w, int gw_dtype) {
    uint8_t* at = reinterpret_cast<uint8_t*>((uintptr_t)256);   // nothing is read: stand-ins with the alignment that a layer's tensors have
    const size_t ws_bytes = work_layout(T, I, O, QM_BF16).gemm_ws_bytes;
    const auto product = [&](int64_t M, int64_t K, int hd, const uint32_t* signs) {
        return with_rotation(qm::make_product(at, at, at, at, M, I, qm::padded_cols(K), 1.0f, at, QM_LAYOUT_TILED, QM_LAYOUT_TILED), at, hd, at, signs, QM_BF16);
    };
    const auto choose = [&](const qm::TileProduct& p, int out) { return qm::choose_product(p, QM_BF16, out, ws_bytes ? at : nullptr, ws_bytes); };
    const qm::TileProduct x = product(T, O, hd_x, signs_x), w = product(O, T, hd_w, signs_w);
    const qm::ProductChoice cx = choose(x, QM_BF16), cw = choose(w, QM_BF16);
    if (gw_dtype != QM_BF16 && cx.splits == 1 && cw.splits == 1) return qm::choose_pair(x, cx, QM_BF16, w, choose(w, gw_dtype), gw_dtype);
    return qm::choose_pair(x, cx, QM_BF16, w, cw, QM_BF16);
}
// Remembered per thread (a small layer's training step is bound by its host): up to 64 layers, 4 KB.  Of the signs only whether they repeat
// every 32 counts.
struct PairPlan {
    int64_t M = -1, N = 0, K = 0;
    int flags = -1;
    qm::PairChoice choice{qm::PairChoice::SEPARATE, 0, 0};
};
qm::PairChoice gradient_pair(int64_t T, int64_t I, int64_t O, int hd_x, int hd_w, const uint32_t* signs_x, const uint32_t* signs_w, int gw_dtype) {
    static thread_local qm::ShapeTable<PairPlan, 4> table;
    const auto form = [](int hd, const uint32_t* signs) {
        bool repeat = true;
        for (int j = 1; signs && j < hd / 32; ++j) repeat = repeat && signs[j] == signs[0];
        return hd / 32 * 2 + (repeat ? 1 : 0);
    };
    const int flags = (form(hd_x, signs_x) * 16 + form(hd_w, signs_w)) * 2 + (gw_dtype == QM_BF16 ? 0 : 1);
    return table.find(T, I, O, flags, [&] { return PairPlan{T, I, O, flags, choose_gradient_pair(T, I, O, hd_x, hd_w, signs_x, signs_w, gw_dtype)}; }).choice;
}
}
}  // namespace

size_t qm_packed_operand_bytes(int64_t rows, int64_t cols) {
    if (rows < 0 || cols < 0 || cols % 32) return 0;
    return packed_layout(rows, cols).total;
}

int qm_packed_operand_offsets(int64_t rows, int64_t cols, size_t* offsets) {
    if (rows < 0 || cols < 0 || cols % 32 || !offsets)
        return fail(QM_ERR_INVALID, "qm_packed_operand_offsets: need cols %% 32 == 0 and a non-null array (rows=%lld cols=%lld)",
                    (long long)rows, (long long)cols);
    const PackedLayout l = packed_layout(rows, cols);
    offsets[0] = l.c; offsets[1] = l.s; offsets[2] = l.m;
    return 0;
}

size_t qm_linear_backward_workspace_bytes(int64_t T, int64_t I, int64_t O, int mid_dtype) {
    if (T < 0 || I < 0 || O < 0 || I % 32 || O % 32 || T % 32 || !valid_dtype(mid_dtype)) return 0;
    return work_layout(T, I, O, mid_dtype).total;
}

int qm_linear_backward_in_one_launch(int64_t T, int64_t I, int64_t O, int hd_x, int hd_w, int gw_dtype, int rotated_flags) {
    if (T <= 0 || I <= 0 || O <= 0 || I % 32 || O % 32 || T % 32 || !valid_hd(hd_x) || !valid_hd(hd_w) || !valid_dtype(gw_dtype)) return 0;
    if (T >= (1ll << 31) || I >= (1ll << 31) || O >= (1ll << 31)) return 0;
    if (I % hd_x || I % hd_w) return 0;
    const qm::PairChoice pair = gradient_pair(T, I, O, hd_x, hd_w, nullptr, nullptr, gw_dtype);
    uint8_t* at = reinterpret_cast<uint8_t*>((uintptr_t)256);   // nothing is read
    const auto product = [&](int64_t M, int64_t K, bool rotate, int hd) {
        const qm::TileProduct p = qm::make_product(at, at, at, at, M, I, qm::padded_cols(K), 1.0f, at, QM_LAYOUT_TILED, QM_LAYOUT_TILED);
        return rotate ? with_rotation(p, at, hd, at, nullptr, QM_BF16) : p;
    };
    const qm::TileProduct x = product(T, O, !(rotated_flags & QM_GX_ROTATED), hd_x), w = product(O, T, !(rotated_flags & QM_GW_ROTATED), hd_w);
    return qm::pair_serves(pair, x, QM_BF16, w, gw_dtype) ? (int)pair.path : 0;
}

int qm_linear_forward(const void* x, int x_dtype, const void* w, int w_dtype, int64_t T, int64_t I, int64_t O, int hd_x,
                      const uint32_t* signs_x, int hd_w, const uint32_t* signs_w, void* packed_x, size_t packed_x_bytes,
                      void* packed_w, size_t packed_w_bytes, int packed_flags, void* y, int y_dtype, int codes_layout,
                      void* stream) {
    if (T < 0 || I < 0 || O < 0) return fail(QM_ERR_INVALID, "qm_linear_forward: negative extent");
    if (!valid_layer_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_linear_forward: unknown codes_layout %d", codes_layout);
    if (T == 0 || O == 0 || I == 0) return 0;
    if (I % 32) return fail(QM_ERR_INVALID, "qm_linear_forward: in_features %lld not a multiple of 32", (long long)I);
    const PackedLayout lx = packed_layout(T, I), lw = packed_layout(O, I);
    if (!packed_x || packed_x_bytes < lx.total || !aligned(packed_x, 256) || !packed_w || packed_w_bytes < lw.total ||
        !aligned(packed_w, 256))
        return fail(QM_ERR_INVALID, "qm_linear_forward: packed operand buffers need %zu and %zu bytes, 256-byte aligned", lx.total,
                    lw.total);
    uint8_t* px = static_cast<uint8_t*>(packed_x);
    uint8_t* pw = static_cast<uint8_t*>(packed_w);
    if (packed_flags & ~(QM_W_IS_PACKED | QM_X_IS_PACKED)) return fail(QM_ERR_INVALID, "qm_linear_forward: unknown packed_flags %d", packed_flags);
    const bool w_is_packed = packed_flags & QM_W_IS_PACKED, x_is_packed = packed_flags & QM_X_IS_PACKED;
    if (!y || !aligned(y, 4)) return fail(QM_ERR_INVALID, "qm_linear_forward: y must be non-null and 4-byte aligned");
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    int rc = 0;
    int64_t K = I;
    if (tiled_layout(codes_layout)) {
        if (O % 8 || !aligned(y, 16)) return fail(QM_ERR_INVALID, "qm_linear_forward: tiled codes need out_features %% 8 == 0 and a 16-byte aligned y");
        if (codes_layout == QM_LAYOUT_TILED && (T % 16 || O % 16 || I % 128))
            return fail(QM_ERR_INVALID, "qm_linear_forward: tiled codes need tokens and out_features %% 16 == 0 and in_features %% 128 == 0 (QM_LAYOUT_PADDED takes any)");
        const qm::RowmajorArgs ax{x, x_dtype, T, I, make_signs(signs_x, hd_x), px + lx.c, px + lx.s, px + lx.m};
        const qm::RowmajorArgs aw{w, w_dtype, O, I, make_signs(signs_w, hd_w), pw + lw.c, pw + lw.s, pw + lw.m};
        const auto bad = [&](const qm::RowmajorArgs& a, int hd) {
            return !a.x || !aligned(a.x, 16) || !valid_dtype(a.dtype) || !valid_hd(hd) || a.cols % hd || a.rows >= (1ll << 31) - 16;
        };
        if ((!x_is_packed && bad(ax, hd_x)) || (!w_is_packed && bad(aw, hd_w)))
            return fail(QM_ERR_INVALID, "qm_linear_forward: x and w must be non-null, 16-byte aligned, of a valid dtype, in_features a multiple of the Hadamard block");
        if (!x_is_packed && !w_is_packed && hd_x == hd_w) {
            rc = from_hip(qm::quantize_layer_forward(ax, &aw, hd_x, hs), "qm_linear_forward");   // both forward quantizers in one grid
        } else {
            if (!x_is_packed) rc = from_hip(qm::quantize_layer_forward(ax, nullptr, hd_x, hs), "qm_linear_forward");
            if (!rc && !w_is_packed) rc = from_hip(qm::quantize_layer_forward(aw, nullptr, hd_w, hs), "qm_linear_forward");
        }
        K = qm::padded_cols(I);
    } else {
        if (!x_is_packed)
            rc = qm_quantize_mxfp4(x, x_dtype, T, I, hd_x, signs_x, QM_QUEST_RTN, 0, nullptr, 0, px + lx.c, px + lx.s, px + lx.m,
                                   nullptr, codes_layout, stream);
        if (!rc && !w_is_packed)
            rc = qm_quantize_mxfp4(w, w_dtype, O, I, hd_w, signs_w, QM_QUEST_RTN, 0, nullptr, 0, pw + lw.c, pw + lw.s, pw + lw.m,
                                   nullptr, codes_layout, stream);
    }
    if (rc) return rc;
    if (!valid_dtype(y_dtype)) return fail(QM_ERR_INVALID, "qm_linear_forward: y_dtype %d", y_dtype);
    if (T <= 64 && O < (1ll << 30) && K < (1ll << 30) && tiled_layout(codes_layout)) {
        const qm::TileProduct p = qm::make_product(px + lx.c, px + lx.s, pw + lw.c, pw + lw.s, T, O, K, 1.0f, y, QM_LAYOUT_TILED, QM_LAYOUT_TILED);
        if (qm::gemm_rows_serves(p)) return from_hip(qm::gemm_rows(p, y_dtype, hs), "qm_linear_forward");
    }
    return from_hip(qm::gemm_mxfp4_tn(px + lx.c, px + lx.s, pw + lw.c, pw + lw.s, T, O, K, 1.0f, y, y_dtype, kernel_layout(codes_layout), kernel_layout(codes_layout), nullptr, 0, hs),
                    "qm_linear_forward");
}

namespace {
// a product of an evaluated model on packed operands in the padded layout, of the extents that those kernels take
bool after_product(int64_t T, int64_t I, int64_t N, const uint8_t* px, const uint8_t* pw, void* c, qm::TileProduct* p) {
    // up to 64 tokens the layers add their terms in another order (gemm_rows.hip)
    if (T <= 64 || I <= 0 || N <= 0 || I % 32 || N % 8 || T >= (1 << 30) || I >= (1 << 23) || N >= (1 << 30)) return false;
    const PackedLayout lx = packed_layout(T, I), lw = packed_layout(N, I);
    *p = qm::make_product(px + lx.c, px + lx.s, pw + lw.c, pw + lw.s, T, N, qm::padded_cols(I), 1.0f, c, QM_LAYOUT_TILED, QM_LAYOUT_TILED);
    return qm::gemm_tile_after_serves(*p);
}
uint8_t* stand_in() { return reinterpret_cast<uint8_t*>((uintptr_t)256); }   // for questions in which nothing is read
}  // namespace

// Against the product on its fastest kernel and the producer behind it: 0.6 us a tile and CU for the quantizer in the epilogue; the
// producer 3.5 us (launch, quantizing) and its bytes (4.66 an element: two bf16 halves, codes, scales, mask) at 4.8 TB/s.  Timed as captured launches of
// the norm, both products and what is between them, 65 to 32768 tokens of widths 640 x 1728 to 4096 x 11008: never slower where it says yes, the gain up
// to 34 us more than estimated.  us in one and in two: 65 x 640 x 1728 16.2 / 17.7, 4096 tokens 31.7 / 39.8, 32768 153 / 206; 4096 x 1536 x 4096 75 / 85,
// 32768 511 / 552; 300 x 4096 x 11008 59 / 74.  Where it says no (1024 x 2560 x 6912, 8192 x 4096 x 11008) one launch is 0 to 15 % faster still.
int qm_linear_swiglu_serves(int64_t T, int64_t I, int64_t hidden) {
    qm::TileProduct p;
    if (hidden <= 0 || hidden % 32 || hidden >= (1 << 23) || !after_product(T, I, 2 * hidden, stand_in(), stand_in(), stand_in(), &p)) return 0;
    return qm::product_after_pays(p, 0.6, 3.5 + (double)T * hidden * 4.66 / 4.8e6) ? 1 : 0;
}

int qm_linear_swiglu_quantize(const void* packed_x, size_t packed_x_bytes, const void* packed_w, size_t packed_w_bytes, int64_t T, int64_t I,
                              int64_t hidden, const uint32_t* sign_bits, void* packed, size_t packed_bytes, void* stream) {
    qm::TileProduct p;
    uint8_t* out = static_cast<uint8_t*>(packed);
    if (hidden <= 0 || hidden % 32 || hidden >= (1 << 23) ||
        !after_product(T, I, 2 * hidden, static_cast<const uint8_t*>(packed_x), static_cast<const uint8_t*>(packed_w), out, &p))
        return fail(QM_ERR_INVALID, "qm_linear_swiglu_quantize: [%lld, %lld] x [2 x %lld] is not served (see qm_linear_swiglu_serves)", (long long)T, (long long)I,
                    (long long)hidden);
    const PackedLayout l = packed_layout(T, hidden);
    if (!packed_x || packed_x_bytes < packed_layout(T, I).total || !aligned(packed_x, 256) || !packed_w || packed_w_bytes < packed_layout(2 * hidden, I).total ||
        !aligned(packed_w, 256) || !packed || packed_bytes < l.total || !aligned(packed, 256))
        return fail(QM_ERR_INVALID, "qm_linear_swiglu_quantize: packed operand buffers too small, null or not 256-byte aligned");
    qm::TileAfter after{};
    p.c = out + l.c;
    after.scales = out + l.s;
    after.sign_word = sign_bits ? sign_bits[0] : 0u;
    after.c = qm::hadamard_scale(32, QM_BF16);
    return from_hip(qm::gemm_tile_swiglu(p, after, reinterpret_cast<hipStream_t>(stream)), "qm_linear_swiglu_quantize");
}

// The same with the rotary split: 0.3 us a tile and CU; the launch of its own 1 us, where it follows its product at once, and 12 bytes an
// element at 5.0 TB/s.  Of 85 sizes of 65 to 32768 tokens and widths 640 to 4096 one is on the other side than the estimate says (256 x 1536, by 0.1
// us).  us in one launch and in two: 65 x 1536 13.8 / 12.3, 128 x 4096 25.8 / 23.6, 200 x 1280 13.9 / 13.1; 300 x 2048 15.8 / 16.6, 512 x 1536 15.1 / 17.4,
// 4096 x 640 19.7 / 26.6, 32768 x 1536 310 / 340.
int qm_linear_rope_serves(int64_t T, int64_t I, int64_t n_embd, int head_dim) {
    qm::TileProduct p;
    if (n_embd <= 0 || n_embd > (1 << 24) || head_dim <= 0 || head_dim % 8 || n_embd % head_dim ||
        !after_product(T, I, 3 * n_embd, stand_in(), stand_in(), stand_in(), &p))
        return 0;
    return qm::product_after_pays(p, 0.3, 1.0 + (double)T * n_embd * 12.0 / 5.0e6) ? 1 : 0;
}

int qm_linear_rope(const void* packed_x, size_t packed_x_bytes, const void* packed_w, size_t packed_w_bytes, int64_t T, int64_t I, int64_t n_embd,
                   int head_dim, int64_t seq_len, const float* table, void* q, void* k, void* v, void* stream) {
    qm::TileProduct p;
    if (n_embd <= 0 || n_embd > (1 << 24) || head_dim <= 0 || head_dim % 8 || n_embd % head_dim || seq_len <= 0 || seq_len > (1 << 30) ||
        !after_product(T, I, 3 * n_embd, static_cast<const uint8_t*>(packed_x), static_cast<const uint8_t*>(packed_w), q, &p))
        return fail(QM_ERR_INVALID, "qm_linear_rope: [%lld, %lld] x [3 x %lld], head_dim %d is not served (see qm_linear_rope_serves)", (long long)T, (long long)I,
                    (long long)n_embd, head_dim);
    if (!packed_x || packed_x_bytes < packed_layout(T, I).total || !aligned(packed_x, 256) || !packed_w || packed_w_bytes < packed_layout(3 * n_embd, I).total ||
        !aligned(packed_w, 256) || !table || !q || !k || !v || !aligned(table, 16) || !aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16))
        return fail(QM_ERR_INVALID, "qm_linear_rope: packed operand buffers too small, null or not 256-byte aligned, or tensors not 16-byte aligned");
    qm::TileAfter after{};
    after.q = q; after.k = k; after.v = v;
    after.table = table;
    after.seq_len = (int)seq_len; after.width = (int)n_embd; after.head_dim = head_dim;
    return from_hip(qm::gemm_tile_rope(p, after, reinterpret_cast<hipStream_t>(stream)), "qm_linear_rope");
}

int qm_linear_decode_serves(int64_t T, int64_t I, int64_t O) { return qm::linear_decode_serves(T, I, O) ? 1 : 0; }

int qm_linear_decode(const void* x, int x_dtype, int64_t T, int64_t I, int64_t O, const uint32_t* signs_x, const void* packed_w,
                     size_t packed_w_bytes, void* y, int y_dtype, void* stream) {
    if (!valid_dtype(x_dtype) || !valid_dtype(y_dtype)) return fail(QM_ERR_INVALID, "qm_linear_decode: dtypes must be QM_BF16/QM_F32");
    if (!qm::linear_decode_serves(T, I, O))
        return fail(QM_ERR_INVALID, "qm_linear_decode: [%lld, %lld] x [%lld] is not served (see qm_linear_decode_serves)", (long long)T, (long long)I, (long long)O);
    const PackedLayout lw = packed_layout(O, I);
    if (!x || !aligned(x, 16) || !y || !aligned(y, 16)) return fail(QM_ERR_INVALID, "qm_linear_decode: x and y must be non-null and 16-byte aligned");
    if (!packed_w || packed_w_bytes < lw.total || !aligned(packed_w, 256))
        return fail(QM_ERR_INVALID, "qm_linear_decode: the packed weight needs %zu bytes, 256-byte aligned", lw.total);
    const uint8_t* pw = static_cast<const uint8_t*>(packed_w);
    return from_hip(qm::linear_decode(x, x_dtype, T, I, O, signs_x ? signs_x[0] : 0u, pw + lw.c, pw + lw.s, y, y_dtype,
                                      reinterpret_cast<hipStream_t>(stream)),
                    "qm_linear_decode");
}

size_t qm_linear_backward_error_workspace_bytes(int64_t T, int64_t I, int64_t O) {
    if (T < 0 || I < 0 || O < 0 || I % 32 || O % 32 || T % 32) return 0;
    return error_layout(T, I, O).total;
}

int qm_linear_backward_error_in_one_launch(int64_t T, int64_t I, int64_t O, int hd, int gw_dtype) {
    if (T <= 0 || I <= 0 || O <= 0 || I % 32 || O % 32 || T % 32 || I >= (1 << 23) || O >= (1 << 23) || T >= (1 << 23) || !valid_hd(hd) || I % hd || !valid_dtype(gw_dtype)) return 0;
    uint8_t* at = reinterpret_cast<uint8_t*>((uintptr_t)256);   // nothing is read
    const size_t ws = error_layout(T, I, O).gemm_ws_bytes;
    const auto product = [&](int64_t M, int64_t R) {
        qm::TileProduct p = qm::make_product(at, at, at, at, M, I, qm::padded_cols(R), 1.0f, at, QM_LAYOUT_TILED, QM_LAYOUT_TILED);
        p.b_e5m2 = 1;
        p.b_wide = qm::six_bits_serve(qm::padded_cols(R)) ? at : nullptr;
        p.mask = at;
        p.hd = hd;
        return p;
    };
    const qm::TileProduct x = product(T, O), w = product(O, T);
    return wide_pair(x, qm::choose_product(x, QM_BF16, QM_BF16, ws ? at : nullptr, ws), w, qm::choose_product(w, QM_BF16, gw_dtype, ws ? at : nullptr, ws)) ? 1 : 0;
}

int qm_linear_backward_error(const void* e, int e_dtype, int64_t T, int64_t I, int64_t O, const void* packed_x, const void* packed_w,
                             int hd_x, const uint32_t* signs_x, int hd_w, const uint32_t* signs_w, int hd_g, const uint32_t* signs_g,
                             int g_mode, const uint64_t* seeds, int x_scale_dtype, int w_scale_dtype, void* workspace,
                             size_t workspace_bytes, void* gx, void* gw, int gw_dtype, void* stream) {
    if (T < 0 || I < 0 || O < 0) return fail(QM_ERR_INVALID, "qm_linear_backward_error: negative extent");
    if (T == 0 || O == 0 || I == 0) return 0;
    if (I % 32 || O % 32 || T % 32 || I >= (1 << 23) || O >= (1 << 23) || T >= (1 << 23))
        return fail(QM_ERR_INVALID, "qm_linear_backward_error: tokens, in_features and out_features must be multiples of 32 below 2^23 (T=%lld I=%lld O=%lld)",
                    (long long)T, (long long)I, (long long)O);
    if (g_mode != QM_ABSMAX_RTN && g_mode != QM_ABSMAX_SR) return fail(QM_ERR_INVALID, "qm_linear_backward_error: g_mode %d", g_mode);
    if (!valid_hd(hd_x) || !valid_hd(hd_w) || !valid_hd(hd_g) || I % hd_x || I % hd_w || T % hd_g || O % hd_g)
        return fail(QM_ERR_INVALID, "qm_linear_backward_error: extents must be multiples of the Hadamard blocks");
    if (!valid_dtype(e_dtype) || !valid_dtype(x_scale_dtype) || !valid_dtype(w_scale_dtype) || !valid_dtype(gw_dtype))
        return fail(QM_ERR_INVALID, "qm_linear_backward_error: dtypes must be QM_BF16/QM_F32");
    if (!e || !seeds || !packed_x || !packed_w || !gx || !gw || !aligned(e, 16) || !aligned(packed_x, 256) || !aligned(packed_w, 256) ||
        !aligned(gx, 16) || !aligned(gw, 16))
        return fail(QM_ERR_INVALID, "qm_linear_backward_error: null or misaligned tensors, seeds or packed operand buffers");
    const ErrorLayout wl = error_layout(T, I, O);
    if (!workspace || workspace_bytes < wl.total || !aligned(workspace, 256))
        return fail(QM_ERR_INVALID, "qm_linear_backward_error: workspace needs %zu bytes, 256-byte aligned", wl.total);
    const PackedLayout lx = packed_layout(T, I), lw = packed_layout(O, I);
    const uint8_t* px = static_cast<const uint8_t*>(packed_x);
    const uint8_t* pw = static_cast<const uint8_t*>(packed_w);
    uint8_t* k = static_cast<uint8_t*>(workspace);
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    const qm::ErrorArgs ae{e, e_dtype, T, O, seeds[0], seeds[1], k + wl.ec, k + wl.es, k + wl.etc, k + wl.ets};
    const qm::E5m2Args ax{px + lx.c, px + lx.s, T, I, k + wl.xv, k + wl.xs, k + wl.xl, qm::six_bits_serve(qm::padded_cols(T)) ? k + wl.xf : nullptr};
    const qm::E5m2Args aw{pw + lw.c, pw + lw.s, O, I, k + wl.wv, k + wl.ws, k + wl.wl, qm::six_bits_serve(qm::padded_cols(O)) ? k + wl.wf : nullptr};
    int rc = from_hip(qm::quantize_error(ae, hd_g, make_signs(signs_g, hd_g), g_mode, ax, aw, hs), "qm_linear_backward_error");
    if (rc) return rc;
    rc = from_hip(qm::expand_e5m2_pair(ax, aw, hs), "qm_linear_backward_error");
    if (rc) return rc;
    // value = code * 2^k * fl32(4/3) on the error signal, code * 2^k on the saved operand
    const float alpha = (float)(1.0 / 0.75);
    void* gws = wl.gemm_ws_bytes ? k + wl.gemm_ws : nullptr;
    // one gradient: the product, then the masked inverse rotation of the forward quantizer, in the product's kernel where that is cheaper
    const auto product_of = [&](size_t ac, size_t as, const qm::E5m2Args& b, int64_t M, void* out, int hd, const uint32_t* signs, int scale_dtype, const uint8_t* mask) {
        qm::TileProduct p = qm::make_product(k + ac, k + as, b.values, b.scales, M, I, qm::padded_cols(b.R), alpha, out, QM_LAYOUT_TILED, QM_LAYOUT_TILED);
        p.b_e5m2 = 1;
        p.b_wide = b.wide;
        p.mask = mask;
        p.hd = hd;
        p.signs = make_signs(signs, hd);
        p.rot_c = qm::hadamard_scale(hd, scale_dtype);
        return p;
    };
    const auto gradient = [&](qm::TileProduct p, const qm::ProductChoice& c, int out_dtype, int scale_dtype) {
        if (c.rotates) return qm::run_product(c, p, QM_BF16, out_dtype, gws, hs);
        void* out = p.c;
        const uint8_t* mask = p.mask;
        p.mask = nullptr;
        p.c = k + wl.plain;
        const hipError_t e1 = qm::run_product(c, p, QM_BF16, QM_BF16, gws, hs);
        return e1 != hipSuccess ? e1 : qm::masked_hadamard_bwd(p.c, QM_BF16, p.M, I, p.hd, scale_dtype, p.signs, mask, out, out_dtype, out_dtype != QM_BF16, hs);
    };
    const qm::TileProduct gxp = product_of(wl.ec, wl.es, aw, T, gx, hd_x, signs_x, x_scale_dtype, px + lx.m);
    const qm::TileProduct gwp = product_of(wl.etc, wl.ets, ax, O, gw, hd_w, signs_w, w_scale_dtype, pw + lw.m);
    const qm::ProductChoice cx = qm::choose_product(gxp, QM_BF16, QM_BF16, gws, wl.gemm_ws_bytes), cw = qm::choose_product(gwp, QM_BF16, gw_dtype, gws, wl.gemm_ws_bytes);
    if (wide_pair(gxp, cx, gwp, cw)) {
        rc = from_hip(O > T ? qm::gemm_wide_pair(gxp, false, gwp, gw_dtype != QM_BF16, hs) : qm::gemm_wide_pair(gwp, gw_dtype != QM_BF16, gxp, false, hs), "qm_linear_backward_error");
        if (rc) return rc;
    } else {
        rc = from_hip(gradient(gxp, cx, QM_BF16, x_scale_dtype), "qm_linear_backward_error");
        if (rc) return rc;
        rc = from_hip(gradient(gwp, cw, gw_dtype, w_scale_dtype), "qm_linear_backward_error");
        if (rc) return rc;
    }
    const auto exact = [&](size_t ac, size_t as, const qm::E5m2Args& b, int64_t M, void* out, int out_dtype, int hd, const uint32_t* signs, int scale_dtype,
                           const uint8_t* mask) {
        return qm::E5m2Exact{k + ac, k + as, b, M, alpha, mask, hd, make_signs(signs, hd), qm::hadamard_scale(hd, scale_dtype), out, out_dtype};
    };
    return from_hip(qm::e5m2_exact_pair(exact(wl.ec, wl.es, aw, T, gx, QM_BF16, hd_x, signs_x, x_scale_dtype, px + lx.m),
                                        exact(wl.etc, wl.ets, ax, O, gw, gw_dtype, hd_w, signs_w, w_scale_dtype, pw + lw.m), hs), "qm_linear_backward_error");
}

int qm_linear_backward(const void* e, int e_dtype, int64_t T, int64_t I, int64_t O, const void* packed_x, const void* packed_w,
                       int hd_x, const uint32_t* signs_x, int hd_w, const uint32_t* signs_w, int hd_g, const uint32_t* signs_g,
                       int g_mode, const uint64_t* seeds, int x_val_dtype, int w_val_dtype, int mid_dtype, int x_scale_dtype,
                       int w_scale_dtype, void* workspace, size_t workspace_bytes, void* gx, void* gw, int gw_dtype,
                       int codes_layout, int rotated_flags, const float* g_matrix, void* stream) {
    return qm_linear_backward_seeded(e, e_dtype, T, I, O, packed_x, packed_w, hd_x, signs_x, hd_w, signs_w, hd_g, signs_g, g_mode, seeds,
                                     x_val_dtype, w_val_dtype, mid_dtype, x_scale_dtype, w_scale_dtype, workspace, workspace_bytes, gx,
                                     gw, gw_dtype, codes_layout, rotated_flags, g_matrix, nullptr, stream);
}

int qm_linear_backward_seeded(const void* e, int e_dtype, int64_t T, int64_t I, int64_t O, const void* packed_x,
                              const void* packed_w, int hd_x, const uint32_t* signs_x, int hd_w, const uint32_t* signs_w, int hd_g,
                              const uint32_t* signs_g, int g_mode, const uint64_t* seeds, int x_val_dtype, int w_val_dtype,
                              int mid_dtype, int x_scale_dtype, int w_scale_dtype, void* workspace, size_t workspace_bytes, void* gx,
                              void* gw, int gw_dtype, int codes_layout, int rotated_flags, const float* g_matrix,
                              const uint64_t* seed_base, void* stream) {
    if (T < 0 || I < 0 || O < 0) return fail(QM_ERR_INVALID, "qm_linear_backward: negative extent");
    if (!valid_layer_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_linear_backward: unknown codes_layout %d", codes_layout);
    if (seed_base && (!aligned(seed_base, 8) || g_matrix || !seed_base_served(codes_layout, T, I, O, hd_x, hd_w, hd_g)))
        return fail(QM_ERR_INVALID, "qm_linear_backward_seeded: a device seed base needs the tiled layout with Hadamard blocks 32, "
                                    "T, I, O multiples of 128, no dense rotation, and an 8-byte aligned pointer");
    if (T == 0 || O == 0 || I == 0) return 0;
    if (g_mode != QM_ABSMAX_RTN && g_mode != QM_ABSMAX_SR)
        return fail(QM_ERR_INVALID, "qm_linear_backward: gradient mode must be QM_ABSMAX_RTN or QM_ABSMAX_SR");
    if (!valid_dtype(mid_dtype)) return fail(QM_ERR_INVALID, "qm_linear_backward: mid_dtype %d", mid_dtype);
    if (gw_dtype != mid_dtype && !(mid_dtype == QM_BF16 && gw_dtype == QM_F32))
        return fail(QM_ERR_INVALID, "qm_linear_backward: gw_dtype must be mid_dtype, or QM_F32 with a bf16 mid_dtype (got %d, mid %d)",
                    gw_dtype, mid_dtype);
    if (I % 32 || O % 32 || T % 32)
        return fail(QM_ERR_INVALID, "qm_linear_backward: tokens, in_features and out_features must be multiples of 32 (T=%lld I=%lld O=%lld)",
                    (long long)T, (long long)I, (long long)O);
    if (!seeds || !packed_x || !aligned(packed_x, 256) || !packed_w || !aligned(packed_w, 256))
        return fail(QM_ERR_INVALID, "qm_linear_backward: null seeds or packed operand buffers");
    const PackedLayout lx = packed_layout(T, I), lw = packed_layout(O, I);
    const WorkLayout wl = work_layout(T, I, O, mid_dtype);
    if (!workspace || workspace_bytes < wl.total || !aligned(workspace, 256))
        return fail(QM_ERR_INVALID, "qm_linear_backward: workspace needs %zu bytes, 256-byte aligned", wl.total);
    const uint8_t* px = static_cast<const uint8_t*>(packed_x);
    const uint8_t* pw = static_cast<const uint8_t*>(packed_w);
    uint8_t* k = static_cast<uint8_t*>(workspace);
    // value = code * 2^k * fl32(4/3) on both operands of the two gradient products
    const float d = (float)(1.0 / 0.75);
    const float alpha = d * d;
    void* gws = wl.gemm_ws_bytes ? k + wl.gemm_ws : nullptr;
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    int rc;
    // rotated_flags: bit 0 (QM_GX_ROTATED): the caller undoes the activation quantizer's rotation itself (fused into its
    // next kernel, or a dense rotation it applies with a library product); the first product then lands in gx directly.
    // Bit 1 (QM_GW_ROTATED): the same for the weight quantizer's rotation and gw.
    if (rotated_flags & ~(QM_GX_ROTATED | QM_GW_ROTATED)) return fail(QM_ERR_INVALID, "qm_linear_backward: unknown rotated flags %d", rotated_flags);
    const bool gx_rotated = rotated_flags & QM_GX_ROTATED, gw_rotated = rotated_flags & QM_GW_ROTATED;
    if (gw_rotated && gw_dtype != mid_dtype) return fail(QM_ERR_INVALID, "qm_linear_backward: QM_GW_ROTATED needs gw_dtype == mid_dtype");
    void* gx_product = gx_rotated ? gx : static_cast<void*>(k + wl.gxq);
    void* gw_product = gw_rotated ? gw : static_cast<void*>(k + wl.gwq);
    // B8: gw in gw_dtype; a bf16 result widened to fp32 keeps its bf16 rounding (what converting it afterwards would give)
    const auto rotate_gw = [&]() -> int {
        if (gw_rotated) return 0;
        if (gw_dtype == mid_dtype)
            return qm_masked_hadamard_bwd(k + wl.gwq, mid_dtype, O, I, hd_w, w_scale_dtype, signs_w, pw + lw.m, gw, mid_dtype, stream);
        if (!valid_hd(hd_w) || I % hd_w || !gw || !aligned(gw, 16) || !valid_dtype(w_scale_dtype))
            return fail(QM_ERR_INVALID, "qm_linear_backward: bad hd_w, w_scale_dtype or gw");
        return from_hip(qm::masked_hadamard_bwd(k + wl.gwq, mid_dtype, O, I, hd_w, w_scale_dtype, make_signs(signs_w, hd_w), pw + lw.m, gw,
                                                gw_dtype, true, hs), "qm_linear_backward");
    };
    if (gx_rotated && hd_x != 32) return fail(QM_ERR_INVALID, "qm_linear_backward: gx_rotated needs hd_x == 32");
    // B3 + B7 and B6 + B8: where the kernel that serves a gradient product applies the masked inverse rotation of the forward
    // quantizer before it stores the result (choose_product tells), the product lands in gx / gw directly; otherwise it goes
    // to the workspace and the rotation is a kernel of its own.
    const bool tiled = tiled_layout(codes_layout);
    if (codes_layout == QM_LAYOUT_TILED && (T % 128 || I % 128 || O % 128))
        return fail(QM_ERR_INVALID, "qm_linear_backward: QM_LAYOUT_TILED needs T, I, O multiples of 128 (QM_LAYOUT_PADDED takes any multiples of 32)");
    const int64_t Kx = tiled ? qm::padded_cols(O) : O, Kw = tiled ? qm::padded_cols(T) : T;
    const int kl = kernel_layout(codes_layout);
    const bool blocks_ok = valid_hd(hd_x) && valid_hd(hd_w) && I % hd_x == 0 && I % hd_w == 0 && valid_dtype(x_scale_dtype) && valid_dtype(w_scale_dtype);
    const qm::PairChoice pair = tiled && !g_matrix && mid_dtype == QM_BF16 && blocks_ok ? gradient_pair(T, I, O, hd_x, hd_w, signs_x, signs_w, gw_dtype)
                                                                                        : qm::PairChoice{qm::PairChoice::SEPARATE, 0, 0};
    const qm::TileProduct gx_plain = qm::make_product(k + wl.ec, k + wl.es, k + wl.wtc, k + wl.wts, T, I, Kx, alpha, gx_product, kl, kl);
    const qm::TileProduct gw_plain = qm::make_product(k + wl.etc, k + wl.ets, k + wl.xtc, k + wl.xts, O, I, Kw, alpha, gw_product, kl, kl);
    qm::TileProduct gx_whole = gx_plain, gw_whole = gw_plain;
    if (pair.path != qm::PairChoice::SEPARATE) {
        if (!gx_rotated) gx_whole = with_rotation(gx_plain, gx, hd_x, px + lx.m, signs_x, x_scale_dtype);
        if (!gw_rotated) gw_whole = with_rotation(gw_plain, gw, hd_w, pw + lw.m, signs_w, w_scale_dtype);
    }
    const bool together = qm::pair_serves(pair, gx_whole, mid_dtype, gw_whole, gw_dtype);
    // a call whose form that launch does not take (no rotation at all) runs two, without K ranges like the others of its layer
    void* cuts = pair.path == qm::PairChoice::SEPARATE ? gws : nullptr;
    const auto plan = [&](const qm::TileProduct& plain, void* dst, bool rotated, int hd, int dtype, const uint8_t* mask, const uint32_t* signs, int scale_dtype) {
        return together ? GradProduct{} : plan_gradient(plain, dst, !rotated, hd, mid_dtype, dtype, mask, signs, scale_dtype, cuts, wl.gemm_ws_bytes);
    };
    const GradProduct gx_plan = plan(gx_plain, gx, gx_rotated, hd_x, mid_dtype, px + lx.m, signs_x, x_scale_dtype);
    const GradProduct gw_plan = plan(gw_plain, gw, gw_rotated, hd_w, gw_dtype, pw + lw.m, signs_w, w_scale_dtype);
    const bool gx_fused = gx_plan.choice.rotates, gw_fused = gw_plan.choice.rotates;
    const auto run = [&](const GradProduct& g) {
        return from_hip(qm::run_product(g.choice, g.p, mid_dtype, g.out_dtype, gws, hs), "qm_linear_backward");
    };
    const auto product_gx = [&]() { return run(gx_plan); };
    const auto product_gw = [&]() { return run(gw_plan); };
    if (g_matrix) {
        // a dense rotation in the gradient quantizer (rerotate="O32"): the same eight steps on the dense-rotation kernels
        if (hd_g != 32 || T % 128 || I % 128 || O % 128)
            return fail(QM_ERR_INVALID, "qm_linear_backward: a dense gradient rotation needs hd_g == 32 and T, I, O multiples of 128 "
                                        "(T=%lld I=%lld O=%lld)", (long long)T, (long long)I, (long long)O);
        rc = qm_quantize_mxfp4_dense(e, e_dtype, T, O, g_matrix, g_mode, 0, seeds[0], k + wl.ec, k + wl.es, nullptr, nullptr, kl, stream);
        if (rc) return rc;
        rc = qm_requantize_transposed_mxfp4_dense(pw + lw.c, pw + lw.s, O, I, 1.0f, w_val_dtype, g_matrix, g_mode, seeds[1], k + wl.wtc,
                                                  k + wl.wts, nullptr, kl, kl, stream);
        if (rc) return rc;
        rc = product_gx();
        if (rc) return rc;
        rc = qm_quantize_mxfp4_dense(e, e_dtype, O, T, g_matrix, g_mode, 1, seeds[2], k + wl.etc, k + wl.ets, nullptr, nullptr, kl, stream);
        if (rc) return rc;
        rc = qm_requantize_transposed_mxfp4_dense(px + lx.c, px + lx.s, T, I, 1.0f, x_val_dtype, g_matrix, g_mode, seeds[3], k + wl.xtc,
                                                  k + wl.xts, nullptr, kl, kl, stream);
        if (rc) return rc;
        rc = product_gw();
        if (rc) return rc;
        if (!gx_rotated && !gx_fused) {
            rc = qm_masked_hadamard_bwd(k + wl.gxq, mid_dtype, T, I, hd_x, x_scale_dtype, signs_x, px + lx.m, gx, mid_dtype, stream);
            if (rc) return rc;
        }
        return gw_fused ? 0 : rotate_gw();
    }
    if (tiled) {
        // the gradient quantizers (Q(e), Q(e^T), Q(Q(W)^T), Q(Q(x)^T)), the two products, the inverse rotations they do not carry
        if (!valid_hd(hd_g) || !valid_hd(hd_x) || !valid_hd(hd_w) || T % hd_g || O % hd_g || I % hd_x || I % hd_w || !e || !gx || !gw || !valid_dtype(e_dtype) ||
            !aligned(e, 16) || !aligned(gx, 16) || !aligned(gw, 16) || !valid_dtype(x_val_dtype) || !valid_dtype(w_val_dtype) ||
            !valid_dtype(x_scale_dtype) || !valid_dtype(w_scale_dtype))
            return fail(QM_ERR_INVALID, "qm_linear_backward: null, misaligned or ill-typed tensors, or extents that are not multiples of the Hadamard blocks");
        const qm::RequantArgs rw{pw + lw.c, pw + lw.s, O, I, w_val_dtype, seeds[1], k + wl.wtc, k + wl.wts};
        const qm::RequantArgs rx{px + lx.c, px + lx.s, T, I, x_val_dtype, seeds[3], k + wl.xtc, k + wl.xts};
        const qm::ErrorArgs ae{e, e_dtype, T, O, seeds[0], seeds[2], k + wl.ec, k + wl.es, k + wl.etc, k + wl.ets};
        rc = from_hip(qm::quantize_layer_backward(ae, hd_g, make_signs(signs_g, hd_g), g_mode, rx, rw, seed_base, hs), "qm_linear_backward");
        if (rc) return rc;
        if (together) return from_hip(qm::run_pair(pair, gx_whole, mid_dtype, gw_whole, gw_dtype, hs), "qm_linear_backward");
        rc = product_gx();
        if (rc) return rc;
        rc = product_gw();
        if (rc) return rc;
        const bool need_x = !gx_rotated && !gx_fused, need_w = !gw_rotated && !gw_fused;
        if (!need_x) return need_w ? rotate_gw() : 0;
        if (!need_w || hd_x != 32 || hd_w != 32) {
            rc = qm_masked_hadamard_bwd(k + wl.gxq, mid_dtype, T, I, hd_x, x_scale_dtype, signs_x, px + lx.m, gx, mid_dtype, stream);
            return rc ? rc : need_w ? rotate_gw() : 0;
        }
        return from_hip(qm::masked_hadamard_bwd_hd32_pair(k + wl.gxq, T * I, x_scale_dtype,
                                                          signs_x ? signs_x[0] : 0u, px + lx.m, gx, k + wl.gwq, O * I,
                                                          w_scale_dtype, signs_w ? signs_w[0] : 0u,
                                                          pw + lw.m, gw, mid_dtype, gw_dtype, hs), "qm_linear_backward");
    }
    if (seed_base) return fail(QM_ERR_INVALID, "qm_linear_backward_seeded: null, misaligned or ill-typed tensors");
    rc = qm_quantize_mxfp4(e, e_dtype, T, O, hd_g, signs_g, g_mode, 0, nullptr, seeds[0], k + wl.ec, k + wl.es, nullptr, nullptr,
                           codes_layout, stream);
    if (rc) return rc;
    rc = qm_requantize_transposed_mxfp4(pw + lw.c, pw + lw.s, O, I, 1.0f, w_val_dtype, hd_g, signs_g, g_mode, nullptr, seeds[1],
                                        k + wl.wtc, k + wl.wts, nullptr, codes_layout, codes_layout, stream);
    if (rc) return rc;
    rc = product_gx();
    if (rc) return rc;
    rc = qm_quantize_mxfp4(e, e_dtype, O, T, hd_g, signs_g, g_mode, 1, nullptr, seeds[2], k + wl.etc, k + wl.ets, nullptr, nullptr,
                           codes_layout, stream);
    if (rc) return rc;
    rc = qm_requantize_transposed_mxfp4(px + lx.c, px + lx.s, T, I, 1.0f, x_val_dtype, hd_g, signs_g, g_mode, nullptr, seeds[3],
                                        k + wl.xtc, k + wl.xts, nullptr, codes_layout, codes_layout, stream);
    if (rc) return rc;
    rc = product_gw();
    if (rc) return rc;
    if (!gx_rotated && !gx_fused) {
        rc = qm_masked_hadamard_bwd(k + wl.gxq, mid_dtype, T, I, hd_x, x_scale_dtype, signs_x, px + lx.m, gx, mid_dtype, stream);
        if (rc) return rc;
    }
    return gw_fused ? 0 : rotate_gw();
}

static int rmsnorm_quantize(const void* x, int x_dtype, const void* add, int add_dtype, void* x_sum, const float* gain, float eps,
                              int64_t rows, int64_t cols, const uint32_t* sign_bits, void* packed, size_t packed_bytes,
                              float* factor, int codes_layout, const qm::RowmajorArgs* weight, void* stream) {
    if (!valid_layer_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: unknown codes_layout %d", codes_layout);
    if (!valid_dtype(x_dtype)) return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: x_dtype %d is not QM_BF16/QM_F32", x_dtype);
    if (rows < 0 || cols <= 0 || cols % 32)
        return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: need rows >= 0 and cols a positive multiple of 32 (got [%lld, %lld])",
                    (long long)rows, (long long)cols);
    if (rows == 0) return 0;
    if (codes_layout == QM_LAYOUT_TILED && (rows % 16 || cols % 128))
        return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: tiled codes need rows %% 16 == 0 and cols %% 128 == 0 (rows=%lld cols=%lld)",
                    (long long)rows, (long long)cols);
    const PackedLayout l = packed_layout(rows, cols);
    if (!x || !gain || !factor || !packed || packed_bytes < l.total)
        return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: x, gain, factor must be non-null and packed hold %zu bytes", l.total);
    if (!aligned(x, 16) || !aligned(gain, 16) || !aligned(packed, 256) || !aligned(factor, 4) || !aligned(add, 16) || !aligned(x_sum, 16))
        return fail(QM_ERR_UNALIGNED, "qm_rmsnorm_quantize_mxfp4: x, add, x_sum and gain need 16-byte, packed 256-byte alignment");
    if (add && (x_dtype != QM_F32 || !valid_dtype(add_dtype) || !x_sum))
        return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_mxfp4: a residual summand needs an fp32 x, a valid add_dtype and x_sum");
    uint8_t* p = static_cast<uint8_t*>(packed);
    return from_hip(qm::rmsnorm_quantize_hd32(x, x_dtype, add, add_dtype, x_sum, gain, eps, rows, cols, sign_bits ? sign_bits[0] : 0u, p + l.c, p + l.s,
                                              p + l.m, factor, tiled_layout(codes_layout), weight, reinterpret_cast<hipStream_t>(stream)),
                    "qm_rmsnorm_quantize_mxfp4");
}

static int swiglu_quantize(const void* h12, int dtype, int64_t rows, int64_t hidden, const uint32_t* sign_bits, void* packed,
                             size_t packed_bytes, int codes_layout, const qm::RowmajorArgs* weight, void* stream) {
    if (!valid_layer_layout(codes_layout)) return fail(QM_ERR_INVALID, "qm_swiglu_quantize_mxfp4: unknown codes_layout %d", codes_layout);
    if (!valid_dtype(dtype)) return fail(QM_ERR_INVALID, "qm_swiglu_quantize_mxfp4: dtype %d is not QM_BF16/QM_F32", dtype);
    if (rows < 0 || hidden <= 0 || hidden % 32)
        return fail(QM_ERR_INVALID, "qm_swiglu_quantize_mxfp4: need rows >= 0 and hidden a positive multiple of 32 (got [%lld, %lld])",
                    (long long)rows, (long long)hidden);
    if (rows == 0) return 0;
    if (codes_layout == QM_LAYOUT_TILED && (rows % 16 || hidden % 128))
        return fail(QM_ERR_INVALID, "qm_swiglu_quantize_mxfp4: tiled codes need rows %% 16 == 0 and hidden %% 128 == 0 (rows=%lld hidden=%lld)",
                    (long long)rows, (long long)hidden);
    const PackedLayout l = packed_layout(rows, hidden);
    if (!h12 || !packed || packed_bytes < l.total)
        return fail(QM_ERR_INVALID, "qm_swiglu_quantize_mxfp4: h12 must be non-null and packed hold %zu bytes", l.total);
    if (!aligned(h12, 16) || !aligned(packed, 256))
        return fail(QM_ERR_UNALIGNED, "qm_swiglu_quantize_mxfp4: h12 needs 16-byte, packed 256-byte alignment");
    uint8_t* p = static_cast<uint8_t*>(packed);
    return from_hip(qm::swiglu_quantize_hd32(h12, dtype, rows, hidden, sign_bits ? sign_bits[0] : 0u, p + l.c, p + l.s, p + l.m,
                                             tiled_layout(codes_layout), weight, reinterpret_cast<hipStream_t>(stream)),
                    "qm_swiglu_quantize_mxfp4");
}

int qm_rmsnorm_quantize_mxfp4(const void* x, int x_dtype, const void* add, int add_dtype, void* x_sum, const float* gain, float eps,
                              int64_t rows, int64_t cols, const uint32_t* sign_bits, void* packed, size_t packed_bytes,
                              float* factor, int codes_layout, void* stream) {
    return rmsnorm_quantize(x, x_dtype, add, add_dtype, x_sum, gain, eps, rows, cols, sign_bits, packed, packed_bytes, factor, codes_layout, nullptr, stream);
}
int qm_swiglu_quantize_mxfp4(const void* h12, int dtype, int64_t rows, int64_t hidden, const uint32_t* sign_bits, void* packed,
                             size_t packed_bytes, int codes_layout, void* stream) {
    return swiglu_quantize(h12, dtype, rows, hidden, sign_bits, packed, packed_bytes, codes_layout, nullptr, stream);
}

namespace {
// the weight that a producer's grid takes along: fp32 [out_features, cols], QM_LAYOUT_PADDED
int weight_args(const char* who, const void* w, int64_t out_features, int64_t cols, const uint32_t* signs_w, void* packed_w, size_t packed_w_bytes,
                qm::RowmajorArgs* a) {
    if (out_features <= 0 || out_features >= (1ll << 31) - 16 || cols <= 0 || cols % 32)
        return fail(QM_ERR_INVALID, "%s: need a weight [out_features, %lld]", who, (long long)cols);
    const PackedLayout l = packed_layout(out_features, cols);
    if (!w || !aligned(w, 16) || !packed_w || packed_w_bytes < l.total || !aligned(packed_w, 256))
        return fail(QM_ERR_INVALID, "%s: w must be non-null and 16-byte aligned, packed_w hold %zu bytes, 256-byte aligned", who, l.total);
    uint8_t* p = static_cast<uint8_t*>(packed_w);
    *a = qm::RowmajorArgs{w, QM_F32, out_features, cols, make_signs(signs_w, 32), p + l.c, p + l.s, p + l.m};
    return 0;
}
}  // namespace

int qm_rmsnorm_quantize_with_weight_mxfp4(const void* x, int x_dtype, const void* add, int add_dtype, void* x_sum, const float* gain, float eps,
                                          int64_t rows, int64_t cols, const uint32_t* sign_bits, void* packed, size_t packed_bytes, float* factor,
                                          const float* w, int64_t out_features, const uint32_t* signs_w, void* packed_w, size_t packed_w_bytes, void* stream) {
    if (x_dtype != QM_F32 || (add && add_dtype != QM_BF16) || rows <= 0)
        return fail(QM_ERR_INVALID, "qm_rmsnorm_quantize_with_weight_mxfp4: needs rows, an fp32 x and a bf16 summand or none");
    qm::RowmajorArgs a;
    if (int rc = weight_args("qm_rmsnorm_quantize_with_weight_mxfp4", w, out_features, cols, signs_w, packed_w, packed_w_bytes, &a)) return rc;
    return rmsnorm_quantize(x, x_dtype, add, add_dtype, x_sum, gain, eps, rows, cols, sign_bits, packed, packed_bytes, factor, QM_LAYOUT_PADDED, &a, stream);
}
int qm_swiglu_quantize_with_weight_mxfp4(const void* h12, int dtype, int64_t rows, int64_t hidden, const uint32_t* sign_bits, void* packed,
                                         size_t packed_bytes, const float* w, int64_t out_features, const uint32_t* signs_w, void* packed_w,
                                         size_t packed_w_bytes, void* stream) {
    if (dtype != QM_BF16 || rows <= 0) return fail(QM_ERR_INVALID, "qm_swiglu_quantize_with_weight_mxfp4: needs rows of a bf16 h12");
    qm::RowmajorArgs a;
    if (int rc = weight_args("qm_swiglu_quantize_with_weight_mxfp4", w, out_features, hidden, signs_w, packed_w, packed_w_bytes, &a)) return rc;
    return swiglu_quantize(h12, dtype, rows, hidden, sign_bits, packed, packed_bytes, QM_LAYOUT_PADDED, &a, stream);
}

size_t qm_rmsnorm_backward_workspace_bytes(int64_t rows, int64_t cols) {
    if (rows < 0 || cols <= 0 || cols % 32 || cols > 8192) return 0;
    return up256(qm::rmsnorm_backward_workspace_bytes(rows, cols));
}

int qm_rmsnorm_backward(const void* gy, int gy_dtype, const void* x, int x_dtype, const float* gain, const float* factor,
                        int64_t rows, int64_t cols, const uint8_t* maskbits, const uint32_t* sign_bits, int scale_dtype,
                        const void* skip, void* dx, void* dx_bf16, float* dgain, void* workspace, size_t workspace_bytes,
                        void* stream) {
    if (!valid_dtype(gy_dtype) || !valid_dtype(x_dtype) || (maskbits && !valid_dtype(scale_dtype)))
        return fail(QM_ERR_INVALID, "qm_rmsnorm_backward: dtypes must be QM_BF16/QM_F32");
    if (rows < 0 || cols <= 0 || cols % 32 || cols > 8192)
        return fail(QM_ERR_INVALID, "qm_rmsnorm_backward: need rows >= 0 and cols a multiple of 32 in [32, 8192] (got [%lld, %lld])",
                    (long long)rows, (long long)cols);
    if (!dgain) return fail(QM_ERR_INVALID, "qm_rmsnorm_backward: dgain must be non-null");
    if (rows > 0 && (!gy || !x || !gain || !factor || !dx || !workspace || workspace_bytes < qm::rmsnorm_backward_workspace_bytes(rows, cols)))
        return fail(QM_ERR_INVALID, "qm_rmsnorm_backward: null tensor, or workspace below %zu bytes", qm_rmsnorm_backward_workspace_bytes(rows, cols));
    if (!aligned(maskbits, 4)) return fail(QM_ERR_UNALIGNED, "qm_rmsnorm_backward: maskbits needs 4-byte alignment");
    if (!aligned(skip, 16) || !aligned(dx_bf16, 8) || !aligned(gy, 8) || !aligned(x, 8) || !aligned(dx, 8) || !aligned(gain, 16) || !aligned(workspace, 16) ||
        (gy_dtype == QM_F32 && !aligned(gy, 16)) || (x_dtype == QM_F32 && (!aligned(x, 16) || !aligned(dx, 16))))
        return fail(QM_ERR_UNALIGNED, "qm_rmsnorm_backward: tensors need 16-byte alignment");
    return from_hip(qm::rmsnorm_backward(gy, gy_dtype, x, x_dtype, gain, factor, rows, cols, maskbits, sign_bits ? sign_bits[0] : 0u,
                                         maskbits ? scale_dtype : QM_F32, skip, dx, dx_bf16, dgain, workspace,
                                         reinterpret_cast<hipStream_t>(stream)),
                    "qm_rmsnorm_backward");
}

int qm_swiglu_backward(const void* g, int g_dtype, const void* h12, int dtype, int64_t rows, int64_t hidden,
                       const uint8_t* maskbits, const uint32_t* sign_bits, int scale_dtype, void* d_h12, void* stream) {
    if (!valid_dtype(g_dtype) || !valid_dtype(dtype) || (maskbits && !valid_dtype(scale_dtype)))
        return fail(QM_ERR_INVALID, "qm_swiglu_backward: dtypes must be QM_BF16/QM_F32");
    if (rows < 0 || hidden <= 0 || hidden % 4 || (maskbits && hidden % 32))
        return fail(QM_ERR_INVALID, "qm_swiglu_backward: need rows >= 0 and hidden a positive multiple of 4 (of 32 with mask bits) "
                                    "(got [%lld, %lld])", (long long)rows, (long long)hidden);
    if (rows == 0) return 0;
    if (!g || !h12 || !d_h12) return fail(QM_ERR_INVALID, "qm_swiglu_backward: g, h12 and d_h12 must be non-null");
    if (!aligned(g, 16) || !aligned(h12, 16) || !aligned(d_h12, 16))
        return fail(QM_ERR_UNALIGNED, "qm_swiglu_backward: tensors need 16-byte alignment");
    return from_hip(qm::swiglu_backward(g, g_dtype, h12, dtype, rows, hidden, maskbits, sign_bits ? sign_bits[0] : 0u,
                                        maskbits ? scale_dtype : QM_F32, d_h12, reinterpret_cast<hipStream_t>(stream)),
                    "qm_swiglu_backward");
}

namespace {
int check_rope(const char* who, int dtype_a, int dtype_b, int64_t rows, int64_t seq_len, int64_t n_embd, int head_dim) {
    if (!valid_dtype(dtype_a) || !valid_dtype(dtype_b)) return fail(QM_ERR_INVALID, "%s: dtypes must be QM_BF16/QM_F32", who);
    if (rows < 0 || seq_len <= 0 || n_embd <= 0 || head_dim <= 0 || head_dim % 8 || n_embd % head_dim || n_embd > (1 << 24) ||
        seq_len > (1 << 30))
        return fail(QM_ERR_INVALID, "%s: need rows >= 0, seq_len > 0, head_dim a positive multiple of 8 and n_embd a multiple of "
                                    "head_dim (rows=%lld seq_len=%lld n_embd=%lld head_dim=%d)",
                    who, (long long)rows, (long long)seq_len, (long long)n_embd, head_dim);
    return 0;
}
}  // namespace

int qm_rope_split_qkv(const void* qkv, int qkv_dtype, int64_t rows, int64_t seq_len, int64_t n_embd, int head_dim,
                      const float* table, void* q, void* k, void* v, int out_dtype, void* stream) {
    if (int rc = check_rope("qm_rope_split_qkv", qkv_dtype, out_dtype, rows, seq_len, n_embd, head_dim)) return rc;
    if (rows == 0) return 0;
    if (!qkv || !table || !q || !k || !v) return fail(QM_ERR_INVALID, "qm_rope_split_qkv: qkv, table, q, k, v must be non-null");
    if (!aligned(qkv, 16) || !aligned(table, 16) || !aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16))
        return fail(QM_ERR_UNALIGNED, "qm_rope_split_qkv: tensors need 16-byte alignment");
    return from_hip(qm::rope_split_qkv(qkv, qkv_dtype, rows, (int)seq_len, (int)n_embd, head_dim, table, q, k, v, out_dtype,
                                       reinterpret_cast<hipStream_t>(stream)),
                    "qm_rope_split_qkv");
}

int qm_rope_merge_qkv_grad(const void* dq, const void* dk, const void* dv, int grad_dtype, int64_t rows, int64_t seq_len,
                           int64_t n_embd, int head_dim, const float* table, void* d_qkv, int out_dtype, void* stream) {
    if (int rc = check_rope("qm_rope_merge_qkv_grad", grad_dtype, out_dtype, rows, seq_len, n_embd, head_dim)) return rc;
    if (rows == 0) return 0;
    if (!dq || !dk || !dv || !table || !d_qkv)
        return fail(QM_ERR_INVALID, "qm_rope_merge_qkv_grad: dq, dk, dv, table, d_qkv must be non-null");
    if (!aligned(dq, 16) || !aligned(dk, 16) || !aligned(dv, 16) || !aligned(table, 16) || !aligned(d_qkv, 16))
        return fail(QM_ERR_UNALIGNED, "qm_rope_merge_qkv_grad: tensors need 16-byte alignment");
    return from_hip(qm::rope_merge_qkv_grad(dq, dk, dv, grad_dtype, rows, (int)seq_len, (int)n_embd, head_dim, table, d_qkv, out_dtype,
                                            reinterpret_cast<hipStream_t>(stream)),
                    "qm_rope_merge_qkv_grad");
}

int qm_rmsnorm(const float* x, const void* add, int add_dtype, const float* gain, float eps, int64_t rows, int64_t cols, void* out, int out_dtype, void* stream) {
    if (!valid_dtype(out_dtype) || (add && !valid_dtype(add_dtype))) return fail(QM_ERR_INVALID, "qm_rmsnorm: dtypes must be QM_BF16/QM_F32");
    if (rows < 0 || rows >= (1ll << 32) || cols <= 0 || cols % 4 || cols > 4096)
        return fail(QM_ERR_INVALID, "qm_rmsnorm: need 0 <= rows < 2^32 and cols a multiple of 4 in [4, 4096] (got [%lld, %lld])", (long long)rows, (long long)cols);
    if (rows == 0) return 0;
    if (!x || !gain || !out) return fail(QM_ERR_INVALID, "qm_rmsnorm: x, gain and out must be non-null");
    if (!aligned(x, 16) || !aligned(add, 16) || !aligned(gain, 16) || !aligned(out, 16)) return fail(QM_ERR_UNALIGNED, "qm_rmsnorm: tensors need 16-byte alignment");
    return from_hip(qm::rmsnorm_rows(x, add, add_dtype, gain, eps, rows, cols, out, out_dtype, reinterpret_cast<hipStream_t>(stream)), "qm_rmsnorm");
}

namespace {
struct LogitsLayout {   // a workspace of qm_logits_loss
    size_t x, w, parts, losses, total;
};
LogitsLayout logits_layout(int64_t T, int64_t K, int64_t V) {
    LogitsLayout l;
    l.x = 0;
    l.w = l.x + up256((size_t)qm::padded_rows(T) * K * 2);
    l.parts = l.w + up256((size_t)qm::padded_rows(V) * K * 2);
    l.losses = l.parts + up256((size_t)qm::gemm_logits_segments(V) * T * 8);
    l.total = l.losses + up256((size_t)T * 4);
    return l;
}
}  // namespace

size_t qm_logits_loss_workspace_bytes(int64_t T, int64_t K, int64_t V) { return qm::gemm_logits_serves(T, V, K) && K <= 4096 ? logits_layout(T, K, V).total : 0; }

int qm_logits_loss(const float* x, const void* add, int add_dtype, const float* gain, float eps, int64_t T, int64_t K, const float* w, int64_t V,
                   const int64_t* targets, int64_t ignore_index, void* workspace, size_t workspace_bytes, void* logits, float* loss, void* stream) {
    if (add && !valid_dtype(add_dtype)) return fail(QM_ERR_INVALID, "qm_logits_loss: add_dtype must be QM_BF16/QM_F32");
    const size_t need = qm_logits_loss_workspace_bytes(T, K, V);
    if (!need)
        return fail(QM_ERR_INVALID, "qm_logits_loss: need rows, in_features a multiple of 32 in [64, 4096] and classes a multiple of 8 (got [%lld, %lld] x %lld)", (long long)T,
                    (long long)K, (long long)V);
    if (!x || !gain || !w || !targets || !logits || !loss || !workspace || workspace_bytes < need)
        return fail(QM_ERR_INVALID, "qm_logits_loss: null tensor, or workspace below %zu bytes", need);
    if (!aligned(x, 16) || !aligned(add, 16) || !aligned(gain, 16) || !aligned(w, 16) || !aligned(logits, 16) || !aligned(workspace, 256) || !aligned(targets, 8) || !aligned(loss, 4))
        return fail(QM_ERR_UNALIGNED, "qm_logits_loss: tensors need 16-byte, the workspace 256-byte alignment");
    const LogitsLayout l = logits_layout(T, K, V);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    float* losses = reinterpret_cast<float*>(ws + l.losses);
    hipError_t e = qm::bf16_blocks(w, V, K, ws + l.w, hs);
    if (e == hipSuccess) e = qm::rmsnorm_rows(x, add, add_dtype, gain, eps, T, K, ws + l.x, QM_BF16, hs, true);
    if (e == hipSuccess) e = qm::gemm_logits(ws + l.x, ws + l.w, T, V, K, logits, ws + l.parts, hs);
    if (e == hipSuccess) e = qm::logits_loss_rows(ws + l.parts, qm::gemm_logits_segments(V), T, logits, V, targets, ignore_index, losses, hs);
    if (e == hipSuccess) e = qm::loss_mean(losses, targets, T, ignore_index, loss, hs);
    return from_hip(e, "qm_logits_loss");
}

int qm_diag_forward_kernel(int64_t T, int64_t I, int64_t O, int y_dtype) {
    if (T <= 0 || I <= 0 || O <= 0 || I % 32 || O % 8 || T >= (1 << 30) || I >= (1 << 23) || O >= (1 << 30) || !valid_dtype(y_dtype)) return 0;
    const PackedLayout lx = packed_layout(T, I), lw = packed_layout(O, I);
    const uint8_t *px = reinterpret_cast<const uint8_t*>((uintptr_t)256), *pw = px + lx.total;   // nothing is read
    const qm::TileProduct p = qm::make_product(px + lx.c, px + lx.s, pw + lw.c, pw + lw.s, T, O, qm::padded_cols(I), 1.0f, const_cast<uint8_t*>(px), QM_LAYOUT_TILED, QM_LAYOUT_TILED);
    if (T <= 64 && qm::gemm_rows_serves(p)) return 1;
    const qm::ProductChoice c = qm::choose_product(p, y_dtype, y_dtype, nullptr, 0);
    if (c.path == qm::ProductChoice::TILE) return c.kind == qm::TILE_128x128 && qm::gemm_tile_deep(p) ? 32 : 16 + c.kind;
    return c.path == qm::ProductChoice::PERSISTENT ? 2 : c.path == qm::ProductChoice::TWO ? 3 : 0;
}

int qm_diag_silu_bf16(uint16_t* out, void* stream) {
    if (!out) return fail(QM_ERR_INVALID, "qm_diag_silu_bf16: out must be non-null");
    return from_hip(qm::silu_of_bf16_table(out, reinterpret_cast<hipStream_t>(stream)), "qm_diag_silu_bf16");
}

int qm_cross_entropy(const void* logits, int logits_dtype, const int64_t* targets, int64_t rows, int64_t classes,
                     int64_t ignore_index, float* row_losses, float* loss, void* stream) {
    if (!valid_dtype(logits_dtype)) return fail(QM_ERR_INVALID, "qm_cross_entropy: logits_dtype must be QM_BF16/QM_F32");
    if (rows < 0 || rows >= (1ll << 31) || classes <= 0)
        return fail(QM_ERR_INVALID, "qm_cross_entropy: need 0 <= rows < 2^31 and classes > 0 (got [%lld, %lld])", (long long)rows, (long long)classes);
    if (!loss || (rows > 0 && (!logits || !targets || !row_losses)))
        return fail(QM_ERR_INVALID, "qm_cross_entropy: logits, targets, row_losses and loss must be non-null");
    if (!aligned(logits, logits_dtype == QM_BF16 ? 2 : 4) || !aligned(targets, 8) || !aligned(row_losses, 4) || !aligned(loss, 4))
        return fail(QM_ERR_UNALIGNED, "qm_cross_entropy: tensors must be aligned to their elements");
    return from_hip(qm::cross_entropy_mean(logits, logits_dtype, targets, rows, classes, ignore_index, row_losses, loss,
                                           reinterpret_cast<hipStream_t>(stream)),
                    "qm_cross_entropy");
}

}  // extern "C"
