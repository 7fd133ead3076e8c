// Internal C++ entry points of the HIP kernels; the public C ABI (include/quartet_hip.h) wraps
// these after validating shapes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qm {

// bit j set = rotated column j is negated (H = c * S * diag(signs)); hd <= 128 columns
struct SignBits {
    uint32_t w[4];
};

// Code-byte layouts of a packed [R, C] tensor.  ROWMAJOR: [R][C/2].  TILED (R % 16 == 0, C % 128 == 0):
// [R/16][C/128][16 rows][64 bytes] -- the 16 rows x 128 elements one GEMM wave-load fetches are 1 KiB contiguous.
enum CodeLayout : int { LAYOUT_ROWMAJOR = 0, LAYOUT_TILED = 1 };

// A tiled operand of any extents is stored with its rows padded to 16 and its columns to 128: the padding columns hold zero
// codes and zero scale bytes (they add exact zeros to a product), the padding rows are never consumed.
__host__ __device__ inline int64_t padded_rows(int64_t r) { return (r + 15) & ~(int64_t)15; }
__host__ __device__ inline int64_t padded_cols(int64_t c) { return (c + 127) & ~(int64_t)127; }

// byte offset of the 64-byte piece (row r, column block kb) in the tiled layout
__host__ __device__ inline int64_t tiled_code_offset(int64_t r, int64_t kb, int64_t kblocks) {
    return (((r >> 4) * kblocks + kb) << 10) + ((r & 15) << 6);
}

hipError_t quantize_mxfp4(const void* x, int dtype, int64_t rows, int64_t cols, int hd, const SignBits& sb, int mode,
                          bool transposed_in, const float* u, uint64_t seed, uint8_t* codes, uint8_t* scales,
                          uint8_t* maskbits, void* dequant, int codes_layout, hipStream_t stream);
// its de-quantized values and clip mask (or null) alone: row-major x, in-kernel random numbers, hd 32, 64 or 128
hipError_t quantize_values(const void* x, int dtype, int64_t rows, int64_t cols, int hd, const SignBits& sb, int mode, uint64_t seed, uint8_t* maskbits,
                           void* values, hipStream_t stream);
// whether quantize_mxfp4 / requantize_transposed_mxfp4 can emit (read) tiled codes for these arguments
bool quantize_supports_tiled(int64_t rows, int64_t cols, int hd, int mode, bool transposed_in, const float* u,
                             const uint8_t* maskbits);
bool requantize_supports_tiled(int64_t R, int64_t C, int hd, int mode, const float* u);
bool gemm_supports_tiled(int64_t M, int64_t N, int64_t K);

// hd = 32 fast path (one MX group per lane, hardware FP4 converts); row-major input, RTN or Philox SR
hipError_t quantize_rowmajor_hd32(const void* x, int dtype, int64_t rows, int64_t cols, uint32_t sign_word, int mode,
                                  uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant,
                                  bool tiled, bool rotate, hipStream_t stream);

hipError_t quantize_rowmajor_wide(const void* x, int dtype, int64_t n, int hd, const SignBits& sb, int mode, uint64_t seed,
                                  uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant, hipStream_t stream);

hipError_t quantize_transposed_hd32(const void* x, int dtype, int64_t P, int64_t Q, uint32_t sign_word, int mode,
                                    uint64_t seed, uint8_t* codes, uint8_t* scales, void* dequant, bool tiled,
                                    hipStream_t stream);
hipError_t requantize_transposed_hd32(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                      int val_dtype, uint32_t sign_word, int mode, uint64_t seed, uint8_t* codes,
                                      uint8_t* scales, void* dequant, bool tiled_in, bool tiled_out, hipStream_t stream);

// The same with a dense 32x32 rotation instead of the Hadamard block (matrix: device pointer, [32][32] fp32, H[k][j])
hipError_t quantize_rowmajor_dense(const void* x, int dtype, int64_t rows, int64_t cols, const float* matrix, int mode,
                                   uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant,
                                   bool tiled, hipStream_t stream);
hipError_t quantize_transposed_dense(const void* x, int dtype, int64_t P, int64_t Q, const float* matrix, int mode,
                                     uint64_t seed, uint8_t* codes, uint8_t* scales, void* dequant, bool tiled,
                                     hipStream_t stream);
hipError_t requantize_transposed_dense(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                       int val_dtype, const float* matrix, int mode, uint64_t seed, uint8_t* codes,
                                       uint8_t* scales, void* dequant, bool tiled_in, bool tiled_out, hipStream_t stream);
// shape-checked front ends of the three (what the C ABI calls); hipErrorInvalidValue for shapes they do not serve
hipError_t quantize_mxfp4_dense(const void* x, int dtype, int64_t rows, int64_t cols, const float* matrix, int mode,
                                bool transposed_in, uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits,
                                void* dequant, int codes_layout, hipStream_t stream);
hipError_t requantize_transposed_mxfp4_dense(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C,
                                             float post, int val_dtype, const float* matrix, int mode, uint64_t seed,
                                             uint8_t* codes_out, uint8_t* scales_out, void* dequant, int in_layout,
                                             int out_layout, hipStream_t stream);

// The quantizer launches of one layer, several independent ones per grid: tiled codes of any extents (see padded_cols),
// Hadamard block 32, 64 or 128.
struct RowmajorArgs {
    const void* x;
    int dtype;
    int64_t rows, cols;   // cols % hd == 0
    SignBits signs;
    uint8_t* codes;
    uint8_t* scales;
    uint8_t* maskbits;
};
struct RequantArgs {
    const uint8_t* codes_in;
    const uint8_t* scales_in;
    int64_t R, C;         // R % hd == 0, C % 32 == 0
    int val_dtype;
    uint64_t seed;
    uint8_t* codes;
    uint8_t* scales;
};
// forward quantizers (quest RTN + clip mask) of x and, unless w is null, of the weight
hipError_t quantize_layer_forward(const RowmajorArgs& x, const RowmajorArgs* w, int hd, hipStream_t stream);
struct ErrorArgs {        // e [T, O], quantized along its rows and, transposed, along T
    const void* e;
    int dtype;
    int64_t T, O;
    uint64_t seed_rows, seed_transposed;
    uint8_t* codes_rows;
    uint8_t* scales_rows;
    uint8_t* codes_transposed;
    uint8_t* scales_transposed;
};
// backward: absmax quantizer of e along its rows and of its transpose, and the transposed, re-quantized packed x and W, in one
// grid.  seed_base: null, or device memory holding a value the kernels add to every seed when they run.
hipError_t quantize_layer_backward(const ErrorArgs& e, int hd, const SignBits& signs, int mode, const RequantArgs& x, const RequantArgs& w,
                                   const uint64_t* seed_base, hipStream_t stream);
// Packed quest-coded tensors [R, C] (padded tiled codes; R and C multiples of 32) as operands of products that contract
// over R (expand.hip): E3M2 or E5M2 values in padded_rows(C) * padded_cols(R) bytes, E8M0 scales [C][padded_cols(R) / 32], and
// one byte per 128 x 128 block, [ceil(C / 128)][padded_cols(R) / 128], nonzero where the block has a value that its format cannot hold
struct E5m2Args {
    const uint8_t* codes_in;
    const uint8_t* scales_in;
    int64_t R, C;
    uint8_t* values;
    uint8_t* scales;
    uint8_t* lost;
    uint8_t* wide;   // [ceil(C / kWideStrip)][blocks of four K steps]: nonzero where the block is in eight bits; null: all of it is
};
constexpr int kWideStrip = 256, kMaxSixBlocks = 2048;
// Contractions that may be in six bits: whole blocks of four steps, of which padding is an eighth at most, and flags that fit
// beside the ring
inline bool six_bits_serve(int64_t K) {
    const int64_t steps = K / 128, blocks = (steps + 3) / 4;
    return steps >= 4 && (4 * blocks - steps) * 8 <= steps && blocks <= kMaxSixBlocks;
}
inline int64_t six_bit_flags(int64_t R, int64_t C) { return (C + kWideStrip - 1) / kWideStrip * (((R + 127) / 128 + 3) / 4); }
// both quantizations of the error signal, and the formats of the operands that their products take (E5m2Args::wide)
hipError_t quantize_error(const ErrorArgs& e, int hd, const SignBits& signs, int mode, const E5m2Args& x, const E5m2Args& w, hipStream_t stream);
hipError_t expand_e5m2_pair(const E5m2Args& a, const E5m2Args& b, hipStream_t stream);
// The columns of a product that such a loss touches, once more and from the packed tensors: c = the masked inverse rotation of
// bf16(alpha * A B), A [M, K] tiled codes, B the packed [R, C] tensor behind `b`.  Two products in one launch, which ends at
// once where nothing was lost.
struct E5m2Exact {
    const uint8_t* a_codes;
    const uint8_t* a_scales;
    E5m2Args b;
    int64_t M;
    float alpha;
    const uint8_t* mask;
    int hd;
    SignBits signs;
    float rot_c;
    void* c;
    int out_dtype;
};
hipError_t e5m2_exact_pair(const E5m2Exact& a, const E5m2Exact& b, hipStream_t stream);
hipError_t masked_hadamard_bwd_hd32_pair(const void* ga, int64_t na, int scale_dtype_a, uint32_t sign_a, const uint8_t* mask_a, void* out_a,
                                         const void* gb, int64_t nb, int scale_dtype_b, uint32_t sign_b, const uint8_t* mask_b, void* out_b,
                                         int dtype, int out_dtype_b, hipStream_t stream);

// Producers fused into the forward quantizer (Hadamard block 32, quest RTN, clip mask) and their backward passes
hipError_t rmsnorm_quantize_hd32(const void* x, int dtype, const void* add, int add_dtype, void* xsum, const float* gain, float eps,
                                 int64_t rows, int64_t cols, uint32_t sign_word, uint8_t* codes, uint8_t* scales, uint8_t* maskbits,
                                 float* factor, bool tiled, const RowmajorArgs* weight, hipStream_t stream);
hipError_t swiglu_quantize_hd32(const void* h12, int dtype, int64_t rows, int64_t hidden, uint32_t sign_word,
                                uint8_t* codes, uint8_t* scales, uint8_t* maskbits, bool tiled, const RowmajorArgs* weight, hipStream_t stream);
// weight: null, or the layer's weight (Hadamard block 32), quantized in the same grid; for tiled codes of these dtypes
bool producer_takes_weight(int dtype, int add_dtype, int w_dtype);   // no summand: BF16
bool swiglu_takes_weight(int dtype, int w_dtype);
// measurement and test aid: the SwiGLU producer's bf16 silu of all 65536 bit patterns
hipError_t silu_of_bf16_table(uint16_t* out, hipStream_t stream);
size_t rmsnorm_backward_workspace_bytes(int64_t rows, int64_t cols);
hipError_t rmsnorm_backward(const void* gy, int gy_dtype, const void* x, int x_dtype, const float* gain,
                            const float* factor, int64_t rows, int64_t cols, const uint8_t* maskbits, uint32_t sign_word,
                            int scale_dtype, const void* skip, void* dx, void* dx_bf16, float* dgain, void* workspace,
                            hipStream_t stream);
hipError_t swiglu_backward(const void* g, int g_dtype, const void* h12, int dtype, int64_t rows, int64_t hidden,
                           const uint8_t* maskbits, uint32_t sign_word, int scale_dtype, void* d_h12, hipStream_t stream);

// Rotary embedding of the fused attention projection: split + rotate, and the merge + inverse rotation of its backward
hipError_t rope_split_qkv(const void* qkv, int qkv_dtype, int64_t rows, int seq_len, int C, int head_dim, const float* table,
                          void* q, void* k, void* v, int out_dtype, hipStream_t stream);
hipError_t rope_merge_qkv_grad(const void* dq, const void* dk, const void* dv, int grad_dtype, int64_t rows, int seq_len, int C,
                               int head_dim, const float* table, void* d_qkv, int out_dtype, hipStream_t stream);

hipError_t requantize_transposed_mxfp4(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C,
                                       float post, int val_dtype, int hd, const SignBits& sb, int mode, const float* u,
                                       uint64_t seed, uint8_t* codes_out, uint8_t* scales_out, void* dequant,
                                       int in_layout, int out_layout, hipStream_t stream);

hipError_t gemm_mxfp4_tn(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                         const uint8_t* b_scales, int64_t M, int64_t N, int64_t K, float alpha, void* c, int c_dtype,
                         int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t stream);
// the reduction of a product cut into K ranges with that rotation applied to the reduced values (hadamard_bwd.hip)
hipError_t splitk_reduce_rotated(const float* partial, int splits, int64_t mn, float alpha, int mid_dtype, const uint8_t* maskbits,
                                 int hd, const SignBits& signs, float c, void* out, int out_dtype, hipStream_t stream);
size_t gemm_workspace_bytes(int64_t M, int64_t N, int64_t K);
// the part of it that the ranges filling the persistent kernel's CUs ask for (0: whole tiles already do, or K is short)
size_t gemm_few_tiles_bytes(int64_t M, int64_t N, int64_t K);
size_t gemm_e5m2_workspace_bytes(int64_t M, int64_t N, int64_t K);   // the same for a product with an eight-bit B

// The product on small and middle-sized tiles (gemm_tile.hip).  Any M; N % 8 == 0; K % 128 == 0, or K % 128 == 64 with
// row-major operands; c 16-byte aligned.  A tiled operand's last block of 16 rows exists in memory whatever its row count.
// mask: null, or the clip-mask bits [M, N / 8] of the masked inverse Hadamard rotation (block hd in {32, 64, 128} along N,
// N % hd == 0, column signs, factor rot_c) that is then applied to the bf16-rounded product; out_f32 stores its bf16
// result widened to fp32.  bf16 c_dtype only.
struct TileProduct {
    const uint8_t* a_codes;
    const uint8_t* a_scales;
    const uint8_t* b_codes;
    const uint8_t* b_scales;
    void* c;
    const uint8_t* mask;
    int M, N, K;
    int splits;            // K ranges; more than one: c receives [splits][M][N] fp32 partial sums, unscaled (fp32 c_dtype, no mask)
    int a_tiled, b_tiled;
    float alpha;
    int hd;
    SignBits signs;
    float rot_c;
    int out_f32;
    int b_e5m2;            // B holds values from expand_e5m2_pair (N % 32 == 0, K % 128 == 0, tiled A)
    const uint8_t* b_wide; // its formats (E5m2Args::wide), or null: eight bits everywhere
};
// What a product in an evaluated model is for (gemm_tile.hip).  SwiGLU: B's rows are (up, gate), c receives the tiled codes of
// Q(silu(up) * gate), quest RTN over Hadamard blocks of 32, [M, N / 2] padded, scales its scale bytes; no clip mask.  RoPE: N is 3 width, c is not used.
struct TileAfter {
    uint8_t* scales;
    uint32_t sign_word;
    float c;
    void* q;
    void* k;
    void* v;
    const float* table;   // [seq_len, head_dim / 2, 2]
    int seq_len, width, head_dim;
};
bool gemm_tile_after_serves(const TileProduct& g);
hipError_t gemm_tile_swiglu(const TileProduct& g, const TileAfter& after, hipStream_t stream);
hipError_t gemm_tile_rope(const TileProduct& g, const TileAfter& after, hipStream_t stream);
// the kinds of an eight-bit B are WIDE_256x256 and 1 .. 3
constexpr int kShortTallSteps = 8;   // see gemm_tile()
enum TileKind : int { TILE_256x128 = 0, WIDE_256x256 = 0, TILE_128x128 = 1, TILE_128x64 = 2, TILE_64x64 = 3, TILE_64x32 = 4 };
bool gemm_tile_serves(int64_t M, int64_t N, int64_t K, int a_tiled, int b_tiled, const void* c);
hipError_t gemm_tile(int kind, const TileProduct& g, int c_dtype, hipStream_t stream);
bool gemm_tile_deep(const TileProduct& g);   // TILE_128x128 with a fourth stage
// two products (bf16 results, or with a mask and *_f32 widened ones) in one grid; TileKinds 128x128 and 64x64
bool gemm_tile_pair_serves(const TileProduct& a, int kind_a, const TileProduct& b, int kind_b);
hipError_t gemm_tile_pair(TileProduct a, int kind_a, bool a_f32, TileProduct b, int kind_b, bool b_f32, hipStream_t stream);
// the gradient products of the error-only scheme in one grid (both WIDE_256x256, rotated, without K ranges)
bool gemm_wide_pair_serves(const TileProduct& a, const TileProduct& b);
hipError_t gemm_wide_pair(TileProduct a, bool a_f32, TileProduct b, bool b_f32, hipStream_t stream);

// Plain bf16 results of tiled operands on 256 x 192 tiles, two workgroups to a CU (gemm_two.hip): K % 128 == 0, K >= 512, N % 8 == 0, c 16-byte aligned
bool gemm_two_serves(const TileProduct& p);
hipError_t gemm_two(const TileProduct& p, hipStream_t stream);

// The logits of an evaluated model on the same tiles, bf16 [T, V], and for its loss per row and 96 columns the largest one and the sum of exponentials
// relative to it, float2 parts [gemm_logits_segments(V)][T]; x and w bf16 in blocks [rows / 16][K / 32][16][64 bytes]
bool gemm_logits_serves(int64_t T, int64_t V, int64_t K);
int64_t gemm_logits_segments(int64_t V);
hipError_t gemm_logits(const void* x, const void* w, int64_t T, int64_t V, int64_t K, void* logits, void* parts, hipStream_t stream);
hipError_t bf16_blocks(const float* w, int64_t V, int64_t K, void* out, hipStream_t stream);   // fp32 rows into such blocks (lm_head.hip)
hipError_t logits_loss_rows(const void* parts, int64_t segments, int64_t T, const void* logits, int64_t V, const int64_t* targets, int64_t ignore, float* losses,
                            hipStream_t stream);

// The product of at most 64 rows with a weight, both tiled (gemm_rows.hip): K % 128 == 0, N % 8 == 0, c 16-byte aligned, no mask, scales 4-byte aligned and,
// for K < 512, behind their codes as in a packed operand (scale_requests.h).
// Its sums are in another order than the other kernels'.
bool gemm_rows_serves(const TileProduct& p);
hipError_t gemm_rows(const TileProduct& p, int c_dtype, hipStream_t stream);

// The forward pass of a layer for a decoded batch in one launch (gemm_rows.hip): quest RTN of x under Hadamard blocks of 32, times
// the packed weight (padded tiled codes, the scales behind them as above); x 16-byte, y 8-byte aligned
bool linear_decode_serves(int64_t T, int64_t I, int64_t O);
hipError_t linear_decode(const void* x, int x_dtype, int64_t T, int64_t I, int64_t O, uint32_t sign_word, const uint8_t* w_codes,
                         const uint8_t* w_scales, void* y, int y_dtype, hipStream_t stream);

// The kernel a product runs on (gemm.hip).  Products with p.mask set ask for the masked inverse rotation; `rotates` tells
// whether that kernel applies it (p.c then holds rot_out_dtype elements: c_dtype, or F32 holding the bf16-rounded result)
// or the caller has to (p.c then holds the plain product in c_dtype).
struct ProductChoice {
    enum Path : int { GENERIC = 0, PERSISTENT = 1, TILE = 2, TWO = 3 } path;
    int kind;      // TileKind
    int splits;    // K ranges (their fp32 partial sums in the workspace, then one ordered reduction)
    bool rotates;
    double cost = 0.0;   // the estimate, in microseconds, a rotation in a pass of its own included
};
TileProduct make_product(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales, int64_t M, int64_t N,
                         int64_t K, float alpha, void* c, int a_layout, int b_layout);
ProductChoice choose_product(const TileProduct& p, int c_dtype, int rot_out_dtype, const void* workspace, size_t workspace_bytes);
bool product_after_pays(const TileProduct& p, double end, double pass);   // see TileAfter
hipError_t run_product(const ProductChoice& c, const TileProduct& p, int c_dtype, int rot_out_dtype, void* workspace, hipStream_t stream);
// The gradient products x and w of a layer in one launch: of which kernel, if that is expected to be faster than running them as cx
// and cw say; p.mask and *_out as in choose_product.  The results are those of the kernel without K ranges.
struct PairChoice {
    enum Path : int { SEPARATE = 0, PERSISTENT = 1, TILE = 2 } path;
    int kind_x, kind_w;   // TileKinds
};
PairChoice choose_pair(const TileProduct& x, const ProductChoice& cx, int x_out, const TileProduct& w, const ProductChoice& cw, int w_out);
// whether that launch takes these products: one of them with its rotation at least
bool pair_serves(const PairChoice& c, const TileProduct& x, int x_out, const TileProduct& w, int w_out);
hipError_t run_pair(const PairChoice& c, const TileProduct& x, int x_out, const TileProduct& w, int w_out, hipStream_t stream);
// the rotation in the persistent kernel's bf16 epilogue (Hadamard block 32)
bool gemm_persistent_rotates(const uint8_t* a_scales, const uint8_t* b_scales, int64_t M, int64_t N, int64_t K);
hipError_t gemm_persistent_rotated(TileProduct p, hipStream_t stream);
// C = alpha * A (packed MXFP4 [M, K]) x B (bf16 [K, N] row-major): K % 64 == 0, N % 8 == 0
bool gemm_fp4_bf16_nn_supported(int64_t M, int64_t N, int64_t K);
hipError_t gemm_fp4_bf16_nn(const uint8_t* a_codes, const uint8_t* a_scales, const void* b, int64_t M, int64_t N, int64_t K,
                            float alpha, void* c, int c_dtype, hipStream_t stream);
// measurement aid: one launch of the persistent kernel that records the shader clock around every tile's K loop and epilogue
int gemm_phase_stamps_per_group();
hipError_t gemm_tile_phases(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                            int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_layout, int b_layout,
                            const uint8_t* rot_mask, unsigned long long* stamps, size_t stamps_bytes, int* grid_out, hipStream_t stream);
// measurement aid: the FP4 matrix instruction alone (see gemm.hip)
int mfma_only_blocks();
hipError_t mfma_only(const uint8_t* operands, float* sink, int iters, hipStream_t stream);

// RMSNorm of (x + add) (norm.hip): fp32 x, add null, bf16 or fp32, out bf16 or fp32; cols % 4 == 0, cols <= 4096
hipError_t rmsnorm_rows(const float* x, const void* add, int add_dtype, const float* gain, float eps, int64_t rows, int64_t cols, void* out, int out_dtype,
                        hipStream_t stream, bool blocks = false);

// mean cross-entropy over the rows whose target is not `ignore` (loss.hip); losses: scratch, one float per row
hipError_t loss_mean(const float* losses, const int64_t* targets, int64_t rows, int64_t ignore, float* loss, hipStream_t stream);   // of the rows not ignored
hipError_t cross_entropy_mean(const void* logits, int dtype, const int64_t* targets, int64_t rows, int64_t classes, int64_t ignore,
                              float* losses, float* loss, hipStream_t stream);

hipError_t masked_hadamard_bwd(const void* g, int g_dtype, int64_t rows, int64_t cols, int hd, int scale_dtype,
                               const SignBits& sb, const uint8_t* maskbits, void* out, int out_dtype,
                               bool round_to_g_dtype, hipStream_t stream);

hipError_t dequantize_mxfp4(const uint8_t* codes, const uint8_t* scales, int64_t R, int64_t C, float post, void* out,
                            int out_dtype, hipStream_t stream);

}  // namespace qm
