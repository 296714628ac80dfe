// Host-side launcher of the projection weight-gradient kernel (internal; public surface is include/wind_rwkv7.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace wkv {

// How a [tokens] x (O, I) problem is cut: tile shape (index into the kernel's table), ntn tiles across the
// narrower dimension, ntiles in all, ksplit token ranges; swap = the input channels take the wider side.
struct WgradPlan {
    int shape, ntn, ntiles, ksplit;
    bool swap;
    size_t partial_bytes;
};
WgradPlan linear_wgrad_plan(long tokens, int O, int I);
// dW[o][i] = sum_t dy[t][o] x[t][i];  dy [tokens, O] (row stride ld_dy), x [tokens, I] (row stride ld_x), bf16;
// dW [O, I] contiguous, fp32 or bf16, overwritten.  O, I multiples of 16; strides multiples of 8 elements.
void launch_linear_wgrad(long tokens, int O, int I, const void* dy, long ld_dy, const void* x, long ld_x, void* dW,
                         bool out_f32, void* workspace, hipStream_t stream);

// Up to nine problems with the same token count, each with the tile shape that suits it: one launch for the products
// and one for the sums of the partial tiles.  Returns false (nothing launched) for n outside 1 .. 9 or no tokens;
// workspace bytes 0 likewise.
size_t linear_wgrad_group_workspace_bytes(int n, long tokens, const int* O, const int* I);
bool launch_linear_wgrad_group(int n, long tokens, const int* O, const int* I, const void* const* dy, const long* ld_dy,
                               const void* const* x, const long* ld_x, void* const* dW, bool out_f32, void* workspace,
                               hipStream_t stream);
// The same, or the first problem in launches of its own ahead of the others, whichever is the faster.
size_t block_wgrads_workspace_bytes(int n, long tokens, const int* O, const int* I);
bool launch_block_wgrads(int n, long tokens, const int* O, const int* I, const void* const* dy, const long* ld_dy,
                         const void* const* x, const long* ld_x, void* const* dW, bool out_f32, void* workspace, hipStream_t stream);

// Column blocks of token-major bf16 matrices (csrc/cols.hip): piece = `width` columns (a multiple of 8) of M rows
// from (src, src_ld, src_col0) to (dst, dst_ld, dst_col0); offsets and strides multiples of 8 elements.
enum { COLS_COPY = 0, COLS_TANH = 1, COLS_TANH_GRAD = 2 };   // TANH_GRAD: src * (1 - aux^2), aux [M, width] contiguous
constexpr int COLS_MAX_PIECES = 8;   // per launch; longer lists take several
struct ColumnPiece {
    const void* src;   // null: zeros
    const void* aux;
    void* dst;
    long long src_ld, dst_ld;
    int src_col0, dst_col0, width, op;
};
void launch_copy_columns(long long M, int n, const ColumnPiece* pieces, hipStream_t stream);

// bf16 copies of n tensors (float32 or bf16, contiguous, numel[t] elements each) written to element offsets
// dst_offset[t] of dst (null: back to back)
constexpr int CAST_MAX_TENSORS = 32;   // per launch; longer lists take several
void launch_cast_to_bf16(int n, const void* const* src, const int* src_f32, const long long* numel,
                         const long long* dst_offset, void* dst, hipStream_t stream);

// x [B,T,C] to out [B,T_out,C]: the first T tokens, zeros behind them; last (may be null) [B,C]: token T - 1, if out has it
struct PadRows {
    int B, T, T_out, C;   // B = 0: nothing to pad
    const void* x;
    void *out, *last;
};
void launch_pad_rows(const PadRows& p, hipStream_t stream);
// rows first .. T-1 of w, k, b [B, T, C] (bf16): decay 1, k = b = 0; kept (may be null) [3, B, T-first, C]: what they were
void launch_neutral_rows(int B, int T, int C, int first, void* w, void* k, void* b, void* kept, hipStream_t stream);

// dst [rows, cols] (bf16, or f32 where dst_f32) from src (f32 or bf16); dstT: null or the transposed bf16 copy, row stride ldT
struct PackTensor {
    const void* src;
    void *dst, *dstT;
    int rows, cols;
    long ldT;
    int src_f32, dst_f32, src_aligned;   // src_aligned: to 16 bytes
};
constexpr int PACK_MAX_TENSORS = 32;
void launch_pack_weights(int n, const PackTensor* tensors, const PadRows& pad, hipStream_t stream);   // pad: in the same launch

// D[m][n] = sum_k A0[m][k] W0[n][k] (+ sum_k A1[m][k] W1[n][k]); see linear_group.hip.  K[1] = 0: one segment.  The columns
// start[t] .. start[t] + width[t] - 1 go to out[t] (row stride ld_out[t]); aux[t]: [M, width[t]].
enum { LINEAR_PLAIN = 0, LINEAR_TANH = 1, LINEAR_TANH_GRAD = 2 };
struct LinearProblem {
    static constexpr int PIECES = 4;
    const __bf16* A[2];
    const __bf16* W[2];
    long lda[2], ldw[2];
    int K[2];
    int N, npieces;
    __bf16* out[PIECES];
    const __bf16* aux[PIECES];
    long ld_out[PIECES];
    int start[PIECES], width[PIECES], op[PIECES];
};
constexpr int LINEAR_GROUP_MAX = 9;   // problems of a launch
void launch_linear_group(int n, long M, const LinearProblem* problems, hipStream_t stream);

}  // namespace wkv
