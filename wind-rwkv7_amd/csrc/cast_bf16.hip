// Many tensors to bf16 in one launch: the bf16 working copies of a block's projection weights.
//
// The reference casts each weight on its own before every matmul (time_mixer.py:120-131, `.to(bf16)` per
// operand).  A framework multi-tensor copy does this in chunks of 65 536 elements per block - 46 blocks for the
// 3 M weights of a 768-channel time mixer, on a chip with 256 compute units - and took 48 us per step in three
// launches.  Here a block takes 2048 elements (8 per thread, 16-byte stores), and one launch covers up to
// CAST_MAX_TENSORS tensors whose copies go to given offsets of one destination buffer (back to back, so that
// weights used together form one matrix, or padded to an alignment).
#include "linear_kernels.hpp"

#include <hip/hip_runtime.h>

#include "pad_rows.hpp"

namespace wkv {
namespace {

constexpr int UNIT = 2048;   // elements per block

struct CastArgs {
    const void* src[CAST_MAX_TENSORS];
    long long unit_begin[CAST_MAX_TENSORS + 1];   // first block of tensor t
    long long dst_off[CAST_MAX_TENSORS];          // first destination element of tensor t
    long long numel[CAST_MAX_TENSORS];
    int src_f32[CAST_MAX_TENSORS];                // 1: float32 source, 0: bf16 source (a plain copy)
    int n;
};

__global__ __launch_bounds__(256) void cast_to_bf16_kernel(CastArgs g, __bf16* __restrict__ dst) {
    const long long unit = blockIdx.x;
    int t = 0;
    while (t + 1 < g.n && unit >= g.unit_begin[t + 1]) t++;   // the same for every thread of the block
    const long long numel = g.numel[t];
    const long long local = (unit - g.unit_begin[t]) * UNIT + threadIdx.x * 8;
    if (local >= numel) return;
    __bf16* out = dst + g.dst_off[t] + local;
    const bool whole = local + 8 <= numel && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    if (g.src_f32[t]) {
        const float* in = static_cast<const float*>(g.src[t]) + local;
        if (whole && reinterpret_cast<uintptr_t>(in) % 16 == 0) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(in), hi = *reinterpret_cast<const f32x4*>(in + 4);
            const bf16x4 a = to_bf16(lo), b = to_bf16(hi);
            *reinterpret_cast<bf16x8*>(out) = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            for (int e = 0; e < 8 && local + e < numel; e++) out[e] = (__bf16)in[e];
        }
    } else {
        const __bf16* in = static_cast<const __bf16*>(g.src[t]) + local;
        if (whole && reinterpret_cast<uintptr_t>(in) % 16 == 0) {
            *reinterpret_cast<bf16x8*>(out) = *reinterpret_cast<const bf16x8*>(in);
        } else {
            for (int e = 0; e < 8 && local + e < numel; e++) out[e] = in[e];
        }
    }
}

// pack: a block takes 64 rows x 64 columns of one tensor, sixteen threads side by side on a row (four elements each, whole
// lines); where a transposed copy is wanted the tile turns in LDS and leaves as rows of the transposed matrix, eight threads on
// a line.  The block's tensor comes from comparisons with all of `first` at once (a loop over them was a scalar load each, one
// after the other).  Sixteen elements of a row per thread and the loop: 8.7, 23.2 us for the training block's weights at 768
// and 1536 channels, 7.7 for a prompt's; so 7.4, 19.4 and 6.4, where their 21, 85 and 15 MB take 4, 17 and 3.
constexpr int PT = 64;
struct PackArgs {
    PackTensor t[PACK_MAX_TENSORS];
    int first[PACK_MAX_TENSORS + 1];   // first block of tensor t; past the last tensor: no block's
    int n;
};
// The blocks behind the last tensor's pad a prompt's rows: they need nothing of the others, nor those of them (a launch of their own before this one:
// 2 x 1003 tokens x 768 channels 3.2 + 6.7 us, so 7.4).
__global__ __launch_bounds__(256) void pack_weights_kernel(const PackArgs g, const PadArgs pad) {
    __shared__ __bf16 s[PT][PT + 2];   // (pitch 33 words: columns are read across the banks)
    const int packing = gridDim.x - pad.blocks;
    if ((int)blockIdx.x >= packing) return pad_rows_block(pad, blockIdx.x - packing);   // (the whole block)
    int t = 0;
#pragma unroll
    for (int k = 1; k < PACK_MAX_TENSORS; k++) t += (int)blockIdx.x >= g.first[k] ? 1 : 0;   // the same for every thread of the block
    const PackTensor& p = g.t[t];
    const int tile = blockIdx.x - g.first[t], ntc = (p.cols + PT - 1) / PT;
    const int r0 = tile / ntc * PT, c0 = tile % ntc * PT;
    const int lr = threadIdx.x >> 4, lc = 4 * (threadIdx.x & 15), c = c0 + lc;   // rows lr + 16 i of the tile
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = r0 + lr + 16 * i;
        if (r >= p.rows || c >= p.cols) continue;
        const long at = (long)r * p.cols + c;
        if (!p.src_aligned) {   // (a parameter that is a view into a larger buffer) element by element
#pragma unroll
            for (int e = 0; e < 4; e++)
                v[i][e] = p.src_f32 ? static_cast<const float*>(p.src)[at + e] : (float)static_cast<const __bf16*>(p.src)[at + e];
        } else if (p.src_f32) {
            v[i] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.src) + at);
        } else {
            v[i] = to_f32(*reinterpret_cast<const bf16x4*>(static_cast<const __bf16*>(p.src) + at));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = r0 + lr + 16 * i;
        if (r >= p.rows || c >= p.cols) continue;
        const long at = (long)r * p.cols + c;
        if (p.dst_f32) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(p.dst) + at) = v[i];
        } else {
            const bf16x4 b = to_bf16(v[i]);
            *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(p.dst) + at) = b;
            if (p.dstT)
#pragma unroll
                for (int e = 0; e < 4; e++) s[lr + 16 * i][lc + e] = b[e];
        }
    }
    if (!p.dstT) return;
    __syncthreads();
    // rows of the transposed copy: eight source rows per thread
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int lt = (threadIdx.x >> 3) + 32 * i, tr = 8 * (threadIdx.x & 7);
        if (c0 + lt >= p.cols || r0 + tr >= p.rows) continue;
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = s[tr + e][lt];
        *reinterpret_cast<bf16x8*>(static_cast<__bf16*>(p.dstT) + (long)(c0 + lt) * p.ldT + r0 + tr) = o;
    }
}

}  // namespace

void launch_pack_weights(int n, const PackTensor* tensors, const PadRows& rows, hipStream_t stream) {
    const PadArgs pad(rows);
    PackArgs g;
    g.n = n;
    g.first[0] = 0;
    for (int t = 0; t < n; t++) {
        g.t[t] = tensors[t];
        g.first[t + 1] = g.first[t] + ((tensors[t].rows + PT - 1) / PT) * ((tensors[t].cols + PT - 1) / PT);
    }
    for (int t = n + 1; t <= PACK_MAX_TENSORS; t++) g.first[t] = 0x7fffffff;
    hipLaunchKernelGGL(pack_weights_kernel, dim3(g.first[n] + pad.blocks), dim3(256), 0, stream, g, pad);
}

void launch_cast_to_bf16(int n, const void* const* src, const int* src_f32, const long long* numel,
                         const long long* dst_offset, void* dst, hipStream_t stream) {
    long long next = 0;   // where a tensor goes when no offsets are given: right after the one before
    for (int first = 0; first < n; first += CAST_MAX_TENSORS) {
        CastArgs g;
        g.n = n - first < CAST_MAX_TENSORS ? n - first : CAST_MAX_TENSORS;
        g.unit_begin[0] = 0;
        for (int t = 0; t < g.n; t++) {
            g.src[t] = src[first + t];
            g.src_f32[t] = src_f32[first + t];
            g.numel[t] = numel[first + t];
            g.dst_off[t] = dst_offset ? dst_offset[first + t] : next;
            next += numel[first + t];
            g.unit_begin[t + 1] = g.unit_begin[t] + (numel[first + t] + UNIT - 1) / UNIT;
        }
        if (g.unit_begin[g.n] > 0)
            hipLaunchKernelGGL(cast_to_bf16_kernel, dim3((unsigned)g.unit_begin[g.n]), dim3(256), 0, stream, g,
                               static_cast<__bf16*>(dst));
    }
}

}  // namespace wkv
