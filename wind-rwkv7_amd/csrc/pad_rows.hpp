// Rows padded to whole chunks (launch_pad_rows), for a launch of their own and for the one that packs the weights.
#pragma once
#include "frag.hpp"
#include "linear_kernels.hpp"

namespace wkv {

struct PadArgs {
    const __bf16* x;
    __bf16 *out, *last;
    int T, T_out, C;
    unsigned blocks;   // of 256 threads, eight channels each
    long vectors;
    explicit PadArgs(const PadRows& p)
        : x(static_cast<const __bf16*>(p.x)), out(static_cast<__bf16*>(p.out)), last(static_cast<__bf16*>(p.last)), T(p.T), T_out(p.T_out), C(p.C),
          blocks((unsigned)(((long)p.B * p.T_out * (p.C / 8) + 255) / 256)), vectors((long)p.B * p.T_out * (p.C / 8)) {}
};
__device__ __forceinline__ void pad_rows_block(const PadArgs& p, unsigned block) {
    const long v = (long)block * 256 + threadIdx.x;
    if (v >= p.vectors) return;
    const int per_row = p.C / 8, col = (int)(v % per_row) * 8;
    const long row = v / per_row, b = row / p.T_out;
    const int t = (int)(row - b * p.T_out);
    bf16x8 r = {};
    if (t < p.T) r = *reinterpret_cast<const bf16x8*>(p.x + (b * p.T + t) * p.C + col);
    store_through(p.out + row * p.C + col, r);
    if (p.last != nullptr && t == p.T - 1) *reinterpret_cast<bf16x8*>(p.last + b * p.C + col) = r;
}

}  // namespace wkv
