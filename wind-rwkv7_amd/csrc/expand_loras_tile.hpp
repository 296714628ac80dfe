// What the expand_loras kernels of both files share: operands, activations, fragments.
#pragma once
#include "row_lines.hpp"
#include "expand_loras_kernels.hpp"

namespace wkv {

constexpr int LORA_TOK = 16;

struct LoraIn {   // the four [M, D] activations
    const __bf16* p[4];   // z, a, ma, mk
};
struct LoraW {    // the four [C, D] matrices and four [C] biases
    const __bf16* W[4];   // Wz, Wa, Wma, Wmk
    const __bf16* bias[4];  // w_bias, a_bias, ma_bias, mk_bias
};

struct LoraDy {
    const __bf16* p[4];   // dw_out, dk_out, dkk_out, db_out
};
struct LoraDIn {
    __bf16* p[4];         // per-head partials of dz_in, da_in, dma_in, dmk_in: [M, H, D]
};

struct LoraReduceOut {   // d*_in [M, D] with row strides ld, dW [C, D], dbias [C]
    __bf16* din[4];
    long ld[4];
    float* dW[4];
    float* db[4];
};
// What the normalisation needs of a (token, head) when the head is not the 64 channels a wavefront holds: written
// by expand_loras_head_kernel, read by the backward kernels in place of their own sums.
struct HeadStat {
    float inorm;   // 1 / sqrt(max(sum_head z^2, 1e-12))
    float proj;    // (sum_head dkk z) inorm^3, or 0 where the norm is clamped
};

// v_rcp_f32 (1 ulp) instead of an IEEE division: the division expands to ten instructions per element
__device__ __forceinline__ float sigmoidf_(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
// log(1 + exp(-|u|)): the argument of the logarithm lies in [1, 2], so the bare v_log_f32 needs none of the
// denormal handling that __logf wraps around it (four instructions per element)
__device__ __forceinline__ float log1pexp_(float u) {
    return 0.6931471805599453f * __builtin_amdgcn_logf(1.f + __expf(-fabsf(u)));
}
__device__ __forceinline__ float tanhf_(float x) {
    const float e = __expf(2.f * fminf(x, 40.f));
    return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

template <int ND>
struct Frags {
    bf16x4 f[ND];
};
// F(in[16 tokens, D])  lane = token, reg = rank index
template <int ND>
__device__ __forceinline__ Frags<ND> load_act(const __bf16* __restrict__ p, long m0, const Lane& L) {
    Frags<ND> r;
    const __bf16* row = p + (m0 + L.n) * (16 * ND) + 4 * L.g;
#pragma unroll
    for (int j = 0; j < ND; j++) r.f[j] = *reinterpret_cast<const bf16x4*>(row + 16 * j);
    return r;
}
// F(W[c0+16cb .. , D])  lane = channel, reg = rank index
template <int ND>
__device__ __forceinline__ Frags<ND> load_w(const __bf16* __restrict__ W, int c, const Lane& L) {
    Frags<ND> r;
    const __bf16* row = W + (long)(c + L.n) * (16 * ND) + 4 * L.g;
#pragma unroll
    for (int j = 0; j < ND; j++) r.f[j] = *reinterpret_cast<const bf16x4*>(row + 16 * j);
    return r;
}
// acc + F(in W^T) for one block of 16 channels  (lane = token, reg = channel)
template <int ND>
__device__ __forceinline__ f32x4 lora_block(f32x4 acc, const Frags<ND>& w, const Frags<ND>& in) {
    if constexpr (ND == 1) {
        acc = mma(acc, w.f[0], in.f[0]);
    } else {
#pragma unroll
        for (int j = 0; j < ND; j += 2) acc = mma2(acc, w.f[j], w.f[j + 1], in.f[j], in.f[j + 1]);
    }
    return acc;
}
__device__ __forceinline__ f32x4 load_bias(const __bf16* __restrict__ b, int c, const Lane& L) {
    return to_f32(*reinterpret_cast<const bf16x4*>(b + c + 4 * L.g));
}

// the rank-16 kernels (expand_loras16.hip); forward: heads of 64 channels; splits: blocks of the backward kernel per head
int lora16_splits(long M, int H);
void launch_loras16_forward(long M, int C, const __bf16* w_in, const __bf16* k_in, const LoraIn& in, const LoraW& lw, __bf16* const outs[4],
                            hipStream_t stream, int padded_T = 0, void* kept = nullptr);
// din: the heads' shares of the four d*_in, [M, H, 2, 16 / 4, 2, 4]: rank index 4g + r of i = 2 half + e at [half][g][e][r].
// stats not null: the norm of each (token, head of HS channels) is read instead of summed over 64 channels
void launch_loras16_backward(long M, int C, const __bf16* w_in, const __bf16* k_in, const LoraIn& in, const LoraW& lw, const LoraDy& dy,
                             __bf16* dw_in, __bf16* dk_in, __bf16* din, float* partial, int nsplit, const HeadStat* stats, int HS,
                             hipStream_t stream);
void launch_loras16_reduce(long M, int C, int nsplit, const __bf16* din, const float* partial, const LoraReduceOut& out, hipStream_t stream);

}  // namespace wkv
