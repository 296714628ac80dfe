// Host-side launcher of the single-token time-mixer step (internal; public surface is include/wind_rwkv7.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace wkv {

// The block's parameters (names as in time_mixer.py:42-104), bf16 device arrays except ln_params.
struct MixerWeights {
    const void *time_maa_x, *time_maa, *time_maa_w1, *time_maa_w2;            // [C], [4,C], [128,C], [4,C,32]
    const void *Wr, *Wk, *Wv, *Wo;                                            // [C,C]
    const void *gate_w1, *time_decay_w1, *time_kkk_w1, *mk_w1, *time_aaa_w1, *ma_w1;   // [rank,C]
    const void *gate_w2, *time_decay_w2, *time_kkk_w2, *mk_w2, *time_aaa_w2, *ma_w2;   // [C,rank]
    const void *time_decay, *time_aaaaa, *time_misc_a, *time_misc_k;          // [C]
    const void* ln_params;                                                    // [3,C] fp32: GroupNorm weight, bias, bonus
};

size_t mixer_decode_workspace_bytes(int B, int C);
// x [B,T,C] bf16; x_prev null or [B,C] bf16, the token before; state_in null or, and state, [B,H,64,64] (bf16 or fp32; may be
// the same); y [B,T,C] bf16; x_carry: null or [B,C] bf16 that receives the last tokens (the next call's x_prev; must not
// alias x_prev).  workspace: mixer_decode_workspace_bytes(B*T, C).
void launch_mixer_decode(int B, int T, int C, int H, int state_f32, const MixerWeights& w, const void* x, const void* x_prev,
                         const void* state_in, void* state, void* y, void* x_carry, void* workspace, hipStream_t stream);

// WKV7 with the GroupNorm + bonus + gate epilogue, token by token on a state in fp32 registers: n tokens from `first` on of
// q, v, a, g and y [B,T,H*64]; of w, k, b [B,wkb_T,H*64] the n from wkb_first on.  State as above.  epilogue not null (the tokens are in
// the last chunk of T, a multiple of 16): in the same launch also the attn_ln epilogue of the chunks before, from their kept output.
struct KeptOutput {
    const void* y_wkv;      // [B,T,H*64], centred with `centers` (see Centred in ln_epilogue.hpp)
    const float* centers;
    const void* k;          // [B,T,H*64]
};
void launch_tokens(int B, int T, int H, int first, int n, int wkb_T, int wkb_first, int state_f32, const void* w, const void* q, const void* k,
                   const void* v, const void* a, const void* b, const void* g, const void* params, const void* state_in, void* state,
                   void* y, hipStream_t stream, const KeptOutput* epilogue = nullptr);

}  // namespace wkv
