// WKV7 in fp32: sequences, state, arithmetic and saved states all fp32 (no matrix cores), head sizes 16 .. 128.
//
// The accuracy mode of the path - what the reference's Triton kernels provide with dot_prec='fp32'
// (rwkv7_attn_triton.py:27-156, :182-190) - and what its large-head variant runs by default
// (rwkv7_attn_triton_bighead.py:31-322, any multiple of 16).  Results are within 1e-4 of the fp64 recurrence, where
// the bf16 kernels are within 1e-2.  It is the token-by-token recurrence itself,
//     sa = S a_t;   S <- S diag(exp(-exp(w_t))) + sa b_t^T + v_t k_t^T;   y_t = S q_t,
// with the state in registers, spread thin so that a token costs few instructions per wavefront and little LDS
// traffic: a thread holds R rows x 4 or 8 columns, LPR lanes share a row.  A block works at a width C of 64 or 128 channels (a smaller
// head is padded: channels and rows past the head size read as zero and are never written).  With 16 lanes to a row (a DPP row) a row
// sum (S a, S q, dS k, dS b) is four DPP adds, with 32 one lane swap more, with 8 three; a column sum over the row groups of a wavefront
// (S^T dy, dS^T v, ...) is three (one) of gfx950's lane swaps (col_sum4, store_col_sums), then LDS across the wavefronts.  The vectors
// of a token are read one token ahead of their use.
// The value rows of a state never mix, so a head is cut over blocks by rows (scan_split).  In the scan, four or eight
// wavefronts of a block carry the recurrence and touch LDS only; four more fetch the next chunk, turn it into operands in
// the other half of a double buffer and carry the results of the chunk before to memory, with one barrier per chunk.
// (Staging by the recurrence's own wavefronts, between barriers, was a fifth of its time: 227 -> 183 us at 8 x 1024 tokens
// x 12 heads of 64, 793 -> 388 us at 4096 tokens x 4 heads.)  Bound: vector issue (a wavefront alone on a SIMD gets an instruction in about
// every seven cycles, two of them one in four) and, with eight columns a lane, LDS reads, so:
//   * what can wait is done for many tokens at once: the row sums of S (decay q) for four (quad_sums), what the row vectors add to y
//     once per chunk by the lane that keeps a token;
//   * the moves take four channels a thread (303 -> 167 vector instructions a chunk);
//   * 8 lanes and 8 columns instead of 16 and 4 where the head is cut in two or not at all (of 128 channels 16 and 8 instead of 32 and 4):
//     half as many row sums, 822 instructions a chunk for eight rows instead of 998.  Twice the LDS reads would undo it (8 x 1024 x 12 heads of
//     64 416 -> 438 us, forward + backward), so a lane reads four of its eight columns, the lane eight away in the DPP row, which has
//     the same columns of another row, the other four, and they are operands of each other's instructions (fma_other_row).
// Forward + backward with these three and bkq as floats, us: 8 x 1024 x 12 heads of 64 419 -> 396, 24 x 1024 x 12 1154 -> 1097, 1 x 1024 x 16
// 235 -> 226, 8 x 1024 x 6 of 128 788 -> 681, 8 x 512 x 8 of 96 422 -> 363, 32 x 128 x 16 of 32 185 -> 168.
// The forward keeps the state every CHUNK tokens and S a of every token.  The backward is the same scan in the other
// direction (it keeps the state gradient arriving at every chunk's end and dsa of every token, and leaves dv and ds0)
// and then a kernel in which every chunk is on its own and makes the other five gradients.
// A caller without a workspace gets the backward in one kernel: two blocks of four wavefronts per head, the walk back in
// windows of recomputed states, and the gradients that sum over value rows added by the two blocks onto zeroed tensors
// with atomics (two addends: the order does not show).  Forward + backward, microseconds, one kernel -> two:
//   1 x 256 tokens x 4 heads of 64   172 -> 67         8 x 1024 x 6 heads of 128   2225 -> 700
//   8 x 1024 x 12 heads of 64        745 -> 388        32 x 1024 x 12 heads of 64  2215 -> 1298
#include "wkv7_f32_kernels.hpp"

#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_info.hpp"

namespace wkv {
namespace {

// a barrier that orders LDS only: loads and stores to memory stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float seq4 __attribute__((ext_vector_type(4), aligned(4)));   // four of a sequence's channels, whose address is a float's

// gfx950's lane-swap instructions, one swap and one add for two values at once: v_permlane32_swap exchanges lanes
// 32-63 of its first register with lanes 0-31 of its second, so with X and Y two values to be summed over the lane
// pairs (l, l + 32), X' + Y' is X summed over the pair in lanes 0-31 and Y summed over the pair in lanes 32-63;
// v_permlane16_swap does the same between neighbouring rows of 16 lanes (even rows keep X, odd rows Y).
__device__ __forceinline__ float swap_add32(float x, float y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap_add16(float x, float y) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// index of element (token t, head h, channel c) of a [B,T,H,C] tensor, b folded into t
__device__ __forceinline__ long seq_index(long bt, int H, int h, int c, int C) { return (bt * H + h) * C + c; }

enum { V_DEC = 0, V_Q, V_K, V_V, V_A, V_B, FWD_VECS };
enum { W_DEC = 0, W_Q, W_K, W_V, W_A, W_B, W_DY, W_DDEC, BWD_VECS };   // W_DDEC: d(decay)/dw = -exp(w) decay
enum { R_DQ = 0, R_DK, R_DB, R_DA, R_DW, RED_VECS };

constexpr int CH64 = WKV7_F32_CHUNK;   // tokens between saved states

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// sum over the 16 lanes of a DPP row, result in all of them (every step adds two values that both lanes hold, so the
// 16 results are the same bits)
__device__ __forceinline__ float row_sum16(float x) {
    x += dpp<0xB1>(x);     // quad_perm [1,0,3,2]
    x += dpp<0x4E>(x);     // quad_perm [2,3,0,1]
    x += dpp<0x141>(x);    // row_half_mirror
    x += dpp<0x140>(x);    // row_mirror
    return x;
}
__device__ __forceinline__ float dot4(f4 x, f4 y) { return ((x[0] * y[0] + x[1] * y[1]) + x[2] * y[2]) + x[3] * y[3]; }
// p: this thread's terms for columns 4 jb .. 4 jb + 3.  Returns the sum over the wavefront's four row groups of column
// 4 jb + ib: lanes 0-31 keep columns 0 and 1, lanes 32-63 columns 2 and 3; then even rows of 16 lanes keep the lower
// of their two, odd rows the upper.
__device__ __forceinline__ float col_sum4(f4 p) {
    const float lo = swap_add32(p[0], p[2]), hi = swap_add32(p[1], p[3]);
    return swap_add16(lo, hi);
}
template <int R>
struct RowVals {
    float x[R];
};
template <int R>
__device__ __forceinline__ RowVals<R> lds_rows(const float* p) {
    RowVals<R> r;
    if constexpr (R % 4 == 0) {
#pragma unroll
        for (int i = 0; i < R / 4; i++) {
            const f4 v = *reinterpret_cast<const f4*>(p + 4 * i);
            r.x[4 * i] = v[0], r.x[4 * i + 1] = v[1], r.x[4 * i + 2] = v[2], r.x[4 * i + 3] = v[3];
        }
    } else if constexpr (R == 2) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        const f2 v = *reinterpret_cast<const f2*>(p);
        r.x[0] = v[0], r.x[1] = v[1];
    } else {
        r.x[0] = *p;
    }
    return r;
}

// element at a 32-bit byte offset from a base that is the same in every lane (scalar base, one register per lane)
template <class V>
__device__ __forceinline__ const V& at_bytes(const float* p, unsigned o) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + o);
}
template <class V>
__device__ __forceinline__ V& at_bytes(float* p, unsigned o) {
    return *reinterpret_cast<V*>(reinterpret_cast<char*>(p) + o);
}

// the value of the lane eight away in a DPP row (row_ror 8), as an operand of the instruction that uses it
__device__ __forceinline__ float other_row(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, true));
}

// acc + other_row(x) y (the compiler does not make a multiply-add of such an operand)
__device__ __forceinline__ float fma_other_row(float x, float y, float acc) {
    asm("v_fmac_f32_dpp %0, %1, %2 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(y));
    return acc;
}

// sum over the LPR lanes that share a state row (16: a DPP row; 32: two neighbouring DPP rows), result in all of them
template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
    if constexpr (LPR == 8) {
        x += dpp<0xB1>(x);     // quad_perm [1,0,3,2]
        x += dpp<0x4E>(x);     // quad_perm [2,3,0,1]
        return x + dpp<0x141>(x);   // row_half_mirror
    }
    x = row_sum16(x);
    if constexpr (LPR == 32) x = swap_add16(x, x);   // both operands the same: every lane gets this row plus its neighbour
    return x;
}
// Column sums over the row groups of a wavefront, stored for the cross-wavefront sum.  p: this thread's terms for
// columns col0 .. col0 + 3; to: the 4 LPR columns of one token and gradient in LDS.  16 lanes per row (four row groups):
// the lane of group ib ends up with column col0 + ib; 32 lanes per row (two groups): with columns col0 + 2 ib, + 1.
template <int LPR>
__device__ __forceinline__ void store_col_sums(float* to, f4 p, int col0, int ib) {
    if constexpr (LPR == 16) {
        to[col0 + ib] = col_sum4(p);
    } else {
        typedef float f2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<f2*>(to + col0 + 2 * ib) = f2{swap_add32(p[0], p[2]), swap_add32(p[1], p[3])};
    }
}

// Several values at once summed over lanes, each lane ending up with ONE of the sums: a halving of the values is a select of
// what a lane keeps, one of what it gives away and an add.  pair_sums: over 16 lanes (a DPP row) or 32 (two), lane l gets the sum
// of x (l even) or y (l odd).  quad_sums: over the LPR lanes of a state row, lane l gets that of x[sums_token(l) % 4], in eleven instructions
// (and a swap; ten for eight lanes) for four sums that would be sixteen one by one, four swaps and four selects.
template <int LANES>
__device__ __forceinline__ float pair_sums(float x, float y, int lane) {
    const bool odd = lane & 1;
    float s = (odd ? y : x) + dpp<0xB1>(odd ? x : y);   // quad_perm [1,0,3,2]
    s += dpp<0x4E>(s);                                  // quad_perm [2,3,0,1]
    s += dpp<0x124>(s);                                 // row_ror 4
    s += dpp<0x128>(s);                                 // row_ror 8
    if constexpr (LANES == 32) s = swap_add16(s, s);
    return s;
}
// which of the first min(LPR, 16) tokens a lane's sums are of
template <int LPR>
__device__ __forceinline__ int sums_token(int lane_of_row) {
    if constexpr (LPR == 8) return 2 * (lane_of_row & 2) + (lane_of_row >> 1 & 2) + (lane_of_row & 1);
    return lane_of_row % 16;
}
template <int LPR>
__device__ __forceinline__ float quad_sums(const float (&x)[4], int lane) {
    const bool odd = lane & 1;
    if constexpr (LPR == 8) {
        const bool upper = lane & 4;   // (the mirror of eight lanes exchanges their halves)
        const float even = (upper ? x[2] : x[0]) + dpp<0x141>(upper ? x[0] : x[2]), odds = (upper ? x[3] : x[1]) + dpp<0x141>(upper ? x[1] : x[3]);
        const float s = (odd ? odds : even) + dpp<0xB1>(odd ? even : odds);
        return s + dpp<0x4E>(s);
    }
    const bool upper = lane & 2;
    const float lo = (odd ? x[1] : x[0]) + dpp<0xB1>(odd ? x[0] : x[1]), hi = (odd ? x[3] : x[2]) + dpp<0xB1>(odd ? x[2] : x[3]);
    float s = (upper ? hi : lo) + dpp<0x4E>(upper ? lo : hi);
    s += dpp<0x124>(s);
    s += dpp<0x128>(s);
    if constexpr (LPR == 32) s = swap_add16(s, s);
    return s;
}

// What the forward keeps for the backward, in one buffer: the state entering every CH64 tokens ([B,H,T/CH64,C,C]) and
// then S a of every token ([B,T,H,C]; the backward's recomputation of the states inside a chunk then needs no row sums).
__host__ __device__ inline long saved_states(long BH, int T, int C) { return BH * (T / CH64) * C * C; }

// ADJ: the same recurrence backwards in time.  With E the state gradient that arrives from the tokens after t,
//     dsa = E b + dy (q . b);   dv = E k + dy (q . k);   E <- E diag(decay) + dsa a^T + dy (decay * q)^T
// is the forward's step with (a, decay q, b, k, v) in the places of (b, k, a, decay q, dy): two row sums on the state
// before its update, a rank-one term with the first of them and one with the row vector.  v, s0, y, ckpt, sT are then
// dy, dsT, dv, the workspace of the gradient kernel below (E arriving at every chunk's end, dsa of every token) and ds0.
template <int C, int LPR, int R, int NW, int NP, bool FULL, bool ADJ>
__global__ __launch_bounds__(64 * (NW + NP)) void wkv7_f32_scan_kernel(int T, int H, int CR, const float* __restrict__ w,
                                                             const float* __restrict__ q, const float* __restrict__ k,
                                                             const float* __restrict__ v, const float* __restrict__ a,
                                                             const float* __restrict__ b, const float* __restrict__ s0,
                                                             float* __restrict__ y, float* __restrict__ ckpt,
                                                             float* __restrict__ sT) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    constexpr int CH = CH64, Q = C / (4 * LPR), GPW = 64 / LPR, ROWS = NW * GPW * R, NSPLIT = C / ROWS;
    constexpr int PT = 64 * NP, QPT = C / 4, TPJ = PT / QPT, PER = CH / TPJ;   // moving: QPT threads, four channels each, per token
    constexpr int LDO = ROWS + 4, QPR = ROWS / 4;                              // results: a token's rows, QPR pieces of four
    constexpr bool SHARE = LPR == 8;                                           // of two pieces a lane reads one
    constexpr int KT = LPR < CH ? LPR : CH, KEPT = CH / KT;                    // of KT tokens a lane keeps one's results, KEPT times
    static_assert(C % ROWS == 0 && PT % QPT == 0 && CH % TPJ == 0 && (CH * QPR) % 64 == 0, "whole tokens and rows per thread");
    __shared__ __attribute__((aligned(16))) float in[2][FWD_VECS][CH][C];   // the slot of q holds decay * q
    // (b . q, k . q) of every token (as floats: the half of a pair that nobody uses is a register the compiler
    // reuses at once, behind a wait for everything in flight, a sixth of the backward scan)
    __shared__ __attribute__((aligned(8))) float bkq[2][CH][2];
    __shared__ __attribute__((aligned(16))) float yout[2][CH][LDO], saout[2][CH][LDO];
    const int bh = blockIdx.x / NSPLIT, part = blockIdx.x % NSPLIT, h = bh % H;
    const long bt0 = (long)(bh / H) * T;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, jb = lane % LPR, rl = (wv * GPW + lane / LPR) * R;
    const int row0 = part * ROWS + rl;
    auto col = [&](int x) { return 4 * jb + 4 * LPR * (SHARE ? x ^ (lane >> 3 & 1) : x); };   // piece x < Q of a lane's columns: four from here on
    const float* const src[FWD_VECS] = {w, q, k, v, a, b};
    float* const sav = ckpt == nullptr ? nullptr : ckpt + saved_states(gridDim.x / NSPLIT, T, CR);
    // Addresses are a base per chunk that is the same in every lane (scalar registers) plus a small 32-bit offset per
    // thread, instead of a 64-bit address per thread and access.
    // CR: the head size itself; C: the width the block works at (channels and rows past CR read as zero, are never
    // written, and stay zero in the state).  FULL: CR == C, no access needs a bound.
    const unsigned ld = (unsigned)H * CR;                                    // floats between consecutive tokens
    const int NC = T / CH;
    auto chunk_start = [&](int n) { return CH * (ADJ ? NC - 1 - n : n); };   // first token of the n-th chunk in the order of the walk
    auto chunk_base = [&](int n) { return seq_index(bt0 + chunk_start(n), H, h, 0, CR); };
    const f4 zero = {0.f, 0.f, 0.f, 0.f};

    // ---- moving data: thread ptid of PT, four channels of every TPJ-th token ----
    const int ptid = threadIdx.x - 64 * NW, pch = 4 * (ptid % QPT), ptok = ptid / QPT;
    const bool stage_ok = FULL || pch < CR;
    const unsigned tok_off = 4 * ((unsigned)ptok * ld + (stage_ok ? pch : 0));   // in bytes
    f4 pre[FWD_VECS][PER];
    auto fetch = [&](int n) {
        const long base = chunk_base(n < NC ? n : NC - 1);   // (past the last chunk: the same one again, not used)
#pragma unroll
        for (int vec = 0; vec < FWD_VECS; vec++) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const f4 x = at_bytes<seq4>(src[vec] + (base + (long)(TPJ * j) * ld), tok_off);
                pre[vec][j] = stage_ok ? x : zero;
            }
        }
    };
    // the fetched chunk into a buffer: the decay instead of w, decay * q instead of q.  With them
    //   y_t = S_t q = S_{t-1} (decay * q) + (S_{t-1} a) (b . q) + v (k . q),
    // so that both row sums of a token work on the state BEFORE its update and neither waits for the other.
    auto stage = [&](int buf) {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int tok = TPJ * j + ptok;
            auto put = [&](int vec, f4 x) { *reinterpret_cast<f4*>(&in[buf][vec][tok][pch]) = x; };
            f4 d;
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] = expf(-expf(pre[V_DEC][j][i]));
            put(V_DEC, d);
            put(V_Q, d * pre[V_Q][j]);
            put(V_K, pre[V_K][j]);
            put(V_V, pre[V_V][j]);
            put(V_A, pre[V_A][j]);
            put(V_B, pre[V_B][j]);
            const float bkq_lane = pair_sums<QPT>(dot4(pre[V_B][j], pre[V_Q][j]), dot4(pre[V_K][j], pre[V_Q][j]), lane);   // even lanes: b . q, odd ones: k . q
            if (pch < 8) bkq[buf][tok][lane & 1] = bkq_lane;
        }
    };
    auto copy_out = [&](int n, int buf) {
        const long base = chunk_base(n);
        constexpr int PIECES = CH * QPR;   // of either result
#pragma unroll
        for (int m = 0; m < (2 * PIECES + PT - 1) / PT; m++) {
            const int e = ptid + PT * m, which = e / PIECES, i = e % PIECES;   // (which: the same for a wavefront)
            const int tok = i / QPR, ch = 4 * (i % QPR);
            const unsigned at = (unsigned)tok * ld + (unsigned)(part * ROWS + ch);
            if (FULL || part * ROWS + ch < CR) {
                if (which == 0) __builtin_nontemporal_store(*reinterpret_cast<const f4*>(&yout[buf][tok][ch]), reinterpret_cast<seq4*>((y + base) + at));
                else if (which == 1 && sav != nullptr)
                    __builtin_nontemporal_store(*reinterpret_cast<const f4*>(&saout[buf][tok][ch]), reinterpret_cast<seq4*>((sav + base) + at));
            }
        }
    };
    if (wv >= NW) {   // (the same number of barriers as below)
        fetch(0);
        stage(0);
        fetch(1);
        lds_barrier();
        for (int n = 0; n < NC; n++) {
            if (n + 1 < NC) stage((n + 1) & 1);
            fetch(n + 2);
            if (n > 0) copy_out(n - 1, (n - 1) & 1);
            lds_barrier();
        }
        copy_out(NC - 1, (NC - 1) & 1);
        return;
    }

    // ---- the recurrence ----
    auto col_ok = [&](int x) { return FULL || col(x) < CR; };
    auto state_off = [&](int r, int x) { return (unsigned)((row0 + r) * CR + col(x)); };  // in a CR x CR state
    auto state_ok = [&](int r, int x) { return FULL || (col_ok(x) && row0 + r < CR); };
    f4 S[R][Q];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int x = 0; x < Q; x++)
            S[r][x] = state_ok(r, x) ? *reinterpret_cast<const f4*>(s0 + (long)bh * CR * CR + state_off(r, x)) : zero;
    const int kept_token = sums_token<LPR>(jb);   // of each KT
    [[maybe_unused]] const bool in_quad[4] = {(lane & 3) == 0, (lane & 3) == 1, (lane & 3) == 2, (lane & 3) == 3};
    // x in lanes 4 k .. 4 k + 3 of every DPP row, `to` elsewhere
    auto into_quad = [](float to, float x, int k) {
        auto move = [&](auto mask) {
            return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, to), __builtin_bit_cast(int, x), 0xE4, 0xf, decltype(mask)::value, false));
        };   // (quad_perm [0,1,2,3])
        using std::integral_constant;
        return k == 0 ? move(integral_constant<int, 1>()) : k == 1 ? move(integral_constant<int, 2>()) : k == 2 ? move(integral_constant<int, 4>())
                                                                                                             : move(integral_constant<int, 8>());
    };
    auto walk = [&](int n, int buf) {
        if (ckpt != nullptr) {
            float* const to = ckpt + ((long)bh * NC + chunk_start(n) / CH) * CR * CR;
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int x = 0; x < Q; x++) {
                    if (state_ok(r, x)) __builtin_nontemporal_store(S[r][x], reinterpret_cast<f4*>(to + state_off(r, x)));
                }
        }
        // a token's operands are requested from LDS one token ahead
        struct Ops {
            f4 dec[Q], x1[Q], x2[Q], u1[Q], u2[Q];   // operands of the two row sums, column vectors of the two rank-one terms
            RowVals<R> vr;
            float bq;
        };
        auto read_ops = [&](int t) {
            Ops o;
            auto read = [&](f4 (&to)[Q], int vec) {
#pragma unroll
                for (int x = 0; x < (SHARE ? 1 : Q); x++) to[x] = *reinterpret_cast<const f4*>(&in[buf][vec][t][col(x)]);
            };
            read(o.dec, V_DEC);
            read(o.x1, ADJ ? V_B : V_A);
            read(o.u1, ADJ ? V_A : V_B);
            read(o.u2, ADJ ? V_Q : V_K);
            read(o.x2, ADJ ? V_K : V_Q);
            o.vr = lds_rows<R>(&in[buf][V_V][t][row0]);
            if constexpr (ADJ) o.bq = bkq[buf][t][0];
            return o;
        };
        Ops ahead = read_ops(ADJ ? CH - 1 : 0);
        RowVals<R> ykeep[KEPT] = {}, sakeep[KEPT] = {};
        float ypart[R][4];   // four tokens' terms of S (decay * q)
        [[maybe_unused]] float sa4[R];
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const int t = ADJ ? CH - 1 - i : i;
            const Ops o = ahead;
            if (i + 1 < CH) ahead = read_ops(ADJ ? t - 1 : t + 1);
            asm volatile("" ::: "memory");   // (else all sixteen tokens' operands are requested at once)
            RowVals<R> sar;
#pragma unroll
            for (int r = 0; r < R; r++) {
                // element c of piece x of a token's vector, times s; the same plus acc
                auto times = [&](const f4 (&v)[Q], int x, int c, float s) { return s * (SHARE && x ? other_row(v[0][c]) : v[x][c]); };
                auto fma_at = [&](const f4 (&v)[Q], int x, int c, float s, float acc) {
                    return SHARE && x ? fma_other_row(v[0][c], s, acc) : fmaf(v[x][c], s, acc);
                };
                float p1[Q], p2[Q];
#pragma unroll
                for (int x = 0; x < Q; x++) {
                    p1[x] = times(o.x1, x, 0, S[r][x][0]), p2[x] = times(o.x2, x, 0, S[r][x][0]);
#pragma unroll
                    for (int c = 1; c < 4; c++) p1[x] = fma_at(o.x1, x, c, S[r][x][c], p1[x]), p2[x] = fma_at(o.x2, x, c, S[r][x][c], p2[x]);
                }
#pragma unroll
                for (int x = 1; x < Q; x++) p1[0] += p1[x], p2[0] += p2[x];
                sar.x[r] = row_sum<LPR>(p1[0]);
                if constexpr (ADJ) sar.x[r] += o.vr.x[r] * o.bq;
                ypart[r][t % 4] = p2[0];
#pragma unroll
                for (int x = 0; x < Q; x++)
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        // (in this order: the small term is the one rounded by itself.  y against fp64 9.14e-8; with the decayed state
                        // rounded first 9.39e-8, with sa b added last 9.57e-8)
                        S[r][x][c] = fma_at(o.u2, x, c, o.vr.x[r], fma_at(o.dec, x, c, S[r][x][c], times(o.u1, x, c, sar.x[r])));
            }
            // a lane of a row keeps one token's results of each KT (a store per token by one lane would be a branch per token,
            // which nothing is scheduled across); 32 lanes per row: both of its DPP rows hold and store the same.  The lanes of a
            // quad keep four tokens in a row, so the selects are between four and a move into one quad.
#pragma unroll
            for (int r = 0; r < R; r++) {
                if constexpr (LPR == 8) {
                    float& sa = sakeep[t / KT].x[r];
                    sa = kept_token == t % KT ? sar.x[r] : sa;
                    if (i % 4 == 3) {
                        const float y4 = quad_sums<LPR>(ypart[r], lane);   // (by every lane, not by those alone that keep it)
                        float& yk = ykeep[t / KT].x[r];
                        yk = kept_token / 4 == t % KT / 4 ? y4 : yk;
                    }
                    asm volatile("" : "+v"(sa));   // (here and now: put off, it keeps every token's operands alive)
                } else {
                    sa4[r] = i % 4 == 0 || in_quad[t % 4] ? sar.x[r] : sa4[r];
                    asm volatile("" : "+v"(sa4[r]));   // (here and now: put off, it keeps every token's operands alive)
                    if (i % 4 == 3) {
                        sakeep[0].x[r] = into_quad(sakeep[0].x[r], sa4[r], t / 4);
                        ykeep[0].x[r] = into_quad(ykeep[0].x[r], quad_sums<LPR>(ypart[r], lane), t / 4);
                    }
                }
            }
        }
        // what the row vectors add to y, once for the tokens that a lane keeps
#pragma unroll
        for (int m = 0; m < KEPT; m++) {
            const int t = KT * m + kept_token;
            const f2 sc = *reinterpret_cast<const f2*>(bkq[buf][t]);
            const RowVals<R> vr = lds_rows<R>(&in[buf][V_V][t][row0]);
#pragma unroll
            for (int r = 0; r < R; r++) {
                float yr = ykeep[m].x[r] + vr.x[r] * sc[1];
                if constexpr (!ADJ) yr += sakeep[m].x[r] * sc[0];
                yout[buf][t][rl + r] = yr;
                saout[buf][t][rl + r] = sakeep[m].x[r];
            }
        }
    };
    lds_barrier();
    for (int n = 0; n < NC; n++) {
        walk(n, n & 1);
        lds_barrier();
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int x = 0; x < Q; x++) {
            if (state_ok(r, x)) *reinterpret_cast<f4*>(sT + (long)bh * CR * CR + state_off(r, x)) = S[r][x];
        }
}

template <int C, int R, int NW, int WIN, bool FULL>
__global__ __launch_bounds__(64 * NW) void wkv7_f32_bwd_thin_kernel(int T, int H, int CR, const float* __restrict__ w,
                                                             const float* __restrict__ q, const float* __restrict__ k,
                                                             const float* __restrict__ v, const float* __restrict__ a,
                                                             const float* __restrict__ b, const float* __restrict__ dy,
                                                             const float* __restrict__ ckpt, const float* __restrict__ dsT,
                                                             float* __restrict__ dw, float* __restrict__ dq,
                                                             float* __restrict__ dk, float* __restrict__ dv,
                                                             float* __restrict__ da, float* __restrict__ db,
                                                             float* __restrict__ ds0) {
    constexpr int CH = CH64, LPR = C / 4, GPW = 64 / LPR, THREADS = 64 * NW, ROWS = NW * GPW * R, NSPLIT = C / ROWS;
    constexpr int PER = CH * C / THREADS, TPJ = THREADS / C;
    static_assert(C == 2 * ROWS && CH % WIN == 0 && (CH * C) % THREADS == 0 && (WIN * C) % THREADS == 0,
                  "two blocks per head (two addends per gradient element), whole windows, whole tokens per thread");
    constexpr int NSRC = 8, W_SA = BWD_VECS;     // the eighth vector per token: the forward's S a
    __shared__ __attribute__((aligned(16))) float in[BWD_VECS + 1][CH][C];
    __shared__ float red[NW][RED_VECS][WIN][C];   // per wavefront: column sums over its 4 R rows, a window of tokens
    __shared__ __attribute__((aligned(16))) float dvout[WIN][ROWS];
    const int bh = blockIdx.x / NSPLIT, part = blockIdx.x % NSPLIT, h = bh % H;
    const long bt0 = (long)(bh / H) * T;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, jb = lane % LPR, ib = lane / LPR, rl = (wv * GPW + ib) * R;
    const int row0 = part * ROWS + rl, col0 = 4 * jb;
    const float* const src[NSRC] = {w, q, k, v, a, b, dy, ckpt + saved_states(gridDim.x / NSPLIT, T, CR)};
    float* const dst[RED_VECS] = {dq, dk, db, da, dw};

    const unsigned ld = (unsigned)H * CR;                                    // (addresses and bounds: as in the forward kernel)
    const bool col_ok = FULL || col0 < CR, stage_ok = FULL || (int)(tid % C) < CR;
    const unsigned state_off = (unsigned)(row0 * CR + (col_ok ? col0 : 0));
    const unsigned tok_off = (unsigned)(tid / C) * ld + (stage_ok ? tid % C : 0);
    auto chunk_base = [&](int c0) { return seq_index(bt0 + c0, H, h, 0, CR); };
    auto row_ok = [&](int r) { return FULL || (col_ok && row0 + r < CR); };
    const f4 zero = {0.f, 0.f, 0.f, 0.f};

    f4 dS[R];
#pragma unroll
    for (int r = 0; r < R; r++)
        dS[r] = row_ok(r) ? *reinterpret_cast<const f4*>(dsT + (long)bh * CR * CR + (state_off + r * CR)) : zero;
    // the eight vectors per token and the saved state of the NEXT chunk (the one before in time) are fetched while the
    // current one runs
    float pre[NSRC][PER];
    f4 pre_s[R];
    auto fetch = [&](int c0) {
        const long base = chunk_base(c0);
#pragma unroll
        for (int vec = 0; vec < NSRC; vec++) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const float x = (src[vec] + base)[tok_off + (unsigned)(TPJ * j) * ld];
                pre[vec][j] = stage_ok ? x : 0.f;
            }
        }
        const float* const from = ckpt + ((long)bh * (T / CH) + c0 / CH) * CR * CR;
#pragma unroll
        for (int r = 0; r < R; r++) pre_s[r] = row_ok(r) ? *reinterpret_cast<const f4*>(from + (state_off + r * CR)) : zero;
    };
    fetch(T - CH);
    for (int c0 = T - CH; c0 >= 0; c0 -= CH) {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int tok = TPJ * j + tid / C, ch = tid % C;
            const float ew = expf(pre[W_DEC][j]), d = expf(-ew);
            in[W_DEC][tok][ch] = d;
            in[W_DDEC][tok][ch] = -ew * d;
#pragma unroll
            for (int vec = 1; vec < NSRC; vec++) in[vec == NSRC - 1 ? W_SA : vec][tok][ch] = pre[vec][j];
        }
        f4 Sx[R];             // the state entering the chunk
#pragma unroll
        for (int r = 0; r < R; r++) Sx[r] = pre_s[r];
        __syncthreads();
        fetch(c0 >= CH ? c0 - CH : c0);   // (after the first chunk in time: the same one again)
        // S_{t+1} = S_t diag(decay_t) + (S a)_t b_t^T + v_t k_t^T, with S a as the forward saved it.  Operands are read
        // from LDS one token ahead; the compiler barrier after each request keeps it from requesting a whole window's
        // operands at once (and from keeping them for the adjoint: 14 registers per token and row group).
        struct AdvOps {
            f4 dec, bv, kv;
            RowVals<R> vr, sar;
        };
        auto read_adv = [&](int t) {
            AdvOps o;
            o.dec = *reinterpret_cast<const f4*>(&in[W_DEC][t][col0]);
            o.bv = *reinterpret_cast<const f4*>(&in[W_B][t][col0]), o.kv = *reinterpret_cast<const f4*>(&in[W_K][t][col0]);
            o.vr = lds_rows<R>(&in[W_V][t][row0]), o.sar = lds_rows<R>(&in[W_SA][t][row0]);
            return o;
        };
        auto advance = [&](const f4 (&from)[R], f4 (&to)[R], const AdvOps& o) {
#pragma unroll
            for (int r = 0; r < R; r++) to[r] = from[r] * o.dec + o.sar.x[r] * o.bv + o.vr.x[r] * o.kv;
        };
        // a token's operands for the adjoint are requested from LDS one token ahead (the stores of the results in
        // between keep the compiler from moving the reads up by itself)
        struct AdjOps {
            f4 dec, av, bv, kv, qv;
            RowVals<R> vr, dyr, sar;
        };
        auto read_adj = [&](int t) {
            AdjOps o;
            o.dec = *reinterpret_cast<const f4*>(&in[W_DEC][t][col0]), o.av = *reinterpret_cast<const f4*>(&in[W_A][t][col0]);
            o.bv = *reinterpret_cast<const f4*>(&in[W_B][t][col0]), o.kv = *reinterpret_cast<const f4*>(&in[W_K][t][col0]);
            o.qv = *reinterpret_cast<const f4*>(&in[W_Q][t][col0]);
            o.vr = lds_rows<R>(&in[W_V][t][row0]), o.dyr = lds_rows<R>(&in[W_DY][t][row0]), o.sar = lds_rows<R>(&in[W_SA][t][row0]);
            return o;
        };
        // the chunk in windows of WIN tokens, last window first: the states of a window are recomputed into registers
        // (from the chunk's first state: the windows before it are run through once more, a running state only), then
        // the adjoint recurrence walks back through them
#pragma unroll 1
        for (int win = CH / WIN - 1; win >= 0; win--) {
            const int t0 = win * WIN;
            f4 St[WIN + 1][R];     // St[t] enters token t0 + t
#pragma unroll
            for (int r = 0; r < R; r++) St[0][r] = Sx[r];
            AdvOps adv = read_adv(0);
#pragma unroll 1
            for (int t = 0; t < t0; t++) {
                const AdvOps o = adv;
                adv = read_adv(t + 1);
                asm volatile("" ::: "memory");
                advance(St[0], St[0], o);
            }
#pragma unroll
            for (int tw = 0; tw < WIN; tw++) {
                const AdvOps o = adv;
                if (tw + 1 < WIN) adv = read_adv(t0 + tw + 1);
                asm volatile("" ::: "memory");
                advance(St[tw], St[tw + 1], o);
            }
            AdjOps ahead = read_adj(t0 + WIN - 1);
#pragma unroll
            for (int tw = WIN - 1; tw >= 0; tw--) {
                const int t = t0 + tw;
                const AdjOps o = ahead;
                if (tw > 0) ahead = read_adj(t - 1);
                asm volatile("" ::: "memory");
                const f4 dec = o.dec, av = o.av, bv = o.bv, kv = o.kv, qv = o.qv;
                const RowVals<R> vr = o.vr, dyr = o.dyr, sar = o.sar;
                // dq = S_t^T dy;  dS_t += dy q^T;  dv = dS k;  dsa = dS b
                f4 pq = St[tw + 1][0] * dyr.x[0];
#pragma unroll
                for (int r = 1; r < R; r++) pq += St[tw + 1][r] * dyr.x[r];
                float dsa[R];
                RowVals<R> dvr;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    dS[r] += dyr.x[r] * qv;
                    dvr.x[r] = row_sum<LPR>(dot4(dS[r], kv));
                    dsa[r] = row_sum<LPR>(dot4(dS[r], bv));
                }
                if (jb == 0) {
#pragma unroll
                    for (int r = 0; r < R; r++) dvout[tw][rl + r] = dvr.x[r];
                }
                // dk = dS^T v;  db = dS^T sa;  da = S_{t-1}^T dsa;  ddecay = sum over rows of dS * S_{t-1}
                f4 pk = dS[0] * vr.x[0], pb = dS[0] * sar.x[0], pa = St[tw][0] * dsa[0], pw = dS[0] * St[tw][0];
#pragma unroll
                for (int r = 1; r < R; r++) {
                    pk += dS[r] * vr.x[r];
                    pb += dS[r] * sar.x[r];
                    pa += St[tw][r] * dsa[r];
                    pw += dS[r] * St[tw][r];
                }
                store_col_sums<LPR>(red[wv][R_DQ][tw], pq, col0, ib);
                store_col_sums<LPR>(red[wv][R_DK][tw], pk, col0, ib);
                store_col_sums<LPR>(red[wv][R_DB][tw], pb, col0, ib);
                store_col_sums<LPR>(red[wv][R_DA][tw], pa, col0, ib);
                store_col_sums<LPR>(red[wv][R_DW][tw], pw, col0, ib);
                // dS_{t-1} = dS_t diag(decay) + dsa a^T
#pragma unroll
                for (int r = 0; r < R; r++) dS[r] = dS[r] * dec + dsa[r] * av;
            }
            __syncthreads();
            // the wavefronts' sums of this window, in a fixed order, and out
#pragma unroll
            for (int vec = 0; vec < RED_VECS; vec++) {
#pragma unroll
                for (int j = 0; j < WIN * C / THREADS; j++) {
                    const int tw = TPJ * j + tid / C, tok = win * WIN + tw, ch = tid % C;
                    float s = red[0][vec][tw][ch];
#pragma unroll
                    for (int g = 1; g < NW; g++) s += red[g][vec][tw][ch];
                    if (vec == R_DW) s *= in[W_DDEC][tok][ch];
                    float* const p = dst[vec] + chunk_base(c0) + (tok_off + (unsigned)(win * WIN + TPJ * j) * ld);
                    if (FULL || ch < CR) unsafeAtomicAdd(p, s);   // (onto zeros; the other block of the head adds its part)
                }
            }
#pragma unroll
            for (int m = 0; m < (WIN * ROWS + THREADS - 1) / THREADS; m++) {
                const int e = tid + THREADS * m;
                const int tw = e / ROWS, ch = e % ROWS;
                if (((WIN * ROWS) % THREADS == 0 || e < WIN * ROWS) && (FULL || part * ROWS + ch < CR))
                    (dv + chunk_base(c0))[(unsigned)(win * WIN + tw) * ld + (unsigned)(part * ROWS + ch)] = dvout[tw][ch];
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (row_ok(r)) *reinterpret_cast<f4*>(ds0 + (long)bh * CR * CR + (state_off + r * CR)) = dS[r];
    }
}

// The gradients of one chunk (16 tokens) of one head and 64 of its columns, from the state S entering the chunk, the state
// gradient E arriving at its end, and S a (sa) and dsa of every token: nothing is left to wait for, every chunk and column
// block is one wavefront on its own.  Inside a chunk the state is S under the decays plus rank-one terms, S_t = S D(0..t) +
// sum_{i<=t} (sa_i b_i^T + v_i k_i^T) D(i+1..t) with D(i..t) the product of the decays of tokens i .. t (never above one and
// never divided by: the range of w stays the recurrence's), and likewise backwards, so
//     dq_j = D(0..j) S^T dy_j + sum_{i<=j} D(i+1..j) ((sa_i.dy_j) b_i + (v_i.dy_j) k_i)       da_j: dsa_j, decays up to j - 1
//     dk_i = D(i+1..15) E^T v_i + sum_{j>=i} D(i+1..j) (v_i.dy_j) q_j + sum_{j>i} D(i+1..j-1) (v_i.dsa_j) a_j       db_i: sa_i
// each of them a Horner scheme in the decays: fifteen multiply-adds per column and pair i <= j instead of thirteen per column,
// token and ROW of the state.  The gradient of a decay, R_t = sum over rows of dS_t * S_{t-1} and dw_t = -exp(w_t) decay_t R_t,
// is two more such schemes: z = sum over rows of S * E, then down the tokens + q xq (R_t so far), * decay, + a xa with xq, xa =
// S^T [dy dsa] for the terms of S, times D(0..t-1); and dk_i, db_i as their own schemes have them at token t, times k_i, b_i and
// D(i+1..t-1).  (W_t = decay_t R_t is also what is left of W_{t-1} after four terms have come and gone, three multiply-adds less,
// but the terms do not carry decay_t: from w = 3.3 on, the difference is rounding, 2e-4 of it there and all of it at 4.)
// What needs the rows of the states - S^T [dy dsa], E^T [v sa], the sums of S * E and the four 16 x 16 products of row
// vectors - is one pass of matrix instructions over them.  All of it in fp64, whose multiply-add is as fast as fp32's here and
// whose matrix instruction takes twice as long: a sum over rows averages the roundings of its terms, a sum of the terms'
// sums does not, and in fp32 the errors would be 1.7e-7 where recomputing the states row by row left 0.9e-7.
// Bound: memory, 90 KB per chunk and 64 columns: 8 x 1024 tokens x 12 heads of 64 152 us for 553 MB (148 with dw as that
// difference; of 142 on another machine, 123 without the matrix instructions, 132 without the pairs of tokens, 118 without
// either; 142 with the states read and the results written past the caches, a pass with its scans' stores so as well 435 -> 417), where
// recomputing the states took 218; 32 x 1024 x 12 852 -> 560, 8 x 1024 x 6 heads of 128 477 -> 221, 8 x 1024 x 16 heads
// of 32 157 -> 101.  Errors at 8 x 1024 x 12 against fp64: dq, dk 0.42e-7, dw 0.64e-7 (0.69 as a difference), da, db 0.98e-7.
template <int CR, int COLS>   // head size, columns of a block
__global__ __launch_bounds__(64, 2) void wkv7_f32_grads_kernel(int T, int H, const float* __restrict__ w, const float* __restrict__ q,
                                                               const float* __restrict__ k, const float* __restrict__ v,
                                                               const float* __restrict__ a, const float* __restrict__ b,
                                                               const float* __restrict__ dy, const float* __restrict__ ckpt,
                                                               const float* __restrict__ work, float* __restrict__ dw,
                                                               float* __restrict__ dq, float* __restrict__ dk,
                                                               float* __restrict__ da, float* __restrict__ db) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef double d4 __attribute__((ext_vector_type(4)));
    constexpr int CH = CH64, HALF = 32, HALVES = COLS / HALF;
    static_assert(CH == 16 && (HALVES == 1 || HALVES == 2), "a chunk is one tile of the matrix instruction; a lane per column");
    enum { Q_V = 0, Q_SA, Q_DY, Q_DSA, Q_VECS };
    enum { G_SY = 0, G_VY, G_SD, G_VD };
    __shared__ __attribute__((aligned(16))) float xs[2][CH][HALF], ys[2][CH][2 * HALF];   // S^T dy and dsa of 32 columns; E^T v and sa
    float(*const es)[2 * HALF] = reinterpret_cast<float(*)[2 * HALF]>(xs);                  // then exp(w) of all tokens and columns
    __shared__ double zs[4][HALF];
    __shared__ d4 gram[CH * (CH + 1) / 2];                                // sa.dy, v.dy, sa.dsa, v.dsa of tokens i <= j
    auto pair = [](int i, int j) { return i * CH - i * (i - 1) / 2 + j - i; };
    const int NC = T / CH, bh = blockIdx.x / NC, chunk = blockIdx.x - bh * NC, h = bh % H;
    const int lane = threadIdx.x, g = lane >> 4, n = lane & 15;
    const int col0 = COLS * blockIdx.y, col = col0 + lane;
    const bool col_ok = (HALVES == 2 || lane < COLS) && (CR % COLS == 0 || col < CR);
    const int colc = col_ok ? col : 0;                                    // (lanes past the columns: column 0, nothing written)
    const long base = seq_index((long)(bh / H) * T + (long)chunk * CH, H, h, 0, CR);
    const unsigned ld = (unsigned)H * CR;
    const long nstate = saved_states(gridDim.x / NC, T, CR), st = (long)blockIdx.x * CR * CR;
    const float* const row_src[Q_VECS] = {v, ckpt + nstate, dy, work + nstate};

    // Matrix instructions of 16 x 16 x 4: lane (g, n) gives element (n, k = g) of the left operand and (k = g, n) of the right
    // one and gets elements (4 i + g, n) of the product.  Row r = 16 u + 4 g + s of a state is index g of step (u, s); column
    // 32 half + 2 n + t is column n of tile t, so that a lane reads two columns of a row and four rows of a token at a time.
    auto mma = [](double x, double y, d4 acc) { return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, acc, 0, 0, 0); };
    float xqv[CH], xav[CH];
    double z = 0.;
    d4 gr[4] = {};
    constexpr int STEPS = CR / 16;
    struct Rows {   // 16 rows of the states and of the tokens' row vectors
        f4 row[Q_VECS];
        f2 S[4], E[4];
    };
    auto fetch = [&](int x) {   // those of step x of both halves (past the end: the last ones again)
        Rows to;
        const int y = min(x, HALVES * STEPS - 1), half = y >= STEPS, u = y - half * STEPS, c = col0 + HALF * half + 2 * n;
        const unsigned lane_at = 4 * (4 * g * CR + (CR % COLS == 0 || c < CR ? c : 0));
#pragma unroll
        for (int v = 0; v < Q_VECS; v++) to.row[v] = at_bytes<f4>(row_src[v] + (base + 16 * u), 4 * ((unsigned)n * ld + 4 * g));
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const long at = st + (16 * u + s) * CR;
            to.S[s] = __builtin_nontemporal_load(&at_bytes<f2>(ckpt + at, lane_at)), to.E[s] = __builtin_nontemporal_load(&at_bytes<f2>(work + at, lane_at));
        }
        return to;
    };
    Rows next0 = fetch(0), next1;
    if (HALVES * STEPS > 1) next1 = fetch(1);
    float cw[CH], cq[CH], ck[CH], ca[CH], cb[CH];   // the columns of the tokens' vectors
    const unsigned lane_col = 4 * colc;
#pragma unroll
    for (int half = 0; half < HALVES; half++) {
        d4 xq[2] = {}, xa[2] = {}, yk[2] = {}, yb[2] = {};
        double zz[2] = {};
        auto multiply = [&](const Rows& at) {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const double vr = at.row[Q_V][s], sar = at.row[Q_SA][s], dyr = at.row[Q_DY][s], dsar = at.row[Q_DSA][s];
                if (half == 0) {
                    gr[G_SY] = mma(sar, dyr, gr[G_SY]), gr[G_VY] = mma(vr, dyr, gr[G_VY]);
                    gr[G_SD] = mma(sar, dsar, gr[G_SD]), gr[G_VD] = mma(vr, dsar, gr[G_VD]);
                }
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const double Sd = at.S[s][t], Ed = at.E[s][t];
                    xq[t] = mma(dyr, Sd, xq[t]), xa[t] = mma(dsar, Sd, xa[t]);
                    yk[t] = mma(vr, Ed, yk[t]), yb[t] = mma(sar, Ed, yb[t]);
                    zz[t] += Sd * Ed;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        const bool some = CR % COLS == 0 || col0 + HALF * half < CR;   // (a column of this half)
        int steps = some ? STEPS - (half == HALVES - 1) : 0;
        asm volatile("" : "+s"(steps));   // (a loop also where it has one step: what follows must not move up into it)
#pragma unroll 1
        for (int u = 0; u < steps; u++) {
            const Rows at = next0;
            next0 = next1;
            if (half < HALVES - 1 || u + 2 < STEPS) next1 = fetch(STEPS * half + u + 2);
            multiply(at);
        }
        if (half == HALVES - 1) {
#pragma unroll
            for (int t = 0; t < CH; t++) {
                const long at = base + (long)t * ld;
                cw[t] = at_bytes<float>(w + at, lane_col), cq[t] = at_bytes<float>(q + at, lane_col);
                ck[t] = at_bytes<float>(k + at, lane_col), ca[t] = at_bytes<float>(a + at, lane_col), cb[t] = at_bytes<float>(b + at, lane_col);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (some) multiply(next0);
        }
        // from tokens 4 i + g and columns 2 n + t to a column per lane
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (half == 0 && 4 * i + g <= n) gram[pair(4 * i + g, n)] = d4{gr[G_SY][i], gr[G_VY][i], gr[G_SD][i], gr[G_VD][i]};
            *reinterpret_cast<f2*>(&xs[0][4 * i + g][2 * n]) = f2{(float)xq[0][i], (float)xq[1][i]};
            *reinterpret_cast<f2*>(&xs[1][4 * i + g][2 * n]) = f2{(float)xa[0][i], (float)xa[1][i]};
            *reinterpret_cast<f2*>(&ys[0][4 * i + g][HALF * half + 2 * n]) = f2{(float)yk[0][i], (float)yk[1][i]};
            *reinterpret_cast<f2*>(&ys[1][4 * i + g][HALF * half + 2 * n]) = f2{(float)yb[0][i], (float)yb[1][i]};
        }
        zs[g][2 * n] = zz[0], zs[g][2 * n + 1] = zz[1];
        __syncthreads();
        if (HALVES == 1 || lane / HALF == half) {
#pragma unroll
            for (int t = 0; t < CH; t++) xqv[t] = xs[0][t][lane % HALF], xav[t] = xs[1][t][lane % HALF];
            z = (zs[0][lane % HALF] + zs[1][lane % HALF]) + (zs[2][lane % HALF] + zs[3][lane % HALF]);
        }
        __syncthreads();
    }
    double qv[CH], av[CH], dqv[CH], dav[CH], R[CH];
    float dec[CH];   // (to fp64 where it is used: sixteen double decays would not fit the registers)
#pragma unroll
    for (int t = 0; t < CH; t++) {
        const float ew = expf(cw[t]);
        es[t][lane] = ew, dec[t] = expf(-ew);
    }
    // the pairs i <= j, i upwards and j downwards; the products of row vectors are read AHEAD pairs early
    constexpr int AHEAD = 1;
    d4 ahead[AHEAD];
    int ni = 0, nj = CH - 1, slot = 0;   // (all known at compile time once the loops are unrolled)
    auto read_next = [&](d4& m) {
        if (ni < CH) m = gram[pair(ni, nj)];
        if (nj > ni) nj--;
        else ni++, nj = CH - 1;
    };
#pragma unroll
    for (int x = 0; x < AHEAD; x++) read_next(ahead[x]);
#pragma unroll
    for (int i = 0; i < CH; i++) {
        asm volatile("" : "+v"(cb[i]), "+v"(ck[i]));   // (fp32 until now)
        const double bi = cb[i], ki = ck[i], deci = dec[i];
        double dki = ys[0][i][lane], dbi = ys[1][i][lane];
#pragma unroll
        for (int j = CH - 1; j >= i; j--) {
            const d4 m = ahead[slot];
            read_next(ahead[slot]);
            slot = (slot + 1) % AHEAD;
            const double decj = dec[j];
            if (i == 0) {   // the terms of the entering state: tokens downwards, as this first round of pairs goes
                asm volatile("" : "+v"(cq[j]), "+v"(ca[j]), "+v"(xqv[j]), "+v"(xav[j]));   // (fp32 until now)
                qv[j] = cq[j], av[j] = ca[j], dqv[j] = xqv[j], dav[j] = xav[j];
                R[j] = z + qv[j] * dqv[j];
                z = R[j] * decj + av[j] * dav[j];
            }
            dqv[j] = dqv[j] * deci + (m[G_SY] * bi + m[G_VY] * ki);
            dki += m[G_VY] * qv[j], dbi += m[G_SY] * qv[j];
            if (j > i) {
                R[j] = R[j] * deci + (ki * dki + bi * dbi);
                dav[j] = dav[j] * deci + (m[G_SD] * bi + m[G_VD] * ki);
                dki = dki * decj + m[G_VD] * av[j], dbi = dbi * decj + m[G_SD] * av[j];
            }
            asm volatile("" : "+v"(dqv[j]), "+v"(dav[j]), "+v"(dki), "+v"(dbi), "+v"(R[j]), "+v"(dec[j]) : : "memory");   // (else every pair's operands are in registers at once)
        }
        if (col_ok) {
            const long at = base + (long)i * ld;
            __builtin_nontemporal_store((float)dqv[i], &at_bytes<float>(dq + at, lane_col)), __builtin_nontemporal_store((float)dav[i], &at_bytes<float>(da + at, lane_col));
            __builtin_nontemporal_store((float)dki, &at_bytes<float>(dk + at, lane_col)), __builtin_nontemporal_store((float)dbi, &at_bytes<float>(db + at, lane_col));
            const double ew = dec[i] > 0.f ? es[i][lane] : 0.f;   // (exp(w) may be infinite where the decay is zero)
            __builtin_nontemporal_store((float)(-ew * deci * R[i]), &at_bytes<float>(dw + at, lane_col));
        }
    }
}

// The same gradients where the chunks are too few to fill the chip: four wavefronts to a chunk and 32 of its columns, which share
// what one does one after the other above.  Bound: that chain, not memory (64 channels, 64 chunks: 11.5 us, of which the pairs 5.7
// and the products 2.5; one wavefront 17.4; the recurrence's states recomputed row by row took 11.2, with twice the error in dq).
//   A wavefront makes three of the twelve products (S or E times a token vector, and one of the four without a state);
//   the 256 threads share the exponentials and the sums of S * E;
//   the pairs are two wavefronts: dq and da, which need the products of row vectors only, and dk, db and dw;
//   in both, the halves of a wavefront are two gradients of the same columns: lanes 0-31 dq | dk, lanes 32-63 da | db.
// In fp64, and sums over rows in the same order as above.  (The pairs as loops over four i, a quarter of the instructions: 12.2 us;
// the pairs' two wavefronts on other SIMDs for every second block: no gain where two blocks share a compute unit.)
template <int CR>
__global__ __launch_bounds__(256, 2) void wkv7_f32_grads_few_kernel(int T, int H, const float* __restrict__ w, const float* __restrict__ q,
                                                                    const float* __restrict__ k, const float* __restrict__ v,
                                                                    const float* __restrict__ a, const float* __restrict__ b,
                                                                    const float* __restrict__ dy, const float* __restrict__ ckpt,
                                                                    const float* __restrict__ work, float* __restrict__ dw,
                                                                    float* __restrict__ dq, float* __restrict__ dk,
                                                                    float* __restrict__ da, float* __restrict__ db) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef double d2 __attribute__((ext_vector_type(2)));
    typedef double d4 __attribute__((ext_vector_type(4)));
    constexpr int CH = CH64, COLS = 32, STEPS = CR / 16, PAIRS = CH * (CH + 1) / 2;
    __shared__ float prod[4][CH][COLS];                                       // S^T dy, S^T dsa, E^T v, E^T sa
    __shared__ __attribute__((aligned(16))) double gx[PAIRS][4], gy[PAIRS][4];   // of tokens i <= j: sa.dy, v.dy | sa.dsa, v.dsa and v.dy, v.dsa | sa.dy, sa.dsa
    __shared__ float es[CH][COLS], ds[CH][COLS];
    __shared__ double zs[8][COLS];
    auto pair = [](int i, int j) { return i * CH - i * (i - 1) / 2 + j - i; };
    const int NC = T / CH, bh = blockIdx.x / NC, chunk = blockIdx.x - bh * NC, h = bh % H;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int cl = lane % COLS, col0 = COLS * blockIdx.y;                     // (tid % COLS is the same column)
    const bool upper = lane >= COLS, col_ok = CR % COLS == 0 || col0 + cl < CR;
    const long base = seq_index((long)(bh / H) * T + (long)chunk * CH, H, h, 0, CR);
    const unsigned ld = (unsigned)H * CR, lane_col = 4 * (col_ok ? col0 + cl : 0);   // (past the columns: column 0, nothing written)
    const long nstate = saved_states(gridDim.x / NC, T, CR), st = (long)blockIdx.x * CR * CR;
    const float *const sa = ckpt + nstate, *const dsa = work + nstate;

    // what is read is asked for before anything waits (of the states and row vectors, four steps of 16 rows)
    const float* const left = wv == 0 || wv == 3 ? sa : v;                    // the product of row vectors: sa.dy, v.dsa, v.dy, sa.dsa
    const float* const right = wv == 0 || wv == 2 ? dy : dsa;
    const float* const state = wv < 2 ? ckpt : work;                          // S with the right one, E with the left one
    constexpr int EARLY = STEPS < 4 ? STEPS : 4;
    f4 lrow[EARLY], rrow[EARLY];
    f2 srow[EARLY][4];
    const int c = col0 + 2 * n;
    const unsigned row_at = 4 * ((unsigned)n * ld + 4 * g), state_at = 4 * (4 * g * CR + (CR % COLS == 0 || c < CR ? c : 0));
    auto fetch = [&](int u) {
        lrow[u % EARLY] = at_bytes<f4>(left + (base + 16 * u), row_at), rrow[u % EARLY] = at_bytes<f4>(right + (base + 16 * u), row_at);
#pragma unroll
        for (int s = 0; s < 4; s++) srow[u % EARLY][s] = at_bytes<f2>(state + (st + (16 * u + s) * CR), state_at);
    };
#pragma unroll
    for (int u = 0; u < EARLY; u++) fetch(u);
    float cw[CH / 8], zS[CR / 8], zE[CR / 8];                                 // eight tokens and eight rows by thread group
    const unsigned group = tid / COLS;
#pragma unroll
    for (int m = 0; m < CH / 8; m++) cw[m] = at_bytes<float>(w + (base + (long)(8 * m) * ld), 4 * group * ld + lane_col);
#pragma unroll
    for (int m = 0; m < CR / 8; m++) {
        zS[m] = at_bytes<float>(ckpt + (st + 8 * m * CR), 4 * group * CR + lane_col);
        zE[m] = at_bytes<float>(work + (st + 8 * m * CR), 4 * group * CR + lane_col);
    }
    float x0[CH], x1[CH], x2[CH];                                             // wavefront 0: b, k; wavefront 1: q, a, and k | b
    if (wv < 2) {
        const float *const p0 = wv == 0 ? b : q, *const p1 = wv == 0 ? k : a, *const p2 = upper ? b : k;
#pragma unroll
        for (int t = 0; t < CH; t++) {
            const long at = base + (long)t * ld;
            x0[t] = at_bytes<float>(p0 + at, lane_col), x1[t] = at_bytes<float>(p1 + at, lane_col);
            if (wv == 1) x2[t] = at_bytes<float>(p2 + at, lane_col);
        }
    }
    {
        double z = 0.;
#pragma unroll
        for (int m = 0; m < CR / 8; m++) z += (double)zS[m] * zE[m];
        zs[group][cl] = z;
#pragma unroll
        for (int m = 0; m < CH / 8; m++) {
            const float ew = expf(cw[m]);
            es[8 * m + group][cl] = ew, ds[8 * m + group][cl] = expf(-ew);
        }
        auto mma = [](double x, double y, d4 acc) { return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, acc, 0, 0, 0); };
        d4 gr = {}, x[2] = {};
#pragma unroll
        for (int u = 0; u < STEPS; u++) {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const double l = lrow[u % EARLY][s], r = rrow[u % EARLY][s], own = wv < 2 ? r : l;
                gr = mma(l, r, gr);
                x[0] = mma(own, srow[u % EARLY][s][0], x[0]), x[1] = mma(own, srow[u % EARLY][s][1], x[1]);
            }
            if (u + EARLY < STEPS) fetch(u + EARLY);
        }
        const int to_x = wv == 0 ? 0 : wv == 1 ? 3 : wv == 2 ? 1 : 2, to_y = wv == 0 ? 2 : wv == 1 ? 1 : wv == 2 ? 0 : 3;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const int i = 4 * m + g;
            *reinterpret_cast<f2*>(&prod[wv][i][2 * n]) = f2{(float)x[0][m], (float)x[1][m]};
            if (i <= n) {
                gx[pair(i, n)][to_x] = gr[m], gy[pair(i, n)][to_y] = gr[m];
            }
        }
    }
    __syncthreads();
    if (wv >= 2) return;
    // the products of the pairs are read AHEAD pairs early (eight of them spill)
    constexpr int AHEAD = 4;
    d2 ahead[AHEAD];
    const double(*const gram)[4] = wv == 0 ? gx : gy;
    int ni = 0, nj = CH - 1, slot = 0;   // (all known at compile time once the loops are unrolled)
    auto read_next = [&](d2& m) {
        if (ni < CH) m = *reinterpret_cast<const d2*>(&gram[pair(ni, nj)][2 * upper]);
        if (nj > ni) nj--;
        else ni++, nj = CH - 1;
    };
    auto next = [&] {
        const d2 m = ahead[slot];
        read_next(ahead[slot]);
        slot = (slot + 1) % AHEAD;
        return m;
    };
#pragma unroll
    for (int x = 0; x < AHEAD; x++) read_next(ahead[x]);
    double dec[CH];
#pragma unroll
    for (int t = 0; t < CH; t++) dec[t] = ds[t][cl];
    if (wv == 0) {
        float* const to = upper ? da : dq;
        double x[CH];
#pragma unroll
        for (int t = 0; t < CH; t++) x[t] = prod[upper][t][cl];
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const double bi = x0[i], ki = x1[i];
#pragma unroll
            for (int j = CH - 1; j >= i; j--) {
                const d2 m = next();
                const double more = x[j] * dec[i] + (m[0] * bi + m[1] * ki);
                x[j] = i == j && upper ? x[j] : more;           // (da_j: tokens before j only)
                asm volatile("" : "+v"(x[j]) : : "memory");   // (in this order, as above)
            }
            if (col_ok) at_bytes<float>(to + (base + (long)i * ld), lane_col) = (float)x[i];
        }
    } else {
        float* const to = upper ? db : dk;
        double R[CH], qv[CH], av[CH], z = 0.;
#pragma unroll
        for (int m = 0; m < 8; m++) z += zs[m][cl];
#pragma unroll
        for (int t = CH - 1; t >= 0; t--) {
            qv[t] = x0[t], av[t] = x1[t];
            R[t] = z + qv[t] * prod[0][t][cl];
            z = R[t] * dec[t] + av[t] * prod[1][t][cl];
            R[t] = upper ? 0. : R[t];
        }
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const double ci = x2[i];
            double y = prod[2 + upper][i][cl];
#pragma unroll
            for (int j = CH - 1; j >= i; j--) {
                const d2 m = next();
                const double yq = m[0] * qv[j];
                if (j > i) {   // (y waits for one multiply-add a pair)
                    R[j] = R[j] * dec[i] + ci * (y + yq);
                    y = y * dec[j] + (yq * dec[j] + m[1] * av[j]);
                } else {
                    y += yq;
                }
                asm volatile("" : "+v"(y), "+v"(R[j]) : : "memory");
            }
            if (col_ok) at_bytes<float>(to + (base + (long)i * ld), lane_col) = (float)y;
        }
#pragma unroll
        for (int t = 0; t < CH; t++) {
            // lanes 0-31: the other half of the sum
            const unsigned long long bits = __builtin_bit_cast(unsigned long long, R[t]);
            const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)bits, (unsigned)bits, false, false);
            const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(bits >> 32), (unsigned)(bits >> 32), false, false);
            const double Rt = R[t] + __builtin_bit_cast(double, (unsigned long long)hi[1] << 32 | lo[1]);
            const float ew = es[t][cl];
            if (col_ok && !upper) at_bytes<float>(dw + (base + (long)t * ld), lane_col) = (float)((dec[t] > 0. ? -ew : 0.f) * dec[t] * Rt);
        }
    }
}

// five tensors of n floats each to zero (what the two-blocks-per-head backward adds its parts onto)
__global__ __launch_bounds__(256) void zero5_kernel(long n4, f4* __restrict__ p0, f4* __restrict__ p1, f4* __restrict__ p2,
                                                    f4* __restrict__ p3, f4* __restrict__ p4) {
    f4* const p[5] = {p0, p1, p2, p3, p4};
    const f4 z = {0.f, 0.f, 0.f, 0.f};
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n4; i += (long)gridDim.x * 256) {
#pragma unroll
        for (int t = 0; t < 5; t++) p[t][i] = z;
    }
}


// Blocks per head in the scan, by the times of the forward one (us).  Up to 64 channels: as many of 4, 2, 1 as still leave every block a compute
// unit of its own (1024 tokens: 97, 130, 203; 96 heads in 4 blocks each 145, in 2 131; 192 heads in 2 blocks each 234, in 1 206),
// and 2 again past one head per compute unit, where several blocks share one and smaller ones fill it more evenly (512 tokens in 1 block
// each, in 2: 288 heads 189, 162; 384 196, 182; 576 289, 273.  Where the heads fill whole rounds of the compute units, or nearly, 1 takes less: 448
// heads 202, 220; 512 214, 232; 1024 411, 459; with the backward pass 4-7 %).  Above 64 channels a block has a compute unit to itself
// (LDS), so the blocks run in rounds: the fewest rounds x time of a round (ns per token, 128 channels: 165, 220, 358 in 8, 4, 2
// blocks; 512 tokens in 4, 2 blocks: 136 heads 341, 371; 192 376, 380; 264 581, 565; 320 628, 574; 448 870, 758).
int scan_split(int BH, int C) {
    const long cus = compute_units(), n = BH;
    if (C <= 64) return 4 * n <= cus ? 4 : 2 * n <= cus || n > cus ? 2 : 1;
    auto cost = [&](int split, int ns) { return (split * n + cus - 1) / cus * ns; };
    const long c8 = cost(8, 165), c4 = cost(4, 220), c2 = cost(2, 358);
    return c8 <= c4 && c8 <= c2 ? 8 : c4 <= c2 ? 4 : 2;
}

}  // namespace

size_t wkv7_f32_saved_bytes(int B, int T, int H, int C) {
    return ((size_t)saved_states((long)B * H, T, C) + (size_t)B * T * H * C) * sizeof(float);
}

// (head sizes up to 64 run at a width of 64 channels, larger ones at 128; FULL: the head fills the width)
template <bool ADJ>
static void launch_scan(int B, int T, int H, int C, const float* w, const float* q, const float* k, const float* v, const float* a,
                        const float* b, const float* s0, float* y, float* ckpt, float* sT, hipStream_t stream) {
    const int split = scan_split(B * H, C);
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3(split * B * H), dim3(threads), 0, stream, T, H, C, w, q, k, v, a, b, s0, y, ckpt, sT);
    };
    // (width, rows per thread, wavefronts of the recurrence, of the moves): rows per block = wavefronts x row groups per
    // wavefront x rows per thread
    auto width64 = [&](auto full) {
        constexpr bool F = decltype(full)::value;
        if (split == 4) launch(wkv7_f32_scan_kernel<64, 16, 1, 4, 4, F, ADJ>, 512);
        else if (split == 2) launch(wkv7_f32_scan_kernel<64, 8, 1, 4, 4, F, ADJ>, 512);
        else launch(wkv7_f32_scan_kernel<64, 8, 1, 8, 4, F, ADJ>, 768);
    };
    auto width128 = [&](auto full) {
        constexpr bool F = decltype(full)::value;
        if (split == 8) launch(wkv7_f32_scan_kernel<128, 32, 2, 4, 4, F, ADJ>, 512);
        else if (split == 4) launch(wkv7_f32_scan_kernel<128, 16, 1, 8, 4, F, ADJ>, 768);
        else launch(wkv7_f32_scan_kernel<128, 16, 2, 8, 4, F, ADJ>, 768);
    };
    if (C == 64) width64(std::true_type());
    else if (C < 64) width64(std::false_type());
    else if (C == 128) width128(std::true_type());
    else width128(std::false_type());
}

void launch_wkv7_f32_forward(int B, int T, int H, int C, const float* w, const float* q, const float* k, const float* v,
                             const float* a, const float* b, const float* s0, float* y, float* ckpt, float* sT,
                             hipStream_t stream) {
    launch_scan<false>(B, T, H, C, w, q, k, v, a, b, s0, y, ckpt, sT, stream);
}

void launch_wkv7_f32_backward_split(int B, int T, int H, int C, const float* w, const float* q, const float* k, const float* v,
                                    const float* a, const float* b, const float* dy, const float* ckpt, const float* dsT,
                                    float* work, float* dw, float* dq, float* dk, float* dv, float* da, float* db, float* ds0,
                                    hipStream_t stream) {
    launch_scan<true>(B, T, H, C, w, q, k, dy, a, b, dsT, dv, work, ds0, stream);
    // Blocks of 32 columns, four wavefronts each, while all of them run at once (two to a compute unit, by registers); then a
    // wavefront on 32 columns, up to one per SIMD, where the wait for the matrix instructions of half as many columns counts for
    // more than half the lanes idling; then one on 64.  us in the three forms:
    //   64 channels     64 chunks 11.5, 17.3, 21.6    256 16.8, 19.5, 23.0    320 28.5, 20.4, 24.1    512 31.8, 23.0, 25.7    640 44.2, 33.3, 26.9
    //   128 channels    64 chunks 16.2, 24.3, 32.9    128 20.5, 25.7, 33.7    160 33.6, 26.6, 34.8    256 39.6, 29.4, 36.6    320 52.4, 45.0, 37.7
    //   32 channels     256 chunks 11.0, 14.9         512 15.3, 16.2          640 25.5, 17.0
    const long blocks = (long)B * H * (T / CH64) * ((C + 31) / 32);
    const bool few = blocks <= 2 * compute_units(), narrow = C <= 32 || blocks <= 4 * compute_units();
    auto go = [&](auto kernel, auto narrow_kernel, auto few_kernel) {
        const int cols = few || narrow ? 32 : 64;
        hipLaunchKernelGGL(few ? few_kernel : narrow ? narrow_kernel : kernel, dim3(B * H * (T / CH64), (C + cols - 1) / cols),
                           dim3(few ? 256 : 64), 0, stream, T, H, w, q, k, v, a, b, dy, ckpt, work, dw, dq, dk, da, db);
    };
    switch (C) {
        case 16: go(wkv7_f32_grads_kernel<16, 32>, wkv7_f32_grads_kernel<16, 32>, wkv7_f32_grads_few_kernel<16>); break;
        case 32: go(wkv7_f32_grads_kernel<32, 32>, wkv7_f32_grads_kernel<32, 32>, wkv7_f32_grads_few_kernel<32>); break;
        case 48: go(wkv7_f32_grads_kernel<48, 64>, wkv7_f32_grads_kernel<48, 32>, wkv7_f32_grads_few_kernel<48>); break;
        case 64: go(wkv7_f32_grads_kernel<64, 64>, wkv7_f32_grads_kernel<64, 32>, wkv7_f32_grads_few_kernel<64>); break;
        case 80: go(wkv7_f32_grads_kernel<80, 64>, wkv7_f32_grads_kernel<80, 32>, wkv7_f32_grads_few_kernel<80>); break;
        case 96: go(wkv7_f32_grads_kernel<96, 64>, wkv7_f32_grads_kernel<96, 32>, wkv7_f32_grads_few_kernel<96>); break;
        case 112: go(wkv7_f32_grads_kernel<112, 64>, wkv7_f32_grads_kernel<112, 32>, wkv7_f32_grads_few_kernel<112>); break;
        default: go(wkv7_f32_grads_kernel<128, 64>, wkv7_f32_grads_kernel<128, 32>, wkv7_f32_grads_few_kernel<128>);
    }
}

void launch_wkv7_f32_backward(int B, int T, int H, int C, const float* w, const float* q, const float* k, const float* v,
                              const float* a, const float* b, const float* dy, const float* ckpt, const float* dsT,
                              float* dw, float* dq, float* dk, float* dv, float* da, float* db, float* ds0,
                              hipStream_t stream) {
    const long n4 = (long)B * T * H * C / 4;
    auto z = [](float* p) { return reinterpret_cast<f4*>(p); };
    hipLaunchKernelGGL(zero5_kernel, dim3((unsigned)((n4 + 255) / 256 < 2048 ? (n4 + 255) / 256 : 2048)), dim3(256), 0, stream, n4,
                       z(dq), z(dk), z(db), z(da), z(dw));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(2 * B * H), dim3(256), 0, stream, T, H, C, w, q, k, v, a, b, dy, ckpt, dsT, dw, dq, dk, dv,
                           da, db, ds0);
    };
    if (C == 64) go(wkv7_f32_bwd_thin_kernel<64, 2, 4, 16, true>);
    else if (C < 64) go(wkv7_f32_bwd_thin_kernel<64, 2, 4, 16, false>);
    else if (C == 128) go(wkv7_f32_bwd_thin_kernel<128, 8, 4, 4, true>);
    else go(wkv7_f32_bwd_thin_kernel<128, 8, 4, 4, false>);
}

}  // namespace wkv
