// One token per sequence, or a few, through the whole RWKV-7 time mixer (decoding, short prompts), for gfx950: four launches.
//
// The reference's block has no single-token form: its forward (time_mixer.py:96-167) is the specification, taken at
// T = 1 with the previous token and the WKV7 state carried by the caller.  A step through the sequence kernels is some
// twenty launches of kernels built for thousands of tokens, each waiting out its own launch and drain; here the B
// tokens are the rows of 16-row tiles (rows past B are zero or repeats and never stored) and every stage is a kernel
// whose grid is as wide as the stage's OUTPUT, so the weights (6 MB) stream once through many compute units:
//   1. mid      the token shift's first product with tanh (rwkv7_ddlerp.py:20-49), 16 of its 128 columns per block
//   2. linear   all first-half products (time_mixer.py:120-131) - r, k, v and the six LoRA first halves, nine weight
//               matrices - in one launch; a block computes the interpolated stream (rwkv7_ddlerp.py:53-84) it multiplies
//               itself, 32 channels at a time, so the four streams never exist in memory (for many rows they do, a launch
//               more: `streams_in_memory`)
//   3. head     per (tile, head): the LoRA second halves with the elementwise tail (rwkv7_expand_loras.py:33-70), the gate's
//               and the decay's second halves, then the single-token WKV7 recurrence with GroupNorm, bonus and gate
//   4. linear   the output projection
// Rounding follows the sequence path: every tensor that path keeps in bf16 between its kernels is rounded to bf16
// here at the same place.
//
// At B = 1 every stage is bound by its launch, one trip to memory and its drain, so what counts is how few stages there
// are and that no stage leaves its loads to a few compute units.  (Five stages with the whole token shift in the ONE
// block of the tile: 18.4 us for that block to fetch 400 KB, 39.8 us per step at 768 channels.)
#include "mixer_decode_kernels.hpp"

#include "device_info.hpp"
#include "linear_kernels.hpp"
#include "row_lines.hpp"
#include "ln_epilogue.hpp"
#include "wkv7_common.hpp"

namespace wkv {

namespace {

constexpr int TOK = 16;
// LoRA ranks of the block (time_mixer.py:42-104)
constexpr int R_MIX = 32, R_DECAY = 64, R_AAA = 16, R_KKK = 16, R_GATE = 128, R_MA = 16, R_MK = 16;

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
__device__ __forceinline__ bf16x4 lo4(bf16x8 v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3); }
__device__ __forceinline__ bf16x4 hi4(bf16x8 v) { return __builtin_shufflevector(v, v, 4, 5, 6, 7); }
__device__ __forceinline__ bf16x8 cat8(bf16x4 a, bf16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// In every 32-wide product below a lane group g holds contraction indices 8g .. 8g+7 of BOTH operands (one 16-byte
// load each): the order of the summed index is free as long as the operands agree.

// ------------------------------------------------------------------------------------------------
// 1. mid = tanh((x + xx alpha) L^T),  xx = x_prev - x.  Block = 16 of the 128 columns x one 16-row tile; its NW wavefronts
// take every NW-th 64-channel step of the contraction, weights and tokens as whole lines through LDS; us, fragments straight from
// memory -> so: 768 channels, one sequence 4.9 -> 4.9, 32 5.9 -> 5.1, 256 6.4 -> 5.4; 2048 channels, 16 sequences 9.6 -> 6.6.
// ------------------------------------------------------------------------------------------------
constexpr int MID = 4 * R_MIX;

struct MixIn {   // the token shift's operands
    const __bf16 *x, *x_prev;   // [B*T, C]; [B, C], the tokens before the sequences' first (null: zeros)
    const __bf16 *R, *beta;     // [4, C, 32], [4, C]
    __bf16* mid;                // [rows padded to 16, 128]
    int rows, T;                // B*T, tokens per sequence
};
// A lane's row of x (a row past the last repeats it) and the row before it; at a sequence's start without x_prev the row
// itself is loaded and `zero` says to take zeros.
struct TokenRows {
    long at, prev;         // element offsets: into x, and into x or x_prev
    const __bf16* prev_of;
    bool zero;
};
__device__ __forceinline__ TokenRows token_rows(const MixIn& in, int row, int C) {
    const int m = row < in.rows ? row : in.rows - 1;
    const int seq = in.T == 1 ? m : m / in.T;   // (a division is 40 instructions at the head of a launch that is all latency)
    TokenRows r;
    r.at = (long)m * C;
    const bool start = m == seq * in.T;
    r.zero = start && in.x_prev == nullptr;
    r.prev_of = start && in.x_prev != nullptr ? in.x_prev : in.x;
    r.prev = start ? (in.x_prev != nullptr ? (long)seq * C : r.at) : r.at - C;
    return r;
}
__device__ __forceinline__ bf16x8 or_zero(bf16x8 v, bool zero) { return zero ? bf16x8{} : v; }

template <int NW, int U>   // wavefronts, and steps of a wavefront in flight at a time
__global__ __launch_bounds__(64 * NW) void decode_mid_kernel(const MixIn in, int C, const __bf16* __restrict__ alpha,
                                                         const __bf16* __restrict__ Lw, __bf16* __restrict__ x_carry) {
    constexpr int AREAS = NW <= 4 ? U : 1;   // all of a round written before the first is read, where there is room
    struct Image {   // of a wavefront's 64 channels, pieces of rows (piece_slot): the weights; the input, hi and lo
        bf16x8 w[TOK * 8], a[2][TOK * 8];
    };
    __shared__ union {
        Image img[NW][AREAS];
        f32x4 part[NW][WAVE];
    } lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l8 = lane >> 3, piece = lane & 7;
    const Lane L;
    const int ob = blockIdx.x, row = blockIdx.y * TOK + L.n;
    const __bf16 *xrow[2], *prow[2];
    bool zero[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const TokenRows tr = token_rows(in, blockIdx.y * TOK + l8 + 8 * i, C);
        xrow[i] = in.x + tr.at + 8 * piece;
        prow[i] = tr.prev_of + tr.prev + 8 * piece;
        zero[i] = tr.zero;
    }
    const unsigned w_bytes = 2 * ((unsigned)l8 * C + 8 * piece), w_rows8 = 16 * (unsigned)C;
    f32x4 acc0 = zero4(), acc1 = zero4();
    const int nk = C / 64;
    for (int s0 = wave; s0 < nk; s0 += NW * U) {   // U steps of this wavefront at a time, all loads before the products
        bf16x8 xc[U][2], xp[U][2], al[U], lw[U][2];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = 64 * (s0 + NW * u < nk ? s0 + NW * u : s0);   // (past the end: the first step again, not used)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                xc[u][i] = *reinterpret_cast<const bf16x8*>(xrow[i] + c);
                xp[u][i] = *reinterpret_cast<const bf16x8*>(prow[i] + c);
                lw[u][i] = piece_at(Lw + (long)16 * ob * C + c, w_bytes + i * w_rows8);
            }
            al[u] = *reinterpret_cast<const bf16x8*>(alpha + c + 8 * piece);
        }
        __builtin_amdgcn_sched_barrier(0);
        auto park = [&](int u) {
            Image& mine = lds.img[wave][u % AREAS];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                // the interpolated input as a bf16 pair (hi + lo), as the sequence kernel has it: it feeds tanh', which
                // is steep, and must not be rounded to 8 bits before the C-term sum
                bf16x4 h[2], l[2];
                const bf16x8 p8 = or_zero(xp[u][i], zero[i]);
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const f32x4 cv = to_f32(half_of(xc[u][i], hf));
                    const f32x4 av = cv + (to_f32(half_of(p8, hf)) - cv) * to_f32(half_of(al[u], hf));
                    h[hf] = to_bf16(av);
                    l[hf] = to_bf16(av - to_f32(h[hf]));
                }
                const int slot = piece_slot(l8 + 8 * i, piece);
                mine.w[slot] = lw[u][i];
                mine.a[0][slot] = join(h[0], h[1]);
                mine.a[1][slot] = join(l[0], l[1]);
            }
        };
        if constexpr (AREAS == U) {
#pragma unroll
            for (int u = 0; u < U; u++) park(u);
            wave_lds_order();
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + NW * u >= nk) break;
            if constexpr (AREAS != U) {
                park(u);
                wave_lds_order();
            }
            const Image& mine = lds.img[wave][u % AREAS];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int slot = piece_slot(L.n, 4 * i + L.g);
                const bf16x8 wf = mine.w[slot];            // lane = mid index
                acc0 = mma8(acc0, wf, mine.a[0][slot]);   // lane = token
                acc1 = mma8(acc1, wf, mine.a[1][slot]);
            }
            if constexpr (AREAS != U) wave_lds_order();
        }
        wave_lds_order();
    }
    __syncthreads();
    lds.part[wave][lane] = acc0 + acc1;
    // the tokens to hand on, the last of each sequence: dealt over all blocks
    if (x_carry) {
        const int per_row = C / 8, nseq = in.rows / in.T;
        const int step = gridDim.x * gridDim.y * 64 * NW;
        for (int v = (blockIdx.y * gridDim.x + ob) * 64 * NW + threadIdx.x; v < nseq * per_row; v += step) {
            const int seq = v / per_row, c = 8 * (v - seq * per_row);
            *reinterpret_cast<bf16x8*>(x_carry + (long)seq * C + c) =
                *reinterpret_cast<const bf16x8*>(in.x + ((long)seq * in.T + in.T - 1) * C + c);
        }
    }
    __syncthreads();
    if (wave != 0) return;
    f32x4 t = lds.part[0][lane];   // lane = token, reg = column 4g + r
#pragma unroll
    for (int w = 1; w < NW; w++) t += lds.part[w][lane];
#pragma unroll
    for (int r = 0; r < 4; r++) t[r] = tanhf_(t[r]);
    *reinterpret_cast<bf16x4*>(in.mid + (long)row * MID + 16 * ob + 4 * L.g) = to_bf16(t);
}

// The four interpolated streams y_k = x + xx (mid_k R_k^T + beta_k) in memory, for the products of many rows: block = 32
// channels x one 16-row tile, a wavefront per stream.
__global__ __launch_bounds__(256) void decode_lerp_kernel(const MixIn in, int C, __bf16* __restrict__ y, long stream_stride) {
    const int ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane L;
    const int row = blockIdx.y * TOK + L.n, c = 32 * blockIdx.x + 8 * L.g;
    const TokenRows tr = token_rows(in, row, C);
    const bf16x8 bm = *reinterpret_cast<const bf16x8*>(in.mid + (long)row * MID + R_MIX * ks + 8 * L.g);
    // row j of the two R fragments: channel 8(n/4) + 4j + n%4, so that the products are the lane's eight channels 8g .. 8g+7
    const __bf16* rrow = in.R + ((long)ks * C + 32 * blockIdx.x + 8 * (L.n >> 2) + (L.n & 3)) * R_MIX + 8 * L.g;
    const bf16x8 r0 = *reinterpret_cast<const bf16x8*>(rrow), r1 = *reinterpret_cast<const bf16x8*>(rrow + 4 * R_MIX);
    const bf16x8 be = *reinterpret_cast<const bf16x8*>(in.beta + (long)ks * C + c);
    const bf16x8 xv = *reinterpret_cast<const bf16x8*>(in.x + tr.at + c);
    const bf16x8 pv = or_zero(*reinterpret_cast<const bf16x8*>(tr.prev_of + tr.prev + c), tr.zero);
    const f32x4 c0 = mma8(to_f32(lo4(be)), r0, bm), c1 = mma8(to_f32(hi4(be)), r1, bm);   // lane = token
    const f32x4 x0 = to_f32(lo4(xv)), x1 = to_f32(hi4(xv));
    if (row < in.rows)
        *reinterpret_cast<bf16x8*>(y + ks * stream_stride + (long)row * C + c) =
            cat8(to_bf16(x0 + (to_f32(lo4(pv)) - x0) * c0), to_bf16(x1 + (to_f32(hi4(pv)) - x1) * c1));
}

// ------------------------------------------------------------------------------------------------
// 2./4. linear: out_s = in_s W_s^T for up to nine (input, weight) pairs.  Block = CB x 16 output columns of one pair
// x RT 16-row tiles; its four wavefronts take every fourth 64-channel step of the contraction.  The weights arrive as whole
// lines and pass through LDS (16 rows per instruction, as fragments lie, cost a compute unit three times the lookups; us, six first-half pairs / output
// projection, then -> now: 768 channels, one sequence 5.8 / 3.8 -> 5.7 / 3.4, 32 10.1 / 3.7 -> 9.0 / 3.6, 64 11.3 / 4.0 -> 10.5 / 3.9; 2048
// channels, 16 sequences 20.7 / 6.4 -> 18.8 / 5.2).  LERP: the input is the
// pair's token-shifted stream y_k = x + xx (mid_k R_k^T + beta_k), made 32 channels at a time where it is multiplied (one
// row of R per lane, ordered so that the two 16-channel results are the lane's eight contiguous channels 8g .. 8g+7).
// Every column block repeats that for its stream, so few columns per block where the launch is latency (a tile or two),
// four and two tiles at a time where the work counts.
// ------------------------------------------------------------------------------------------------
struct alignas(32) LinSeg {
    const __bf16* W;     // [N, C]
    __bf16* out;         // [rows, N]
    int N;               // multiple of 16
    int tanh_out;        // the output is tanh of the (bf16-rounded) product
    int stream;          // LERP: which interpolation
};
constexpr int MAX_SEGS = 9;
typedef int i32x16 __attribute__((ext_vector_type(16), aligned(32)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int mix_words8 __attribute__((ext_vector_type(8), aligned(8)));   // (as a MixIn lies)
typedef int mix_words4 __attribute__((ext_vector_type(4), aligned(8)));
// As many pairs as a launch has, and beside them only the input that it reads: the host writes a kernel's arguments anew for every
// launch, and that bounds a step of few sequences (12 heads, one sequence, called eagerly, a process at the lower or the higher of the two
// speeds at which the host runs: with 496 bytes for either kernel 19.5 or 17.4 us, with 400 and 104 19.3 or 17.1; replayed 16.7, 16.5).
template <int SEGS>
struct LinArgs {
    i32x16 plan;   // of the launch: blocks of each pair (0 past the last one); PLAN_C and so on
    LinSeg seg[SEGS];
};
template <bool LERP>
using LinInput = std::conditional_t<LERP, MixIn, const __bf16*>;   // what is interpolated; else [Bp, C]

enum { PLAN_C = 13, PLAN_ROWS, PLAN_TILES };   // rows: output rows that exist (stores beyond are dropped)
static_assert(MAX_SEGS <= PLAN_C && sizeof(LinSeg) == 32 && sizeof(MixIn) == 48, "what the kernel below takes into scalar registers");
static_assert(alignof(i32x8) <= alignof(LinSeg) && alignof(mix_words8) <= alignof(MixIn) && alignof(mix_words4) <= alignof(MixIn), "what is read as such");

template <class T>
__device__ __forceinline__ T* global_pointer(int lo, int hi) {   // (an address that the compiler has lost sight of, to global memory all the same)
    return (T*)(__attribute__((address_space(1))) T*)((unsigned long)(unsigned)lo | (unsigned long)(unsigned)hi << 32);
}

template <bool LERP, int CB, int RT>
__global__ __launch_bounds__(256) void decode_linear_kernel(const LinArgs<LERP ? MAX_SEGS : 1> A, const LinInput<LERP> input) {
    constexpr int NW = 4, SEGS = LERP ? MAX_SEGS : 1;
    constexpr int U = CB * RT == 1 ? 3 : CB * RT <= 4 ? 2 : 1;   // steps of a wavefront in flight
    // R too passes through LDS where there are several column blocks: its fragments touch two lines per four lanes, not four, and
    // a launch that is all latency pays the way (one sequence 6.1 us instead of 5.7; 64 sequences 10.5 instead of 10.9).
    constexpr bool R_LINES = LERP && CB > 1;
    constexpr int AREAS = CB * RT == 1 ? U : 1;                 // (latency: all of them written before the first is read)
    struct Weights {   // of a wavefront's 64 channels: W as pieces of rows (piece_slot), R as rows of four pieces (r_slot)
        bf16x8 w[CB][16 * 8], r[R_LINES ? 64 * 4 : 1];
    };
    __shared__ union {
        Weights weights[NW][AREAS];
        f32x4 part[NW][RT][CB][WAVE];
    } lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l8 = lane >> 3, piece = lane & 7;
    const Lane L;
    // Which pair this block belongs to.  The plan and the token shift's operands come in one cluster of scalar loads, then the pair's
    // own in another: left to the compiler each is loaded where it is looked at, a chain of twelve before the first load of a weight
    // (a replayed step of 12 heads, 1, 16, 64, 128 sequences 16.9, 19.1, 25.4, 32.0 -> 16.6, 18.7, 24.6, 31.2 us).
    i32x16 plan = A.plan;
    MixIn mix{};
    const __bf16* in = nullptr;
    if constexpr (LERP) {
        mix_words8 m8 = *reinterpret_cast<const mix_words8*>(&input);
        mix_words4 m4 = *reinterpret_cast<const mix_words4*>(&input.mid);
        asm volatile("" : "+s"(plan), "+s"(m8), "+s"(m4));
        mix = {global_pointer<const __bf16>(m8[0], m8[1]), global_pointer<const __bf16>(m8[2], m8[3]), global_pointer<const __bf16>(m8[4], m8[5]),
               global_pointer<const __bf16>(m8[6], m8[7]), global_pointer<__bf16>(m4[0], m4[1]), m4[2], m4[3]};
    } else {
        unsigned long at = (unsigned long)input;
        asm volatile("" : "+s"(plan), "+s"(at));
        in = global_pointer<const __bf16>(at, at >> 32);
    }
    int blk = blockIdx.x, pair = -1, col_block = 0;
#pragma unroll
    for (int i = 0; i < SEGS; i++) {
        const bool found = pair < 0 && blk < plan[i];
        pair = found ? i : pair, col_block = found ? blk : col_block;
        blk -= plan[i];
    }
    if (pair < 0) return;   // (whole block; the grid is exactly the sum of the pairs' blocks)
    i32x8 s8 = *reinterpret_cast<const i32x8*>(&A.seg[pair]);
    asm volatile("" : "+s"(s8));
    const __bf16* __restrict__ W = global_pointer<const __bf16>(s8[0], s8[1]);
    __bf16* __restrict__ out = global_pointer<__bf16>(s8[2], s8[3]);
    const int N = s8[4], act = s8[5], ks = s8[6], C = plan[PLAN_C], rows = plan[PLAN_ROWS], ntiles = plan[PLAN_TILES];
    const int col0 = 16 * CB * col_block;
    int trow[RT];       // this lane's row of each tile (a tile past the last repeats it and is not stored)
    const __bf16 *irow[RT], *prow[RT];
    bf16x8 bm[RT];
    bool zero[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int tile = blockIdx.y * RT + t < (unsigned)ntiles ? blockIdx.y * RT + t : ntiles - 1;
        trow[t] = tile * TOK + L.n;
        if constexpr (LERP) {
            const TokenRows tr = token_rows(mix, trow[t], C);
            irow[t] = mix.x + tr.at + 8 * L.g;
            prow[t] = tr.prev_of + tr.prev + 8 * L.g;
            zero[t] = tr.zero;
            bm[t] = *reinterpret_cast<const bf16x8*>(mix.mid + (long)trow[t] * MID + R_MIX * ks + 8 * L.g);
        } else {
            irow[t] = in + (long)trow[t] * C + 8 * L.g;
        }
    }
    const __bf16* wcol[CB];   // the column blocks' first rows of W
#pragma unroll
    for (int cb = 0; cb < CB; cb++) wcol[cb] = W + (long)(col0 + 16 * cb < N ? col0 + 16 * cb : col0) * C;
    const unsigned w_bytes = 2 * ((unsigned)l8 * C + 8 * piece), w_rows8 = 16 * (unsigned)C;
    // row j of a 32-channel step's two R fragments: channel 8(n/4) + 4j + n%4
    const __bf16* rrow = LERP ? mix.R + ((long)ks * C + (R_LINES ? 0 : 8 * (L.n >> 2) + (L.n & 3))) * R_MIX + (R_LINES ? 8 * lane : 8 * L.g) : nullptr;
    // in LDS sixteen such rows' pieces lie in different banks of 16 bytes
    auto r_slot = [](int channel, int p) { return 4 * channel + (p ^ (channel >> 3 & 3)); };
    const __bf16* brow = LERP ? mix.beta + (long)ks * C + 8 * L.g : nullptr;
    f32x4 acc[RT][CB];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) acc[t][cb] = zero4();
    const int nk = C / 64;
    for (int s0 = wave; s0 < nk; s0 += NW * U) {   // U steps of this wavefront at a time, all loads before the products
        bf16x8 wv[U][CB][2], iv[U][RT][2], pv[U][RT][2], rv[U][4], be[U][2];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = 64 * (s0 + NW * u < nk ? s0 + NW * u : s0);   // (past the end: the first step again, not used)
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
#pragma unroll
                for (int i = 0; i < 2; i++) wv[u][cb][i] = piece_at(wcol[cb] + c, w_bytes + i * w_rows8);
#pragma unroll
            for (int t = 0; t < RT; t++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    iv[u][t][i] = *reinterpret_cast<const bf16x8*>(irow[t] + c + 32 * i);
                    if constexpr (LERP) pv[u][t][i] = *reinterpret_cast<const bf16x8*>(prow[t] + c + 32 * i);
                }
            if constexpr (LERP) {
#pragma unroll
                for (int i = 0; i < 4; i++) rv[u][i] = *reinterpret_cast<const bf16x8*>(rrow + (long)(c + (R_LINES ? 16 * i : 32 * (i >> 1) + 4 * (i & 1))) * R_MIX);
#pragma unroll
                for (int i = 0; i < 2; i++) be[u][i] = *reinterpret_cast<const bf16x8*>(brow + c + 32 * i);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        auto park = [&](int u) {
            Weights& mine = lds.weights[wave][u % AREAS];
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
#pragma unroll
                for (int i = 0; i < 2; i++) mine.w[cb][piece_slot(l8 + 8 * i, piece)] = wv[u][cb][i];
            if constexpr (R_LINES) {
#pragma unroll
                for (int i = 0; i < 4; i++) mine.r[r_slot(16 * i + (lane >> 2), lane & 3)] = rv[u][i];
            }
        };
        if constexpr (AREAS == U) {
#pragma unroll
            for (int u = 0; u < U; u++) park(u);
            wave_lds_order();
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + NW * u >= nk) break;
            if constexpr (AREAS != U) {
                park(u);
                wave_lds_order();
            }
            const Weights& mine = lds.weights[wave][u % AREAS];
#pragma unroll
            for (int i = 0; i < 2; i++) {   // 32 channels
                bf16x8 wf[CB], r0 = rv[u][2 * i], r1 = rv[u][2 * i + 1];
                if constexpr (R_LINES) {
                    const int channel = 32 * i + 8 * (L.n >> 2) + (L.n & 3);
                    r0 = mine.r[r_slot(channel, L.g)], r1 = mine.r[r_slot(channel + 4, L.g)];
                }
#pragma unroll
                for (int cb = 0; cb < CB; cb++) wf[cb] = mine.w[cb][piece_slot(L.n, 4 * i + L.g)];
#pragma unroll
                for (int t = 0; t < RT; t++) {
                    bf16x8 in8 = iv[u][t][i];
                    if constexpr (LERP) {
                        const f32x4 c0 = mma8(to_f32(lo4(be[u][i])), r0, bm[t]);   // lane = token, channels 8g + r
                        const f32x4 c1 = mma8(to_f32(hi4(be[u][i])), r1, bm[t]);   // channels 8g + 4 + r
                        const bf16x8 p8 = or_zero(pv[u][t][i], zero[t]);
                        const f32x4 x0 = to_f32(lo4(in8)), x1 = to_f32(hi4(in8));
                        in8 = cat8(to_bf16(x0 + (to_f32(lo4(p8)) - x0) * c0), to_bf16(x1 + (to_f32(hi4(p8)) - x1) * c1));
                    }
#pragma unroll
                    for (int cb = 0; cb < CB; cb++) acc[t][cb] = mma8(acc[t][cb], wf[cb], in8);
                }
            }
            if constexpr (AREAS != U) wave_lds_order();
        }
        wave_lds_order();
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) lds.part[wave][t][cb][lane] = acc[t][cb];
    __syncthreads();
    for (int o = wave; o < RT * CB; o += NW) {   // a wavefront finishes a 16 x 16 result
        const int t = o / CB, cb = o % CB;
        f32x4 r = lds.part[0][t][cb][lane];   // lane = token, reg = column 4g + r
#pragma unroll
        for (int w = 1; w < NW; w++) r += lds.part[w][t][cb][lane];
        if (act) {
            r = to_f32(to_bf16(r));
#pragma unroll
            for (int q = 0; q < 4; q++) r[q] = tanhf_(r[q]);
        }
        const int row = (blockIdx.y * RT + t) * TOK + L.n;
        if (row < rows && col0 + 16 * cb < N) *reinterpret_cast<bf16x4*>(out + (long)row * N + col0 + 16 * cb + 4 * L.g) = to_bf16(r);
    }
}

// ------------------------------------------------------------------------------------------------
// 3. head: per head of 64 channels and 16 tokens, by four wavefronts (16 channels each)
//     g  = tanh(g1) Wg2^T ;   w2 = tanh(w1) Ww2^T ;   w = -softplus(-(w_bias + w2)) - 0.5
//     z  = tanh(kk1) Wz^T + k ;   kk = z / sqrt(max(sum_head z^2, 1e-12))
//     a  = sigmoid(a1 Wa^T + a_bias) ;  ma, mk likewise ;   k' = k (ma + a - ma a) exp(w mk) ;   b = -kk a
// with the results as bf16 in LDS (the decay exp(-exp(w)) of the rounded w in fp32); then per token, a wavefront per 16 value
// rows of the state,
//     sa = S kk ;   S <- S diag(exp(-exp(w))) + sa b^T + v k'^T ;   y = S r ;   out = g (groupnorm(y) + (sum r k' bonus) v)
// ------------------------------------------------------------------------------------------------
struct HeadArgs {
    int rows, T, C, H, state_f32;                                         // rows = B*T
    const __bf16 *r, *k, *v;                                              // [rows padded to 16, C]
    const __bf16 *tg1, *tw1, *kk1, *mk1, *a1, *ma1;                       // likewise x 128, 64, 4 times 16
    const __bf16 *gate_w2, *decay_w2, *kkk_w2, *aaa_w2, *ma_w2, *mk_w2;   // [C, rank]
    const __bf16 *time_decay, *time_aaaaa, *time_misc_a, *time_misc_k;   // [C]
    const float* ln_params;                                               // [3, C]
    const void* state_in;                                                 // [B, H, 64, 64], null: zeros
    void* state;                                                          // may be state_in itself
    __bf16* ya;                                                           // [rows padded to 16, C]
};
struct HeadTile {   // 16 tokens of a head
    static constexpr int LD = HEAD + 8, LF = HEAD + 4;   // (row pitches: 16 bytes off a multiple of the bank width)
    __attribute__((aligned(16))) __bf16 r[TOK][LD], v[TOK][LD], k[TOK][LD], kk[TOK][LD], b[TOK][LD], g[TOK][LD];
    __attribute__((aligned(16))) float decay[TOK][LF];
    float ss[NBLK][TOK], y[TOK][HEAD];
};

// The tile's operands into LDS: token n of the tile is row first + n (past `last`: row `last` again).  The first 256 threads
// load r and v, the first four wavefronts expand; every wavefront of the block takes part in the barriers.
__device__ __forceinline__ void expand_tile(HeadTile& s, const HeadArgs& A, int h, int first, int last, int wave, const Lane& L) {
    const int C = A.C, ib = wave & 3;
    if (threadIdx.x < 256) {   // 16 bytes per thread
        const int t = threadIdx.x & 127, n = t >> 3, c = 8 * (t & 7);
        const __bf16* src = threadIdx.x < 128 ? A.r : A.v;
        __bf16(*dst)[HeadTile::LD] = threadIdx.x < 128 ? s.r : s.v;
        *reinterpret_cast<bf16x8*>(&dst[n][c]) =
            *reinterpret_cast<const bf16x8*>(src + (long)(first + n < last ? first + n : last) * C + h * HEAD + c);
    }
    f32x4 z, av;
    if (wave < 4) {
        const int row = first + L.n < last ? first + L.n : last, c = h * HEAD + 16 * ib;   // lane n: token as an operand's row; channel c + n as a weight row
        bf16x8 tg1[R_GATE / 32], tw1[R_DECAY / 32], gw[R_GATE / 32], dw[R_DECAY / 32];
        // every load before the first product (else each weight fragment is loaded right before its use and waited for)
#pragma unroll
        for (int j = 0; j < R_GATE / 32; j++) {
            tg1[j] = *reinterpret_cast<const bf16x8*>(A.tg1 + (long)row * R_GATE + 32 * j + 8 * L.g);
            gw[j] = *reinterpret_cast<const bf16x8*>(A.gate_w2 + (long)(c + L.n) * R_GATE + 32 * j + 8 * L.g);
        }
#pragma unroll
        for (int j = 0; j < R_DECAY / 32; j++) {
            tw1[j] = *reinterpret_cast<const bf16x8*>(A.tw1 + (long)row * R_DECAY + 32 * j + 8 * L.g);
            dw[j] = *reinterpret_cast<const bf16x8*>(A.decay_w2 + (long)(c + L.n) * R_DECAY + 32 * j + 8 * L.g);
        }
        auto act16 = [&](const __bf16* p) { return *reinterpret_cast<const bf16x4*>(p + (long)row * 16 + 4 * L.g); };
        auto w16 = [&](const __bf16* W) { return *reinterpret_cast<const bf16x4*>(W + (long)(c + L.n) * 16 + 4 * L.g); };
        auto bias4 = [&](const __bf16* p) { return *reinterpret_cast<const bf16x4*>(p + c + 4 * L.g); };
        const bf16x4 kk1 = act16(A.kk1), a1 = act16(A.a1), ma1 = act16(A.ma1), mk1 = act16(A.mk1);
        const bf16x4 wz = w16(A.kkk_w2), wa = w16(A.aaa_w2), wma = w16(A.ma_w2), wmk = w16(A.mk_w2);
        const bf16x4 bd = bias4(A.time_decay), ba = bias4(A.time_aaaaa), bma = bias4(A.time_misc_a), bmk = bias4(A.time_misc_k);
        const bf16x4 kq = *reinterpret_cast<const bf16x4*>(A.k + (long)row * C + c + 4 * L.g);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 t = to_f32(kk1);
#pragma unroll
        for (int q = 0; q < 4; q++) t[q] = tanhf_(t[q]);
        f32x4 gacc = zero4(), w2 = zero4();
#pragma unroll
        for (int j = 0; j < R_GATE / 32; j++) gacc = mma8(gacc, gw[j], tg1[j]);
#pragma unroll
        for (int j = 0; j < R_DECAY / 32; j++) w2 = mma8(w2, dw[j], tw1[j]);
        const f32x4 kin = to_f32(kq);
        z = mma(kin, wz, to_bf16(t));
        const f32x4 pa = mma(to_f32(ba), wa, a1), pma = mma(to_f32(bma), wma, ma1), pmk = mma(to_f32(bmk), wmk, mk1);
        const f32x4 u = to_f32(bd) + to_f32(to_bf16(w2));   // (w2 is a bf16 tensor in the sequence path)
        f32x4 w, k;
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float a = sigmoidf_(pa[q]), ma = sigmoidf_(pma[q]), mk = sigmoidf_(pmk[q]);
            w[q] = -(fmaxf(-u[q], 0.f) + log1pexp_(u[q])) - 0.5f;
            k[q] = kin[q] * (ma + a - ma * a) * __expf(w[q] * mk);
            av[q] = a;
            ss += z[q] * z[q];
        }
        f32x4 d = to_f32(to_bf16(w));
#pragma unroll
        for (int q = 0; q < 4; q++) d[q] = __expf(-__expf(d[q]));
        const int at = 16 * ib + 4 * L.g;
        *reinterpret_cast<bf16x4*>(&s.g[L.n][at]) = to_bf16(gacc);
        *reinterpret_cast<f32x4*>(&s.decay[L.n][at]) = d;
        *reinterpret_cast<bf16x4*>(&s.k[L.n][at]) = to_bf16(k);
        ss = group_sum(ss);
        if (L.g == 0) s.ss[ib][L.n] = ss;
    }
    lds_barrier();
    if (wave < 4) {
        const float inorm = rsqrtf(fmaxf((s.ss[0][L.n] + s.ss[1][L.n]) + (s.ss[2][L.n] + s.ss[3][L.n]), 1e-12f));
        const f32x4 kk = z * inorm;
        const int at = 16 * ib + 4 * L.g;
        *reinterpret_cast<bf16x4*>(&s.kk[L.n][at]) = to_bf16(kk);
        *reinterpret_cast<bf16x4*>(&s.b[L.n][at]) = to_bf16(-kk * av);
    }
    lds_barrier();
}

// A wavefront's sixteen value rows of the state, 16 ib ..: register i of lane (n, g) is columns 4n .. 4n + 3 of row 4i + g, so that
// a load or store is 1 KiB in one piece and a token's vectors are four channels per lane.  (As the fragments of the sequence
// kernels, four lanes to a row and sixteen columns each, every access touched sixteen rows, 28 ns of a compute unit's time
// instead of 9 to load and 20 to store, the vectors were four times the LDS reads, and the sums over a row went through the LDS
// crossbar: the head kernel of a step at 768 channels and 1, 32, 256, 512 sequences 6.9, 9.4, 25.4, 38.8 -> 5.9, 7.7, 20.5, 35.8
// us, where the states of 256 sequences are 100 MB to move, 20 us at the rate of a copy.)
__device__ __forceinline__ void load_state(f32x4 (&S)[NBLK], const void* s, int state_f32, int bh, int ib, const Lane& L) {
    const long off = ((long)bh * HEAD + 16 * ib + L.g) * HEAD + 4 * L.n;
#pragma unroll
    for (int i = 0; i < NBLK; i++) {
        if (s == nullptr) S[i] = zero4();
        else if (state_f32) S[i] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(s) + off + 4 * i * HEAD);
        else S[i] = to_f32(*reinterpret_cast<const bf16x4*>(static_cast<const __bf16*>(s) + off + 4 * i * HEAD));
    }
}
template <bool THROUGH = false>   // a float32 state through the L2 (store_through_at)
__device__ __forceinline__ void store_state(const f32x4 (&S)[NBLK], void* s, int state_f32, int bh, int ib, const Lane& L) {
    if (s == nullptr) return;
    const int in_head = (16 * ib + L.g) * HEAD + 4 * L.n;
    const long head = (long)bh * HEAD * HEAD, off = head + in_head;
#pragma unroll
    for (int i = 0; i < NBLK; i++) {
        if (THROUGH && state_f32) store_through_at(static_cast<float*>(s) + head, 4 * (in_head + 4 * i * HEAD), S[i]);
        else if (state_f32) *reinterpret_cast<f32x4*>(static_cast<float*>(s) + off + 4 * i * HEAD) = S[i];
        else *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(s) + off + 4 * i * HEAD) = to_bf16(S[i]);
    }
}
// a lane's part of a token's vectors: its four columns, and of v its four rows
struct TokenVectors {
    bf16x4 kk, b, k, r;
    f32x4 decay;
    __bf16 v[NBLK];
};
__device__ __forceinline__ TokenVectors token_vectors(const HeadTile& s, int n, int ib, const Lane& L) {
    TokenVectors t;
    auto vec = [&](const __bf16 (&a)[TOK][HeadTile::LD]) { return *reinterpret_cast<const bf16x4*>(&a[n][4 * L.n]); };
    t.kk = vec(s.kk), t.b = vec(s.b), t.k = vec(s.k), t.r = vec(s.r);
    t.decay = *reinterpret_cast<const f32x4*>(&s.decay[n][4 * L.n]);
#pragma unroll
    for (int i = 0; i < NBLK; i++) t.v[i] = s.v[n][16 * ib + 4 * i + L.g];
    return t;
}
// token n of the tile on a wavefront's rows of the state; y goes to LDS
__device__ __forceinline__ void update_state(HeadTile& s, f32x4 (&S)[NBLK], const TokenVectors& t, int n, int ib, const Lane& L) {
    const f32x4 a = to_f32(t.kk), b = to_f32(t.b), k = to_f32(t.k), r = to_f32(t.r), d = t.decay;
    float sa[NBLK], y[NBLK];
#pragma unroll
    for (int i = 0; i < NBLK; i++) sa[i] = (S[i][0] * a[0] + S[i][1] * a[1]) + (S[i][2] * a[2] + S[i][3] * a[3]);
#pragma unroll
    for (int i = 0; i < NBLK; i++) sa[i] = row_sum(sa[i]);   // over the sixteen lanes that share the state's row
#pragma unroll
    for (int i = 0; i < NBLK; i++) {
        const float vrow = (float)t.v[i];
#pragma unroll
        for (int q = 0; q < 4; q++) S[i][q] = S[i][q] * d[q] + sa[i] * b[q] + vrow * k[q];
        y[i] = (S[i][0] * r[0] + S[i][1] * r[1]) + (S[i][2] * r[2] + S[i][3] * r[3]);
    }
#pragma unroll
    for (int i = 0; i < NBLK; i++) y[i] = row_sum(y[i]);
    const float out = L.n < 2 ? (L.n == 0 ? y[0] : y[1]) : (L.n == 2 ? y[2] : y[3]);   // lanes n < 4: row 4n + g
    if (L.n < NBLK) s.y[n][16 * ib + 4 * L.n + L.g] = out;
}
// tokens 0 .. n - 1 of the tile one after the other, the next one's vectors on their way
__device__ __forceinline__ void update_tokens(HeadTile& s, f32x4 (&S)[NBLK], int n, int ib, const Lane& L) {
    TokenVectors t = token_vectors(s, 0, ib, L);
    for (int i = 0; i < n; i++) {
        const TokenVectors next = token_vectors(s, i + 1 < n ? i + 1 : i, ib, L);
        update_state(s, S, t, i, ib, L);
        t = next;
    }
}

// GroupNorm, bonus and gate of tokens first, first + step, .. below end, lane = channel; row(n): token n's row of the output.
// AT_ONCE at a time: a token is three sums over the wavefront, two of them one after the other.
template <int AT_ONCE, class Row>
__device__ __forceinline__ void finish_tokens(const HeadTile& s, const float* ln_params, int C, int h, int first, int step, int end, int lane,
                                              Row row) {
    auto head_sum = [](float x) {
        x = row_sum(x);
        return group_sum(x);
    };
    const float* lp = ln_params + h * HEAD + lane;
    const float scale = lp[0], shift = lp[C], bonus = lp[2 * (long)C];
    for (int n0 = first; n0 < end; n0 += AT_ONCE * step) {
        int n[AT_ONCE];
        float y[AT_ONCE], mean[AT_ONCE], var[AT_ONCE], dot[AT_ONCE];
#pragma unroll
        for (int j = 0; j < AT_ONCE; j++) {
            n[j] = n0 + j * step < end ? n0 + j * step : n0;   // (past the last: the first again, not stored)
            y[j] = s.y[n[j]][lane];
            mean[j] = head_sum(y[j]) * (1.f / HEAD);
            dot[j] = head_sum((float)s.r[n[j]][lane] * (float)s.k[n[j]][lane] * bonus);
        }
#pragma unroll
        for (int j = 0; j < AT_ONCE; j++) var[j] = head_sum((y[j] - mean[j]) * (y[j] - mean[j])) * (1.f / HEAD);
#pragma unroll
        for (int j = 0; j < AT_ONCE; j++) {
            const float istd = rsqrtf(var[j] + LN_EPS);
            const float out = ((y[j] - mean[j]) * istd * scale + shift + dot[j] * (float)s.v[n[j]][lane]) * (float)s.g[n[j]][lane];
            if (n0 + j * step < end) row(n[j])[h * HEAD + lane] = (__bf16)out;
        }
    }
}

// One token per sequence: block = (some rows of a 16-row tile, head).  Every wavefront asks for the first state it updates
// before the expansion starts, and for the next before it updates one.
template <int GROUPS, bool THROUGH>   // row groups: a wavefront updates every GROUPS-th of the block's rows
__global__ __launch_bounds__(256 * GROUPS) void decode_head_kernel(const HeadArgs A, int rows_per_block) {
    __shared__ HeadTile s;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane L;
    const int h = blockIdx.x;
    const int first = blockIdx.y * rows_per_block;                      // the block's rows: first .. first + count - 1
    const int row0 = first / TOK * TOK, r0 = first - row0;              // (inside the tile: r0 .. end - 1)
    const int end = r0 + (A.rows - first < rows_per_block ? A.rows - first : rows_per_block);
    const int ib = wave & 3, group = wave >> 2;
    f32x4 S[NBLK], Sn[NBLK];
    auto fetch = [&](f32x4 (&D)[NBLK], int r) {
        load_state(D, A.state_in, A.state_f32, (row0 + (r < end ? r : end - 1)) * A.H + h, ib, L);
    };
    fetch(S, r0 + group);
    expand_tile(s, A, h, row0, A.rows - 1, wave, L);
    for (int r = r0 + group; r < end; r += GROUPS) {
        fetch(Sn, r + GROUPS);   // (past the last row: that row again, unused)
        update_state(s, S, token_vectors(s, r, ib, L), r, ib, L);
        store_state<THROUGH>(S, A.state, A.state_f32, (row0 + r) * A.H + h, ib, L);
#pragma unroll
        for (int i = 0; i < NBLK; i++) S[i] = Sn[i];
    }
    lds_barrier();
    finish_tokens<1>(s, A.ln_params, A.C, h, r0 + wave, 4 * GROUPS, end, lane, [&](int r) { return A.ya + (long)(row0 + r) * A.C; });
}

// T tokens per sequence, one after the other on a state that stays in registers: block = (sequence, head).
__global__ __launch_bounds__(256) void prompt_head_kernel(const HeadArgs A) {
    __shared__ HeadTile s;
    const int lane = threadIdx.x & 63, ib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane L;
    const int h = blockIdx.x, seq = blockIdx.y, bh = seq * A.H + h;
    f32x4 S[NBLK];
    load_state(S, A.state_in, A.state_f32, bh, ib, L);
    for (int t0 = 0; t0 < A.T; t0 += TOK) {
        const int first = seq * A.T + t0, n = A.T - t0 < TOK ? A.T - t0 : TOK;
        expand_tile(s, A, h, first, first + n - 1, ib, L);
        update_tokens(s, S, n, ib, L);
        lds_barrier();
        finish_tokens<4>(s, A.ln_params, A.C, h, ib, 4, n, lane, [&](int t) { return A.ya + (long)(first + t) * A.C; });
        lds_barrier();   // (the next tile overwrites what the epilogue reads)
    }
    store_state(S, A.state, A.state_f32, bh, ib, L);
}

// The recurrence alone, token by token, with its operands in memory: the tokens of a prompt after its last whole chunk, whose
// state the sequence kernels would multiply in bf16.  Block = (sequence, head).  Bound by latency: 11 tokens x 2 x 12 heads take
// 8.5 us, of a token's two row sums one after the other, a barrier and the epilogue (one token at a time there and no vectors
// asked for ahead: 9.3; with fragments of the state 10.8).  The same tokens through the four kernels of a step instead: 26 us more for the prompt.
struct TokensArgs {
    const __bf16 *w, *k, *b, *r, *v, *kk, *g;   // at the sequences' first token
    __bf16* y;
    long wkb_seq, seq;                          // elements from one sequence to the next: of w, k, b; of the others and y
    int n, H, C, state_f32;                     // n tokens of each
    const float* ln_params;
    const void* state_in;                       // null: zeros
    void* state;                                // may be state_in itself
};
__device__ __forceinline__ void tokens_block(HeadTile& s, const TokensArgs& A, const int bh) {
    const int lane = threadIdx.x & 63, ib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane L;
    const int seq = bh / A.H, h = bh - seq * A.H;
    f32x4 S[NBLK];
    load_state(S, A.state_in, A.state_f32, bh, ib, L);
    // 16 bytes per thread and load: eight channels of one of the sixteen tokens, two tensors at a time (wavefronts 0, 1 and 2, 3)
    const int row = (threadIdx.x & 127) >> 3, c = 8 * (threadIdx.x & 7);
    const bool second = threadIdx.x >= 128;
    for (int t0 = 0; t0 < A.n; t0 += TOK) {
        const int n = A.n - t0 < TOK ? A.n - t0 : TOK;
        const long t = t0 + (row < n ? row : n - 1);   // (a row past the last repeats it and is not used)
        const long at = (long)seq * A.seq + t * A.C + h * HEAD + c, at_wkb = (long)seq * A.wkb_seq + t * A.C + h * HEAD + c;
        auto load = [](const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); };
        const bf16x8 x0 = load((second ? A.b : A.k) + at_wkb), x1 = load((second ? A.v : A.r) + at), x2 = load((second ? A.g : A.kk) + at);
        const bf16x4 wv = *reinterpret_cast<const bf16x4*>(A.w + at_wkb + (second ? 4 : 0));
        *reinterpret_cast<bf16x8*>(second ? &s.b[row][c] : &s.k[row][c]) = x0;
        *reinterpret_cast<bf16x8*>(second ? &s.v[row][c] : &s.r[row][c]) = x1;
        *reinterpret_cast<bf16x8*>(second ? &s.g[row][c] : &s.kk[row][c]) = x2;
        f32x4 d = to_f32(wv);
#pragma unroll
        for (int q = 0; q < 4; q++) d[q] = __expf(-__expf(d[q]));
        *reinterpret_cast<f32x4*>(&s.decay[row][c + (second ? 4 : 0)]) = d;
        lds_barrier();
        update_tokens(s, S, n, ib, L);
        lds_barrier();
        finish_tokens<4>(s, A.ln_params, A.C, h, ib, 4, n, lane, [&](int i) { return A.y + (long)seq * A.seq + (long)(t0 + i) * A.C; });
        lds_barrier();   // (the next sixteen overwrite what the epilogue reads)
    }
    store_state(S, A.state, A.state_f32, bh, ib, L);
}
__global__ __launch_bounds__(256) void tokens_kernel(const TokensArgs A) {
    __shared__ HeadTile s;
    tokens_block(s, A, blockIdx.x);
}
// The same as the first blocks of the launch that applies the epilogue to the chunks before those tokens (all but a sequence's last
// chunk: the tokens are in that one).  Neither stage fills the chip or waits for the other: 2 x 1003 tokens x 12 heads 6.6 + 8.6 us in two launches,
// so 10.0 (the blocks' LDS leaves seven of them to a compute unit, which the epilogue does not need).
__global__ __launch_bounds__(256) void epilogue_tokens_kernel(const TokensArgs A, int tokens_blocks, const LnForwardArgs E, int chunks) {
    __shared__ HeadTile s;
    if ((int)blockIdx.x < tokens_blocks) return tokens_block(s, A, blockIdx.x);   // (the whole block)
    const int wid = (blockIdx.x - tokens_blocks) * 4 + (threadIdx.x >> 6);
    if (wid >= chunks) return;
    const int NC = E.T / CHUNK, i = E.H >= 16 ? head_major_chunk(wid, chunks, E.T - CHUNK) : wid, bh = i / (NC - 1);
    ln_forward_chunk(E, i + bh, Lane());   // (chunk c of NC - 1 of each (batch, head), as one of NC)
}

constexpr size_t A256(size_t x) { return (x + 255) / 256 * 256; }
int padded_rows(int B) { return (B + TOK - 1) / TOK * TOK; }
}  // namespace

// B: tokens in all (sequences times tokens per sequence).  (Four planes, eight with the streams in memory, and the hidden
// activations are used and thirteen planes asked for: callers size the workspace with this, some with the number of an earlier release, and nothing is gained by less: 768 channels, 256
// sequences 5 MB.)
size_t mixer_decode_workspace_bytes(int B, int C) {
    const size_t Bp = padded_rows(B);
    return 13 * A256(Bp * C * 2) + A256(Bp * R_GATE * 2) + A256(Bp * R_DECAY * 2) + 4 * A256(Bp * 16 * 2);
}

// (us below: a whole step, replayed from a graph)

// A block repeats the expansion of its whole tile for the rows it updates, so it takes as many rows (up to 8) as leave about
// one block per compute unit.  In blocks of 1, 2, 4, 8 rows: 768 channels, 17 sequences 20.8, 20.9, 21.8, 23.3; 48 26.3, 25.1,
// 23.7, 26.0; 128 41.1, 38.1, 33.7, 33.5; 256 60.2, 54.9, 47.9, 45.2; 192 channels, 176 23.3, 21.7, 21.1, 22.1.
namespace {
int head_rows_per_block(int B, int H) {
    int rpb = 1;
    while (rpb < 8 && (long)H * ((B + rpb - 1) / rpb) > compute_units()) rpb *= 2;
    return rpb;
}

// The new states are written through the L2s while these, 32 MiB in all, hold most of them at the kernel's end and would be
// written back then; more than that leaves in the course of the kernel by itself.  12 heads, left to the end / through, 8 sequences (a row to a block) 19.6 /
// 19.6, 32 23.0 / 22.6, 64 26.9 / 25.9, 96 31.5 / 30.8, 128 (24 MiB) 32.6 / 32.1, 170 38.3 / 39.0, 256 43.7 / 44.1.
bool states_through(int B, int H) { return (long)B * H * HEAD * HEAD * (long)sizeof(float) <= 24 << 20; }

// Blocks of a linear kernel for each tile (or two), of so many columns.
template <int SEGS>
int column_blocks(const LinArgs<SEGS>& a, int columns) {
    int n = 0;
    for (int i = 0; i < SEGS; i++) n += (a.seg[i].N + columns - 1) / columns;
    return n;
}

// The first-half products of many rows: every column block of the linear kernel makes its stream again, so from some rows on
// the streams are written once (decode_lerp_kernel, a launch more) and multiplied by the grouped kernel of the sequence path,
// whose tiles share both operands through LDS: where the linear kernel's widest blocks take more than one round of the compute
// units, and below 768 channels, where a round more costs less than the launch, from rows x channels^2 = 4e8 on.  Linear at its
// best / streams: 768 channels, 160 rows (one round) 34.8/38.7, 176 42.0/42.5, 256 45.6/45.2, 512 66.5/66.8, 768 94.6/88.2;
// 832 channels, 160 40.4/43.5, 192 44.0/44.5, 256 47.6/48.0, 384 64.4/63.1; 1024 channels, 128 (one round) 38.4/40.6, 160
// 47.3/45.5, 256 54.8/51.9, 512 87.4/80.0; 1280 channels, 96 (one round) 40.9/42.4, 112 50.6/47.8; 2048 channels, 64 (one round)
// 48.7/49.0, 96 66.0/57.0, 512 214/179; 704 channels, 224 40.8/43.0, 384 55.4/60.9, 768 84.9/85.3, 1024 100.8/98.1; 512
// channels, 512 46.9/48.7, 1024 74.9/76.1, 1536 104.6/100.8.
bool streams_in_memory(const LinArgs<MAX_SEGS>& a, long rows) {
    const long C = a.plan[PLAN_C];
    const bool one_round = (long)column_blocks(a, 64) * ((a.plan[PLAN_TILES] + 1) / 2) <= compute_units();
    return rows > 32 && ((C >= 768 && !one_round) || rows * C * C >= 400000000);
}
// The output projection alone makes nothing again, and the grouped kernel's tiles are few for it.  Linear / grouped: 1024
// channels, 1024 rows 147.8/148.3, 1536 226.5/224.9; 1536 channels, 512 rows 114.3/116.5, 768 190.3/194.0, 1024 241.0/239.7;
// 2048 channels, 512 rows 177.8/179.0, 640 218.9/223.8, 768 249.9/248.1, 1536 442.9/438.2.
bool output_grouped(long rows, long C) { return rows * C * C >= 3000000000; }

// How much of the output a block of a linear kernel takes: the least that leaves a compute unit no second block.  Narrower blocks
// spread the loads wider; past one round they repeat the interpolation and re-read the inputs without any more of the chip to
// use (16 columns of the products with it for one tile only: of two they lose to 32 already, 384 channels 18.4, 18.0).  In
// columns x tiles of 16 x 1, 32 x 1, 64 x 1, 64 x 2: with the interpolation, 768 channels, 1 sequence 17.0, 18.2, 18.8, 19.3; 33
// 22.5, 21.2, 23.0, 23.7; 64 27.1, 27.5, 26.3, 26.2; 128 38.7, 35.6, 35.7, 33.4; 384 channels, 48 21.4, 18.9, 19.4, 20.7; 1536
// channels, 1 24.1, 21.9, 24.6, 26.5; 48 46.9, 38.8, 37.4, 40.8; the output, 768 channels, 48 23.8, 24.7, 25.4, 25.7; 256 45.0,
// 45.3, 44.7, 45.5; 1024 channels, 96 38.0, 36.3, 37.1, 38.1; 2048 channels, 144 79.6, 75.1, 75.3, 73.1.
template <bool LERP>
void launch_linear(LinArgs<LERP ? MAX_SEGS : 1>& a, const LinInput<LERP>& input, hipStream_t stream) {   // (the blocks of each pair: filled in here)
    const int ntiles = a.plan[PLAN_TILES];
    auto one_round = [&](int columns) { return column_blocks(a, columns) * ntiles <= compute_units(); };
    auto go = [&](auto kernel, int columns, int tiles) {
        int blocks = 0;
        for (int i = 0; i < (LERP ? MAX_SEGS : 1); i++) blocks += a.plan[i] = (a.seg[i].N + columns - 1) / columns;
        hipLaunchKernelGGL(kernel, dim3(blocks, (ntiles + tiles - 1) / tiles), dim3(256), 0, stream, a, input);
    };
    if ((!LERP || ntiles == 1) && one_round(16)) go(decode_linear_kernel<LERP, 1, 1>, 16, 1);
    else if (one_round(32)) go(decode_linear_kernel<LERP, 2, 1>, 32, 1);
    else if (one_round(64)) go(decode_linear_kernel<LERP, 4, 1>, 64, 1);
    else go(decode_linear_kernel<LERP, 4, 2>, 64, 2);
}
}  // namespace

void launch_mixer_decode(int B, int T, int C, int H, int state_f32, const MixerWeights& mw, const void* x, const void* x_prev,
                         const void* state_in, void* state, void* y, void* x_carry, void* workspace, hipStream_t stream) {
    const int rows = B * T, Bp = padded_rows(rows), ntiles = Bp / TOK;
    char* p = static_cast<char*>(workspace);
    auto take = [&](size_t elems) {
        __bf16* r = reinterpret_cast<__bf16*>(p);
        p += A256(elems * 2);
        return r;
    };
    const size_t BC = (size_t)Bp * C;
    __bf16 *mid = take((size_t)Bp * MID), *r = take(BC), *k = take(BC), *v = take(BC), *ya = take(BC);   // (inside the workspace, see above)
    __bf16 *tg1 = take((size_t)Bp * R_GATE), *tw1 = take((size_t)Bp * R_DECAY);
    __bf16 *kk1 = take((size_t)Bp * 16), *mk1 = take((size_t)Bp * 16), *a1 = take((size_t)Bp * 16), *ma1 = take((size_t)Bp * 16);
    auto c = [](const void* q) { return static_cast<const __bf16*>(q); };
    const MixIn mix{c(x), c(x_prev), c(mw.time_maa_w2), c(mw.time_maa), mid, rows, T};

    // (one round of loads for four wavefronts up to 768 channels; beyond, sixteen.  us, a step in 4 / 16: 768 channels, 1 sequence
    // 17.0/17.0, 48 23.6/24.2; 832 channels, 1 18.9/18.1; 2048 channels, 1 31.0/29.2, 256 92.8/91.4)
    if (C <= 768)
        hipLaunchKernelGGL((decode_mid_kernel<4, 3>), dim3(MID / 16, ntiles), dim3(256), 0, stream, mix, C, c(mw.time_maa_x),
                           c(mw.time_maa_w1), static_cast<__bf16*>(x_carry));
    else
        hipLaunchKernelGGL((decode_mid_kernel<16, 2>), dim3(MID / 16, ntiles), dim3(1024), 0, stream, mix, C, c(mw.time_maa_x),
                           c(mw.time_maa_w1), static_cast<__bf16*>(x_carry));
    {
        LinArgs<MAX_SEGS> a{};
        enum { XRG, XWA, XK, XV };
        a.seg[0] = {c(mw.Wr), r, C, 0, XRG};
        a.seg[1] = {c(mw.Wk), k, C, 0, XK};
        a.seg[2] = {c(mw.Wv), v, C, 0, XV};
        a.seg[3] = {c(mw.gate_w1), tg1, R_GATE, 1, XRG};
        a.seg[4] = {c(mw.time_decay_w1), tw1, R_DECAY, 1, XWA};
        a.seg[5] = {c(mw.time_kkk_w1), kk1, R_KKK, 0, XK};
        a.seg[6] = {c(mw.mk_w1), mk1, R_MK, 0, XK};
        a.seg[7] = {c(mw.time_aaa_w1), a1, R_AAA, 0, XWA};
        a.seg[8] = {c(mw.ma_w1), ma1, R_MA, 0, XWA};
        a.plan[PLAN_C] = C, a.plan[PLAN_ROWS] = Bp, a.plan[PLAN_TILES] = ntiles;
        if (streams_in_memory(a, rows)) {
            const long plane = (long)Bp * C;
            __bf16* const streams = take(4 * BC);
            hipLaunchKernelGGL(decode_lerp_kernel, dim3(C / 32, ntiles), dim3(256), 0, stream, mix, C, streams, plane);
            LinearProblem p[MAX_SEGS]{};
            for (int i = 0; i < MAX_SEGS; i++) {
                const LinSeg& s = a.seg[i];
                p[i].A[0] = streams + s.stream * plane, p[i].W[0] = s.W;
                p[i].lda[0] = p[i].ldw[0] = p[i].K[0] = C;
                p[i].N = s.N, p[i].npieces = 1;
                p[i].out[0] = s.out, p[i].ld_out[0] = p[i].width[0] = s.N;
                p[i].op[0] = s.tanh_out ? LINEAR_TANH : LINEAR_PLAIN;
            }
            launch_linear_group(MAX_SEGS, rows, p, stream);
        } else {
            launch_linear<true>(a, mix, stream);
        }
    }
    {
        const HeadArgs a{rows, T, C, H, state_f32, r, k, v, tg1, tw1, kk1, mk1, a1, ma1,
                         c(mw.gate_w2), c(mw.time_decay_w2), c(mw.time_kkk_w2), c(mw.time_aaa_w2), c(mw.ma_w2), c(mw.mk_w2),
                         c(mw.time_decay), c(mw.time_aaaaa), c(mw.time_misc_a), c(mw.time_misc_k),
                         static_cast<const float*>(mw.ln_params), state_in, state, ya};
        const int rpb = head_rows_per_block(B, H);
        const dim3 grid(H, (B + rpb - 1) / rpb);
        if (T > 1)
            hipLaunchKernelGGL(prompt_head_kernel, dim3(H, B), dim3(256), 0, stream, a);
        else if (rpb == 1)
            hipLaunchKernelGGL((decode_head_kernel<1, false>), grid, dim3(256), 0, stream, a, rpb);
        else if (states_through(B, H))
            hipLaunchKernelGGL((decode_head_kernel<2, true>), grid, dim3(512), 0, stream, a, rpb);
        else
            hipLaunchKernelGGL((decode_head_kernel<2, false>), grid, dim3(512), 0, stream, a, rpb);
    }
    {
        LinArgs<1> a{};
        a.seg[0] = {c(mw.Wo), static_cast<__bf16*>(y), C, 0, 0};
        a.plan[PLAN_C] = C, a.plan[PLAN_ROWS] = rows, a.plan[PLAN_TILES] = ntiles;
        if (output_grouped(rows, C)) {
            LinearProblem p{};
            p.A[0] = ya, p.W[0] = c(mw.Wo);
            p.lda[0] = p.ldw[0] = p.K[0] = p.N = C;
            p.npieces = 1, p.out[0] = static_cast<__bf16*>(y), p.ld_out[0] = p.width[0] = C;
            launch_linear_group(1, rows, &p, stream);
        } else {
            launch_linear<false>(a, ya, stream);
        }
    }
}

void launch_tokens(int B, int T, int H, int first, int n, int wkb_T, int wkb_first, int state_f32, const void* w, const void* q, const void* k,
                   const void* v, const void* a, const void* b, const void* g, const void* params, const void* state_in, void* state,
                   void* y, hipStream_t stream, const KeptOutput* epilogue) {
    const int C = H * HEAD;
    auto at = [&](const void* p, int token) { return static_cast<const __bf16*>(p) + (long)token * C; };
    const TokensArgs A{at(w, wkb_first), at(k, wkb_first), at(b, wkb_first), at(q, first), at(v, first), at(a, first), at(g, first),
                       static_cast<__bf16*>(y) + (long)first * C, (long)wkb_T * C, (long)T * C, n, H, C, state_f32,
                       static_cast<const float*>(params), state_in, state};
    if (epilogue == nullptr || T <= CHUNK) {
        hipLaunchKernelGGL(tokens_kernel, dim3((unsigned)(B * H)), dim3(256), 0, stream, A);
        return;
    }
    auto whole = [&](const void* p) { return static_cast<const __bf16*>(p); };
    const LnForwardArgs E{T, H, whole(epilogue->y_wkv), epilogue->centers, whole(q), whole(epilogue->k), whole(v), whole(g), A.ln_params, static_cast<__bf16*>(y)};
    const int chunks = B * H * (T / CHUNK - 1);
    hipLaunchKernelGGL(epilogue_tokens_kernel, dim3((unsigned)(B * H + (chunks + 3) / 4)), dim3(256), 0, stream, A, B * H, E, chunks);
}

}  // namespace wkv
