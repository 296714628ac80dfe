// ddlerp: data-dependent token-shift interpolation of RWKV-7, forward and backward, for gfx950.
//
// Replaces the six Triton kernels of the reference (rwkv7_ddlerp.py: fw1 :20-49, fw2 :53-84, bw1 :93-139,
// bw2 :143-167, bw3 :189-265, bw4 :269-303).  Spec (tests/test_ddlerp.py:5-13), per token m = (b, t):
//     xx   = x[t-1] - x[t]                       (zero row before t = 0)
//     a    = x + xx * alpha                       [C]
//     bmid = tanh(a L^T)                          [4D]      L: [4D, C]
//     c_k  = bmid_k R_k^T + beta_k                [C]       R: [4, C, D], k = 0..3
//     y_k  = x + xx * c_k
// The work is bandwidth-bound (x in, four streams out), but its inner products (C x 4D and 4D x C per
// token) only stay off the critical path on the matrix cores, so every contraction is a 16x16x32 MFMA on
// fragments (see frag.hpp): token tiles of 16 rows, channel blocks of 64.
#include "row_lines.hpp"
#include "device_info.hpp"
#include "ddlerp_kernels.hpp"
#include <type_traits>

namespace wkv {

namespace {

constexpr int TOK = 16;  // tokens per tile

struct Dy4 {  // the four upstream gradients, each [M, C]
    const __bf16* p[4];
};

}  // namespace

// ------------------------------------------------------------------------------------------------
// The two contractions over all C channels (forward 1 and backward 1) give a block TPB token tiles (16 tokens each) and
// walk the channel blocks of 64: eight lanes fetch the 128 bytes of one row of a channel block, of the weights as of the
// streams, a thread does the elementwise part for its eight channels of a token once, and everything passes through a
// double-buffered LDS image from which the matrix instructions take their fragments (one barrier per channel block); each
// tile is finished by 4 / TPB wavefronts, which split the output blocks.
// What bounds these kernels is the number of lookups of a compute unit's vector cache: four lanes on four rows, the order
// of a fragment, are four lookups, and a wavefront's 16-byte load takes 28 ns of the compute unit, against 9 for eight lanes
// on each whole line (measured with everything in L2; stores 28 and 20).  Fragments straight from memory took 16.8 (forward 1)
// and 22.2 us (backward 1) at 8192 tokens x 768 channels, no less with twice the wavefronts; this way 11.2 and 14.4, and 17.5
// and 34.5 at 16384 tokens instead of 24.5 and 38.5.  What is left is a round of load, LDS and barrier per channel block,
// which neither two blocks of channels at a time nor four sets of operands in flight made shorter; backward 1 moves 63 MB at
// 8192 tokens, 12.4 us at the rate of a copy.
// ------------------------------------------------------------------------------------------------
// a token's 8 channels and those of the token before it, as they lie in memory
struct Shifted {
    bf16x8 cur, prev;
};
// Whether each of a block's TPB tiles begins a sequence (sequences are whole tiles): one division, of 32-bit numbers that the whole block
// shares.  (A remainder of 64-bit numbers per row was 180 instructions for each ahead of a block's first load, and two of them a tile in forward 2;
// so 2016 tokens x 768 channels, forward 1 and 2, 7.9, 7.1 -> 7.7, 6.3 us, 8192, backward 1 and 2 too, 12.8, 12.9, 17.1, 35.8 -> 12.6, 12.5, 16.8, 35.2.)
template <int TPB>
struct TileStarts {
    bool start[TPB];
    __device__ __forceinline__ explicit TileStarts(int T) {
        const unsigned per_sequence = (unsigned)T / TOK;
        unsigned pos = blockIdx.x * TPB % per_sequence;
#pragma unroll
        for (int p = 0; p < TPB; p++) {
            start[p] = pos == 0;
            pos = pos + 1 == per_sequence ? 0 : pos + 1;
        }
    }
};
template <int TPB>
struct TokenRows {   // this thread's tokens of a block's tiles: token t8 + 32 i, channels 8 piece of every channel block
    static constexpr int N = TPB / 2;
    const __bf16* row[N];
    bool has_prev[N];
    long m[N];
    __device__ __forceinline__ TokenRows(const __bf16* __restrict__ x, long M, int T, int C, int t8, int piece) {
        const TileStarts<TPB> tiles(T);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const long want = (long)blockIdx.x * (TPB * TOK) + t8 + 32 * i;
            m[i] = want < M ? want : M - 1;   // (rows of a spare tile: the last one again, never stored)
            has_prev[i] = t8 % TOK != 0 || !(t8 < TOK ? tiles.start[2 * i] : tiles.start[2 * i + 1]);
            row[i] = x + m[i] * C + 8 * piece;
        }
    }
    __device__ __forceinline__ Shifted load(int i, int C, int c0) const {
        return {*reinterpret_cast<const bf16x8*>(row[i] + c0), *reinterpret_cast<const bf16x8*>(row[i] + c0 - (has_prev[i] ? C : 0))};
    }
};

// a = x + xx*alpha as a bf16 pair (hi + lo): the pre-activation feeds tanh', which is steep, so the interpolated input must
// not be rounded to 8 bits before the 768-term sum (L itself is bf16)
__device__ __forceinline__ void interpolate(const bf16x8 cur, const bf16x8 prev, const bf16x4 al0, const bf16x4 al1, bf16x8& hi, bf16x8& lo) {
    f32x4 av[2];
#pragma unroll
    for (int hlf = 0; hlf < 2; hlf++) {
        const f32x4 c = to_f32(hlf ? __builtin_shufflevector(cur, cur, 4, 5, 6, 7) : __builtin_shufflevector(cur, cur, 0, 1, 2, 3));
        const f32x4 q = to_f32(hlf ? __builtin_shufflevector(prev, prev, 4, 5, 6, 7) : __builtin_shufflevector(prev, prev, 0, 1, 2, 3));
        av[hlf] = c + (q - c) * to_f32(hlf ? al1 : al0);
    }
    const bf16x4 h0 = to_bf16(av[0]), h1 = to_bf16(av[1]);
    hi = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
    lo = __builtin_shufflevector(to_bf16(av[0] - to_f32(h0)), to_bf16(av[1] - to_f32(h1)), 0, 1, 2, 3, 4, 5, 6, 7);
}
// tanh and its derivative 1 - tanh^2 = 4e/(e+1)^2, e = exp(2s).  The derivative is stored on its own:
// recovering it from a bf16-rounded tanh loses all precision where the unit saturates.
__device__ __forceinline__ void store_activation(f32x4 s, __bf16* __restrict__ bmid, __bf16* __restrict__ bder, long off) {
    f32x4 t, dt;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float e = __expf(2.f * fminf(s[r], 40.f));
        const float inv = __builtin_amdgcn_rcpf(e + 1.f);   // 1 ulp; an IEEE division is ten instructions
        t[r] = 1.f - 2.f * inv;
        dt[r] = 4.f * e * inv * inv;
    }
    *reinterpret_cast<bf16x4*>(bmid + off) = to_bf16(t);
    *reinterpret_cast<bf16x4*>(bder + off) = to_bf16(dt);
}

// forward 1 for few tokens: a block takes TPB tiles and one of SPLIT parts of the outputs, its four wavefronts a quarter of
// the channel blocks each, every one through its own part of LDS; one sum over the wavefronts at the end.  What bounds a
// launch of this size is what ONE compute unit can fetch, so the weights are spread over the blocks.  The kernel below
// fetches all of them per block, a barrier per channel block.  Whole lines as above,
// 768 channels and 1024, 4096 tokens, 2048 channels and 4096 tokens: 9.3, 13.7, 28.5 -> 7.5, 10.9, 18.7 us.
template <int D, int SPLIT, int TPB>
__global__ __launch_bounds__(256) void ddlerp_fwd_mid_few_kernel(long M, int T, int C, const __bf16* __restrict__ x,
                                                                 const __bf16* __restrict__ alpha,
                                                                 const __bf16* __restrict__ Lw, __bf16* __restrict__ bmid,
                                                                 __bf16* __restrict__ bder) {
    constexpr int NB = 4 * D / 16 / SPLIT, NA = NB * TPB;   // output blocks of 16; with the tiles: accumulators
    constexpr int NW = 2 * NB, NR = 2 * TPB;                // rows of the weights and tokens per lane
    struct Image {   // of one wavefront and channel block
        bf16x8 w[16 * NB * 8], a[2][16 * TPB * 8];
    };
    __shared__ union {
        Image img[4];
        f32x4 part[4][NA][WAVE];
    } lds;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l8 = lane >> 3, piece = lane & 7;
    const Lane L;
    const long ntiles = M / TOK;
    const int ncb = C / 64, db0 = NB * blockIdx.y;
    const __bf16* row[NR];
    bool has_prev[NR];
    const TileStarts<TPB> tiles(T);
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const long want = (long)blockIdx.x * (TPB * TOK) + l8 + 8 * i, m = want < M ? want : M - 1;   // (a spare tile stores nothing)
        has_prev[i] = (l8 + 8 * i) % TOK != 0 || !tiles.start[i / 2];
        row[i] = x + m * C + 8 * piece;
    }
    f32x4 acc[TPB][NB];
#pragma unroll
    for (int p = 0; p < TPB; p++)
#pragma unroll
        for (int i = 0; i < NB; i++) acc[p][i] = zero4();
    struct Set {
        bf16x8 w[NW];
        Shifted x[NR];
        bf16x4 al[2];
    };
    auto fetch = [&](Set& st, int cb) {
        const int c0 = 64 * (cb < ncb ? cb : ncb - 1);   // (past the last block: it again, not used)
#pragma unroll
        for (int i = 0; i < NW; i++) st.w[i] = piece_at(Lw + ((long)(16 * db0 + 8 * i) * C + c0), 2 * ((unsigned)l8 * C + 8 * piece));
#pragma unroll
        for (int i = 0; i < NR; i++)
            st.x[i] = {*reinterpret_cast<const bf16x8*>(row[i] + c0), *reinterpret_cast<const bf16x8*>(row[i] + c0 - (has_prev[i] ? C : 0))};
#pragma unroll
        for (int h = 0; h < 2; h++) st.al[h] = *reinterpret_cast<const bf16x4*>(alpha + c0 + 8 * piece + 4 * h);
    };
    Image& img = lds.img[wave];
    auto use = [&](const Set& st) {
#pragma unroll
        for (int i = 0; i < NW; i++) img.w[piece_slot(l8 + 8 * i, piece)] = st.w[i];
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const bf16x8 zero = {};
            bf16x8 hi, lo;
            interpolate(st.x[i].cur, has_prev[i] ? st.x[i].prev : zero, st.al[0], st.al[1], hi, lo);
            img.a[0][piece_slot(l8 + 8 * i, piece)] = hi;
            img.a[1][piece_slot(l8 + 8 * i, piece)] = lo;
        }
        wave_lds_order();
        bf16x8 l[NB][2];
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int pr = 0; pr < 2; pr++) l[i][pr] = img.w[piece_slot(16 * i + L.n, 4 * pr + L.g)];
#pragma unroll
        for (int p = 0; p < TPB; p++)
#pragma unroll
            for (int hl = 0; hl < 2; hl++)
#pragma unroll
                for (int pr = 0; pr < 2; pr++) {
                    const bf16x8 a = img.a[hl][piece_slot(16 * p + L.n, 4 * pr + L.g)];
#pragma unroll
                    for (int i = 0; i < NB; i++) acc[p][i] = mma8(acc[p][i], l[i][pr], a);
                }
        wave_lds_order();
    };
    constexpr int SETS = 3;   // channel blocks in flight
    Set st[SETS];
#pragma unroll
    for (int d = 0; d < SETS; d++) fetch(st[d], wave + 4 * d);
    __builtin_amdgcn_sched_barrier(0);
    for (int cb = wave; cb < ncb; cb += 4 * SETS) {
#pragma unroll
        for (int d = 0; d < SETS; d++) {
            if (cb + 4 * d < ncb) {
                use(st[d]);
                if (cb + 4 * (d + SETS) < ncb) fetch(st[d], cb + 4 * (d + SETS));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // the sums over the wavefronts, each by one wavefront and in their order
    __syncthreads();
#pragma unroll
    for (int p = 0; p < TPB; p++)
#pragma unroll
        for (int i = 0; i < NB; i++) lds.part[wave][p * NB + i][lane] = acc[p][i];
    __syncthreads();
    for (int e = wave; e < NA; e += 4) {
        const int p = e / NB, i = e % NB;
        const long tile = (long)blockIdx.x * TPB + p;
        if (tile >= ntiles) break;
        const f32x4 s = (lds.part[0][e][lane] + lds.part[1][e][lane]) + (lds.part[2][e][lane] + lds.part[3][e][lane]);
        store_activation(s, bmid, bder, (tile * TOK + L.n) * (4 * D) + 16 * (db0 + i) + 4 * L.g);
    }
}

// forward 1: bmid = tanh((x + xx*alpha) L^T), bder = 1 - bmid^2
template <int D, int TPB>
__global__ __launch_bounds__(256) void ddlerp_fwd_mid_kernel(long M, int T, int C, const __bf16* __restrict__ x,
                                                             const __bf16* __restrict__ alpha,
                                                             const __bf16* __restrict__ Lw, __bf16* __restrict__ bmid,
                                                             __bf16* __restrict__ bder) {
    constexpr int NB = 4 * D / 16;       // output blocks of 16
    constexpr int WPT = 4 / TPB;         // wavefronts per tile
    constexpr int NBW = NB / WPT;        // output blocks per wavefront
    constexpr int NW = 4 * D / 32, NR = TokenRows<TPB>::N;   // rows of the weights and tokens per thread
    __shared__ bf16x8 s_w[2][4 * D * 8], s_a[2][2][TPB * TOK * 8];   // a: hi, lo
    const int wave = threadIdx.x >> 6, t8 = threadIdx.x >> 3, piece = threadIdx.x & 7;
    const Lane L;
    const long tile = (long)blockIdx.x * TPB + wave / WPT;
    const int db0 = (wave % WPT) * NBW, row0 = TOK * (wave / WPT);
    const TokenRows<TPB> tokens(x, M, T, C, t8, piece);

    f32x4 acc[NBW];
#pragma unroll
    for (int i = 0; i < NBW; i++) acc[i] = zero4();
    // Blocks start at different channel blocks: all of them asking for the same 16 KiB of weights at the same
    // moment queue on the few L2 channels that hold it.
    const int ncb = C / 64;
    auto advance = [&](int c) { return c + 1 < ncb ? c + 1 : 0; };
    // Two sets of streamed operands, each refilled right after the round that used it, so a load has two rounds to arrive.
    // The operands stay raw registers until the round that uses them: a conversion at the point of the load, or a load
    // under a condition, makes the compiler wait for the data right there.
    struct Set {
        bf16x8 w[NW];
        Shifted x[NR];
        bf16x4 al[2];
    };
    auto fetch = [&](Set& st, int cbk) {
        const int c0 = 64 * cbk;
#pragma unroll
        for (int i = 0; i < NW; i++) st.w[i] = piece_at(Lw + ((long)32 * i * C + c0), 2 * ((unsigned)t8 * C + 8 * piece));
#pragma unroll
        for (int i = 0; i < NR; i++) st.x[i] = tokens.load(i, C, c0);
#pragma unroll
        for (int h = 0; h < 2; h++) st.al[h] = *reinterpret_cast<const bf16x4*>(alpha + c0 + 8 * piece + 4 * h);
    };
    int next_cb = blockIdx.x % ncb;
    Set sa, sb;
    fetch(sa, next_cb);
    next_cb = advance(next_cb);
    fetch(sb, next_cb);
    next_cb = advance(next_cb);
    auto round = [&](Set& st, int buf) {
#pragma unroll
        for (int i = 0; i < NW; i++) s_w[buf][piece_slot(t8 + 32 * i, piece)] = st.w[i];
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const bf16x8 zero = {};
            bf16x8 hi, lo;
            interpolate(st.x[i].cur, tokens.has_prev[i] ? st.x[i].prev : zero, st.al[0], st.al[1], hi, lo);
            s_a[buf][0][piece_slot(t8 + 32 * i, piece)] = hi;
            s_a[buf][1][piece_slot(t8 + 32 * i, piece)] = lo;
        }
        __syncthreads();
        fetch(st, next_cb);   // (the last two rounds fetch blocks that are not used)
        next_cb = advance(next_cb);
        bf16x8 a[2][2];
#pragma unroll
        for (int hl = 0; hl < 2; hl++)
#pragma unroll
            for (int pr = 0; pr < 2; pr++) a[hl][pr] = s_a[buf][hl][piece_slot(row0 + L.n, 4 * pr + L.g)];
#pragma unroll
        for (int i = 0; i < NBW; i++) {
            bf16x8 l[2];   // F(L[16db.., c0..]) lane = output
#pragma unroll
            for (int pr = 0; pr < 2; pr++) l[pr] = s_w[buf][piece_slot(16 * (db0 + i) + L.n, 4 * pr + L.g)];
#pragma unroll
            for (int hl = 0; hl < 2; hl++)
#pragma unroll
                for (int pr = 0; pr < 2; pr++) acc[i] = mma8(acc[i], l[pr], a[hl][pr]);   // + F(a L^T) lane = token
        }
    };
    int it = 0;
    for (; it + 2 <= ncb; it += 2) {
        round(sa, 0);
        round(sb, 1);
    }
    if (it < ncb) round(sa, 0);
    if (tile * TOK >= M) return;
#pragma unroll
    for (int i = 0; i < NBW; i++) store_activation(acc[i], bmid, bder, (tile * TOK + L.n) * (4 * D) + 16 * (db0 + i) + 4 * L.g);
}

// ------------------------------------------------------------------------------------------------
// backward 1: dpre = ((dy_k * xx) R_k) * (1 - bmid^2)        [M, 4D]   (the factor 1 - bmid^2 was saved by forward)
// Same structure as forward 1; the weights are R [4, C, D], 64 rows of D elements per channel block and interpolation,
// kept in LDS as they lie in memory and read back transposed (ds_read_b64_tr_b16, the lanes' addresses as in the WKV7
// backward kernels: lane p of a group of 16 points at the 8 bytes of row p/4, columns 4(p%4).. of its four rows).
// ------------------------------------------------------------------------------------------------
// A transposing read takes 32 bytes of each of rows 8g' .. 8g'+3 for two groups at a time: four rows of 64 bytes (D = 32) are
// the banks once over, two of 128 (D = 64) as well, so pieces move by pairs for odd g' and, at D = 64, rows 2 and 3.
template <int D>
__device__ __forceinline__ int r_slot(int channel, int piece) {
    return (D / 8) * channel + (D == 32 ? piece ^ (channel >> 2 & 2) : piece ^ (channel & 2) ^ (channel >> 1 & 4));
}
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3))) lds_s16x4;
typedef unsigned char __attribute__((address_space(3))) lds_u8;
template <int D, int TPB>
__global__ __launch_bounds__(256) void ddlerp_bwd_mid_kernel(long M, int T, int C, const __bf16* __restrict__ x,
                                                             Dy4 dy,
                                                             const __bf16* __restrict__ R,
                                                             const __bf16* __restrict__ bder,
                                                             __bf16* __restrict__ dpre) {
    constexpr int ND = D / 16, NB = 4 * ND;
    constexpr int WPT = 4 / TPB, NBW = NB / WPT;
    static_assert(NBW % ND == 0, "a wavefront owns whole interpolations k");
    constexpr int NW = 4 * D / 32, NR = TokenRows<TPB>::N;
    __shared__ bf16x8 s_r[2][4][64 * D / 8], s_dc[2][4][TPB * TOK * 8];
    const int wave = threadIdx.x >> 6, t8 = threadIdx.x >> 3, piece = threadIdx.x & 7;
    const Lane L;
    const long tile = (long)blockIdx.x * TPB + wave / WPT;
    const int db0 = (wave % WPT) * NBW, k0 = db0 / ND, row0 = TOK * (wave / WPT);
    const TokenRows<TPB> tokens(x, M, T, C, t8, piece);

    f32x4 acc[NBW];
#pragma unroll
    for (int i = 0; i < NBW; i++) acc[i] = zero4();
    struct Set {
        bf16x8 r[NW], dy[4][NR];
        Shifted x[NR];
    };
    auto fetch = [&](Set& st, int c0) {
#pragma unroll
        for (int i = 0; i < NW; i++)   // R_k from channel c0 on: NW / 4 contiguous runs of 4 KiB
            st.r[i] = piece_at(R + ((long)(i / (NW / 4)) * C + c0) * D + 2048 * (i % (NW / 4)), 16 * threadIdx.x);
#pragma unroll
        for (int i = 0; i < NR; i++) {
            st.x[i] = tokens.load(i, C, c0);
#pragma unroll
            for (int k = 0; k < 4; k++) st.dy[k][i] = *reinterpret_cast<const bf16x8*>(dy.p[k] + tokens.m[i] * C + c0 + 8 * piece);
        }
    };
    auto round = [&](Set& st, int buf, int next) {
#pragma unroll
        for (int i = 0; i < NW; i++) {
            const int p = threadIdx.x + 256 * (i % (NW / 4));
            s_r[buf][i / (NW / 4)][r_slot<D>(p / (D / 8), p % (D / 8))] = st.r[i];
        }
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const bf16x8 zero = {}, prev = tokens.has_prev[i] ? st.x[i].prev : zero;
            f32x4 xx[2];
#pragma unroll
            for (int h = 0; h < 2; h++) xx[h] = to_f32(half_of(prev, h)) - to_f32(half_of(st.x[i].cur, h));
#pragma unroll
            for (int k = 0; k < 4; k++)
                s_dc[buf][k][piece_slot(t8 + 32 * i, piece)] =
                    join(to_bf16(to_f32(half_of(st.dy[k][i], 0)) * xx[0]), to_bf16(to_f32(half_of(st.dy[k][i], 1)) * xx[1]));
        }
        __syncthreads();
        fetch(st, next);   // (the last rounds fetch blocks that are not used)
#pragma unroll
        for (int k = 0; k < NBW / ND; k++) {
#pragma unroll
            for (int pr = 0; pr < 2; pr++) {
                const bf16x8 dc = s_dc[buf][k0 + k][piece_slot(row0 + L.n, 4 * pr + L.g)];
#pragma unroll
                for (int j = 0; j < ND; j++) {
                    bf16x4 rt[2];   // F(R_k^T) lane = mid index 16j + n, channels 32pr + 8g + 4h ..
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const int ch = 32 * pr + 8 * L.g + 4 * h + (L.n >> 2), col = 16 * j + 4 * (L.n & 3);
                        rt[h] = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (lds_s16x4*)((lds_u8*)&s_r[buf][k0 + k][r_slot<D>(ch, col / 8)] + 2 * (col & 7))));
                    }
                    acc[k * ND + j] = mma8(acc[k * ND + j], join(rt[0], rt[1]), dc);   // + F(dc R_k) lane = token
                }
            }
        }
    };
    auto block = [&](int cb) { return cb < C ? cb : C - 64; };
    Set sa, sb;
    fetch(sa, 0);
    fetch(sb, block(64));
    int c0 = 0;
    for (; c0 + 128 <= C; c0 += 128) {
        round(sa, 0, block(c0 + 128));
        round(sb, 1, block(c0 + 192));
    }
    if (c0 < C) round(sa, 0, C - 64);
    if (tile * TOK >= M) return;
#pragma unroll
    for (int i = 0; i < NBW; i++) {
        const long off = (tile * TOK + L.n) * (4 * D) + 16 * (db0 + i) + 4 * L.g;
        *reinterpret_cast<bf16x4*>(dpre + off) = to_bf16(acc[i] * to_f32(*reinterpret_cast<const bf16x4*>(bder + off)));
    }
}

// ------------------------------------------------------------------------------------------------
// Forward 2 gives a block one 64-channel block and a range of token tiles: the block's 16 KiB of weight
// fragments (R) are staged in LDS once, in the order the matrix instructions take them (16 bytes per lane), and
// every wavefront walks its tiles, the next one's operands on their way.  A tile's rows of x, of bmid and of the four
// streams move as whole lines (see above) through the wavefront's own part of LDS; as pieces of 16 rows, 20
// instructions of 28 ns of a compute unit's time per tile and channel block, 4096, 8192, 16384, 32768 tokens x 768 channels
// took 12.1, 20.3, 33.4, 72 us; now 9.0, 13.6, 25.7, 59, of which the bytes are 6, 13, 25, 50 at the rate of a copy.  Stored through the L2 it
// takes 6.9 instead of 8.6 in a prompt of 2016 tokens, 13.2 instead of 14.7 in a block of 8192.
// ------------------------------------------------------------------------------------------------
// A lane group g holds mid indices 8g .. 8g+7 of each 32: the order of a contraction is free if both operands agree.
template <int D>
struct LerpWeights {   // LDS image for one 64-channel block
    bf16x8 R[4][NBLK][D / 32][WAVE];   // F(R_k[c.., 32j + 8g ..])  lane = channel
    float beta[4][64];
};
template <int D>
__device__ __forceinline__ void stage_lerp_weights(LerpWeights<D>& w, const __bf16* __restrict__ R,
                                                   const __bf16* __restrict__ beta, int C, int c0) {
    const int thread = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int i = 0; i < D / 32; i++) {   // R_k from channel c0 on, as it lies in memory: 256 pieces a time
            const int p = thread + 256 * i, ch = p / (D / 8), j = p % (D / 8) / 4, g = p % 4;
            // channel block and lane of a channel: chan16 the other way round
            const int cb = 2 * (ch >> 5) + (ch >> 2 & 1), n = 4 * (ch >> 3 & 3) + (ch & 3);
            w.R[k][cb][j][n + 16 * g] = piece_at(R + ((long)k * C + c0) * D, 16 * p);
        }
    w.beta[thread >> 6][thread & 63] = (float)beta[(long)(thread >> 6) * C + c0 + (thread & 63)];
}

// forward 2: y_k = x + xx * (bmid_k R_k^T + beta_k).  Block = (64 channels, range of token tiles).
template <int D>
__global__ __launch_bounds__(256) void ddlerp_fwd_out2_kernel(long M, int T, int C, int tiles_per_split,
                                                              const __bf16* __restrict__ x,
                                                              const __bf16* __restrict__ R, const __bf16* __restrict__ beta,
                                                              const __bf16* __restrict__ bmid, __bf16* __restrict__ y) {
    constexpr int MP = 4 * D / 8;   // pieces of a row of bmid
    struct Image {                  // of one wavefront's tile
        bf16x8 x[(TOK + 1) * 8], mid[TOK * MP], out[TOK * 8];   // x: from the row before the tile on
    };
    __shared__ LerpWeights<D> w;
    __shared__ Image img_all[4];
    const int lane = threadIdx.x & 63, l8 = lane >> 3, piece = lane & 7;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Image& img = img_all[wave];
    const Lane L;
    const int c0 = blockIdx.x * 64;
    const long ntiles = M / TOK;
    const long tile_begin = (long)blockIdx.y * tiles_per_split;
    const long tile_end = tile_begin + tiles_per_split < ntiles ? tile_begin + tiles_per_split : ntiles;
    const unsigned row_bytes = 2 * C, lane_bytes = l8 * row_bytes + 16 * piece;   // (16 rows: 32 C bytes, below 2^32)
    struct Rows {
        bf16x8 x[2], before, mid[MP / 4];
        bool inside;   // the tile does not begin a sequence
    };
    const unsigned per_sequence = (unsigned)T / TOK;   // (tiles are few enough for 32 bits)
    auto fetch = [&](long tile) {
        Rows r;
        const long m0 = tile * TOK;
        const __bf16* xt = x + m0 * C + c0;
#pragma unroll
        for (int i = 0; i < 2; i++) r.x[i] = piece_at(xt, lane_bytes + 8 * i * row_bytes);
        r.inside = (unsigned)tile % per_sequence != 0;
        r.before = piece_at(r.inside ? xt - C : xt, 16 * piece);
#pragma unroll
        for (int i = 0; i < MP / 4; i++) r.mid[i] = piece_at(bmid + m0 * (4 * D) + 512 * i, 16 * lane);
        return r;
    };
    // a column of sixteen rows in sixteen different banks of 16 bytes
    auto mid_slot = [](int row, int p) { return MP * row + (p ^ row); };
    long tile = tile_begin + wave;
    Rows next;
    if (tile < tile_end) next = fetch(tile);
    stage_lerp_weights<D>(w, R, beta, C, c0);
    __syncthreads();
    for (; tile < tile_end; tile += 4) {
        const long m0 = tile * TOK;
        const bf16x8 zero = {};
#pragma unroll
        for (int i = 0; i < 2; i++) img.x[piece_slot(1 + l8 + 8 * i, piece)] = next.x[i];
        if (l8 == 0) img.x[piece_slot(0, piece)] = next.inside ? next.before : zero;
#pragma unroll
        for (int i = 0; i < MP / 4; i++) img.mid[mid_slot((lane + 64 * i) / MP, (lane + 64 * i) % MP)] = next.mid[i];
        wave_lds_order();
        next = fetch(tile + 4 < tile_end ? tile + 4 : tile);   // (past the end: this one again, not used)
        f32x4 xv[NBLK], xx[NBLK];
#pragma unroll
        for (int cb = 0; cb < NBLK; cb++) {
            xv[cb] = to_f32(half_of(img.x[piece_slot(L.n + 1, 4 * (cb >> 1) + L.g)], cb & 1));
            xx[cb] = to_f32(half_of(img.x[piece_slot(L.n, 4 * (cb >> 1) + L.g)], cb & 1)) - xv[cb];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            bf16x8 bm[D / 32];
#pragma unroll
            for (int j = 0; j < D / 32; j++) bm[j] = img.mid[mid_slot(L.n, (D / 8) * k + 4 * j + L.g)];
            bf16x4 o[NBLK];
#pragma unroll
            for (int cb = 0; cb < NBLK; cb++) {
                f32x4 c = *reinterpret_cast<const f32x4*>(&w.beta[k][chan16(cb, 4 * L.g)]);
#pragma unroll
                for (int j = 0; j < D / 32; j++) c = mma8(c, w.R[k][cb][j][lane], bm[j]);
                o[cb] = to_bf16(xv[cb] + xx[cb] * c);
            }
            wave_lds_order();
#pragma unroll
            for (int pr = 0; pr < 2; pr++) img.out[piece_slot(L.n, 4 * pr + L.g)] = join(o[2 * pr], o[2 * pr + 1]);
            wave_lds_order();
            __bf16* dst = y + ((long)k * M + m0) * C + c0;
#pragma unroll
            for (int i = 0; i < 2; i++)
                store_through_at(dst, lane_bytes + 8 * i * row_bytes, img.out[piece_slot(l8 + 8 * i, piece)]);
        }
        wave_lds_order();
    }
}

// backward 2: everything that walks the tokens a second time, in one pass: dx and the parameter gradients.
//   da  = dpre L ;  dxx = da*alpha + sum_k dy_k*c_k ;  dx[t] = da + sum_k dy_k - dxx[t] + dxx[t+1]
//   dR_k = (dy_k*xx)^T bmid_k,  dbeta_k = sum_t dy_k*xx,  dL = dpre^T a,  dalpha = sum_t da*xx
// Block = (64 channels, a contiguous range of token tiles); each of its four wavefronts owns 16 of the channels for
// the whole range and never meets the others: it reads its 8-byte pieces of x, x[t-1] and the four dy rows, the full
// 256-byte rows of bmid and dpre (16 bytes per lane), and keeps dR[:, its channels, :], dL[:, its channels] and the
// two vectors in registers.  The tiles are walked from the last one down, so the shifted term of the tile above is
// the carry; only the first tile a wavefront touches has none, and when the token after the range continues the
// sequence the wavefront evaluates that tile first without storing or accumulating anything.
// The contraction index of a 32-wide product may be permuted at will as long as both operands agree, so a lane
// group g holds mid indices 8g .. 8g+7 of each interpolation (one 16-byte load); as two 16-wide fragments that is
// index dmap(jj, 4g + r), and the transposed fragments and the accumulators built from them carry the same map.
// (Separate kernels for dx, for dR/dbeta and for dL/dalpha read x three times and dy twice at one wavefront per
// SIMD, 98 us together at 8192 tokens x 768 channels.  One wavefront per interpolation k instead of per channel
// group repeated the x arithmetic four times and added four partial dx tiles through LDS: 47 us.  This
// organisation with every wavefront loading its own pieces from memory: 58 us, bound by the L2-to-CU traffic of
// quarter-used lines; with the shared LDS images: 35 us, of which about 30 are the arithmetic.)
template <int D>
struct ParamPartial {   // per (split, 64-channel block); element counts
    static constexpr int DR = 4 * 64 * D, DL = 4 * D * 64, DBETA = 4 * 64, DALPHA = 64;
    static constexpr int TOTAL = DR + DL + DBETA + DALPHA;
};
__host__ __device__ constexpr int dmap(int jj, int j) { return 8 * (j >> 2) + 4 * jj + (j & 3); }

// G groups of four wavefronts per block, each with a range of its own; their sums meet in LDS before the record is written.
template <int D, int G>
__global__ __launch_bounds__(256 * G, D == 32 ? 2 : 1) void ddlerp_bwd_main_kernel(long M, int T, int C, int tiles_per_split,
                                                                 const __bf16* __restrict__ x, Dy4 dy,
                                                                 const __bf16* __restrict__ alpha,
                                                                 const __bf16* __restrict__ Lw,
                                                                 const __bf16* __restrict__ R,
                                                                 const __bf16* __restrict__ beta,
                                                                 const __bf16* __restrict__ bmid,
                                                                 const __bf16* __restrict__ dpre,
                                                                 __bf16* __restrict__ dx, float* __restrict__ partial) {
    static_assert(D % 32 == 0 && D <= 64, "32-wide contractions, HH of them per interpolation");
    using P = ParamPartial<D>;
    constexpr int HH = D / 32;
    // Each wavefront's own weight fragments, [k][32-wide half]: 8 KiB in LDS at rank 32 ([wavefront][k][lane]); at
    // rank 64 the streamed images below leave no room for 16 KiB per wavefront and they stay in registers.
    constexpr bool W_LDS = HH == 1;
    bf16x8 r_R[W_LDS ? 1 : 4][HH], r_L[W_LDS ? 1 : 4][HH];
    // LDS images of a tile's streamed rows (elements; row pitches padded by 16 bytes against bank conflicts)
    constexpr int ROW_LD = 64 + 8, MID_LD = 4 * D + 8;
    struct Images {
        __bf16 x[2][17 * ROW_LD], row[2][4][16 * ROW_LD], mid[2][2][16 * MID_LD];
    };
    constexpr int NEX = 16 * HH + 5;   // the group's sums: dR, dL, dbeta, dalpha
    __shared__ __attribute__((aligned(16))) union {
        struct {
            bf16x8 R[W_LDS ? 4 : 1][W_LDS ? 4 : 1][W_LDS ? WAVE : 1], L[W_LDS ? 4 : 1][W_LDS ? 4 : 1][W_LDS ? WAVE : 1];
            Images img[G];
        } s;
        f32x4 ex[G > 1 ? 4 : 1][G > 1 ? NEX : 1][WAVE];   // at the end
    } lds;
    auto &s_R = lds.s.R, &s_L = lds.s.L;
    const int lane = threadIdx.x & 63, group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6 & 3);
    auto &s_x = lds.s.img[group].x;
    auto &s_row = lds.s.img[group].row;
    auto &s_mid = lds.s.img[group].mid;
    const Lane L;
    const int cw = blockIdx.x * 64 + 16 * w;   // this wavefront's channel j is cw + j
    const long ntiles = M / TOK;
    const long lo = ((long)blockIdx.y * G + group) * tiles_per_split;
    const long hi = lo + tiles_per_split < ntiles ? lo + tiles_per_split : ntiles;   // (a last group's range can be empty)
    const bf16x4 eye = identity_bf16(L);
    const int cl = cw + 4 * L.g;          // the four contiguous channels of this lane in token layout

    f32x4 al, be[4];
    al = to_f32(*reinterpret_cast<const bf16x4*>(alpha + cl));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        be[k] = to_f32(*reinterpret_cast<const bf16x4*>(beta + (long)k * C + cl));
#pragma unroll
        for (int hh = 0; hh < HH; hh++) {
            // F(R_k[c.., 32hh ..]) lane = channel, mid indices 32hh + 8g .. 8g+7
            const bf16x8 fr = *reinterpret_cast<const bf16x8*>(R + ((long)k * C + cw + L.n) * D + 32 * hh + 8 * L.g);
            // L is [4D, C]: rows kD + 32hh + dmap(jj, n), four contiguous channels per lane, transposed on the matrix cores
            const bf16x8 fl = __builtin_shufflevector(
                transpose(*reinterpret_cast<const bf16x4*>(Lw + (long)(k * D + 32 * hh + dmap(0, L.n)) * C + cl), eye),
                transpose(*reinterpret_cast<const bf16x4*>(Lw + (long)(k * D + 32 * hh + dmap(1, L.n)) * C + cl), eye), 0, 1, 2, 3, 4, 5, 6, 7);
            if constexpr (W_LDS) {
                if (G == 1 || k * G / 4 == group) {   // (read behind the first barrier)
                    s_R[w][k][lane] = fr;
                    s_L[w][k][lane] = fl;
                }
            } else {
                r_R[k][hh] = fr;
                r_L[k][hh] = fl;
            }
        }
    }
    // F(dR_k[c.., 32hh + dmap(jj, .)]) lane = channel;  F(dL[kD + 32hh + dmap(jj, .), c..]) lane = mid index; [k][2hh + jj]
    f32x4 accR[4][2 * HH], accL[4][2 * HH];
    f32x4 vbeta[4], valpha = zero4();   // per-token partial sums, lane = token
    f32x4 carry = zero4();              // lane 15: the shifted term of the first token of the tile above
#pragma unroll
    for (int k = 0; k < 4; k++) {
        vbeta[k] = zero4();
#pragma unroll
        for (int j = 0; j < 2 * HH; j++) accR[k][j] = accL[k][j] = zero4();
    }
    // The streamed operands of a tile - 17 rows of x (one above the tile), 16 rows of each dy, of bmid and of dpre,
    // 18 KiB - are fetched ONCE per block with full 128-byte lines (16 bytes per thread, five loads each), parked in
    // registers for a tile, and written to one of two LDS images from which the wavefronts take their pieces.
    // (Each wavefront fetching its own 32-byte pieces of the rows, and all four the same rows of bmid and dpre,
    // moved four times the bytes between L2 and the compute units and ran at the rate of that link.)
    const int t = threadIdx.x & 255;
    auto stage_tile = [&](long tile) { return tile < lo ? lo : tile; };   // (past the range: loaded and never used)
    // bmid / dpre: 16 rows of 4D elements, 8 per thread and pass, HH passes
    auto mid_row = [&](int ps) { return (8 * t + 2048 * ps) / (4 * D); };
    auto mid_col = [&](int ps) { return (8 * t + 2048 * ps) % (4 * D); };
    const int row_thread = ((t & 127) >> 3) * C + blockIdx.x * 64 + 8 * (t & 7);   // dy: 8 threads per row, two arrays per pass
    const __bf16* __restrict__ dya = t < 128 ? dy.p[0] : dy.p[1];
    const __bf16* __restrict__ dyb = t < 128 ? dy.p[2] : dy.p[3];
    const int xrow = (t >> 3) - 1;                                       // x: rows -1 .. 15, threads 0 .. 135
    bf16x8 g_bm[HH], g_dp[HH], g_dya, g_dyb, g_x;
    auto fetch = [&](long tile) {
        tile = stage_tile(tile);
        const long m0 = tile * TOK;
#pragma unroll
        for (int ps = 0; ps < HH; ps++) {
            g_bm[ps] = *reinterpret_cast<const bf16x8*>(bmid + m0 * (4 * D) + 8 * t + 2048 * ps);
            g_dp[ps] = *reinterpret_cast<const bf16x8*>(dpre + m0 * (4 * D) + 8 * t + 2048 * ps);
        }
        g_dya = *reinterpret_cast<const bf16x8*>(dya + m0 * C + row_thread);
        g_dyb = *reinterpret_cast<const bf16x8*>(dyb + m0 * C + row_thread);
        if (t < 17 * 8) {
            const long m = m0 + xrow > 0 ? m0 + xrow : 0;   // (the row above token 0 is masked at the use)
            g_x = *reinterpret_cast<const bf16x8*>(x + m * C + blockIdx.x * 64 + 8 * (t & 7));
        }
    };
    auto park = [&](int buf) {
#pragma unroll
        for (int ps = 0; ps < HH; ps++) {
            *reinterpret_cast<bf16x8*>(&s_mid[buf][0][mid_row(ps) * MID_LD + mid_col(ps)]) = g_bm[ps];
            *reinterpret_cast<bf16x8*>(&s_mid[buf][1][mid_row(ps) * MID_LD + mid_col(ps)]) = g_dp[ps];
        }
        *reinterpret_cast<bf16x8*>(&s_row[buf][t < 128 ? 0 : 1][((t & 127) >> 3) * ROW_LD + 8 * (t & 7)]) = g_dya;
        *reinterpret_cast<bf16x8*>(&s_row[buf][t < 128 ? 2 : 3][((t & 127) >> 3) * ROW_LD + 8 * (t & 7)]) = g_dyb;
        if (t < 17 * 8) *reinterpret_cast<bf16x8*>(&s_x[buf][(t >> 3) * ROW_LD + 8 * (t & 7)]) = g_x;
    };
    // One tile, out of LDS image buf.  tpos: position of its first token in the sequence.  KEEP = false is the
    // warm-up tile, which only produces the carry.
    auto body = [&](long tile, int tpos, int buf, auto keep_c) {
        constexpr bool KEEP = decltype(keep_c)::value;
        const bool has_prev = (tpos + L.n) != 0;
        const bool chain = tpos != 0;   // the tile below is followed by this tile's first token in the same sequence
        const int piece = 16 * w + 4 * L.g;
        const bf16x4 zero = {};
        const f32x4 xv = to_f32(*reinterpret_cast<const bf16x4*>(&s_x[buf][(L.n + 1) * ROW_LD + piece]));
        const bf16x4 xp = *reinterpret_cast<const bf16x4*>(&s_x[buf][L.n * ROW_LD + piece]);
        const f32x4 xxv = to_f32(has_prev ? xp : zero) - xv;
        bf16x4 aT;
        if constexpr (KEEP) aT = transpose(to_bf16(xv + xxv * al), eye);   // F(a^T) lane = channel
        f32x4 da = zero4(), dxx = zero4(), dxd = zero4();
#pragma unroll
        for (int k = 0; k < 4; k++) {
            bf16x8 bm[HH], dp[HH];
            f32x4 c = be[k];
#pragma unroll
            for (int hh = 0; hh < HH; hh++) {
                bm[hh] = *reinterpret_cast<const bf16x8*>(&s_mid[buf][0][L.n * MID_LD + k * D + 32 * hh + 8 * L.g]);
                dp[hh] = *reinterpret_cast<const bf16x8*>(&s_mid[buf][1][L.n * MID_LD + k * D + 32 * hh + 8 * L.g]);
                bf16x8 fr, fl;
                if constexpr (W_LDS) {
                    fr = s_R[w][k][lane];
                    fl = s_L[w][k][lane];
                } else {
                    fr = r_R[k][hh];
                    fl = r_L[k][hh];
                }
                c = mma8(c, fr, bm[hh]);     // F(c_k) lane = token, reg = channel
                da = mma8(da, fl, dp[hh]);   // F(dpre L)
            }
            const f32x4 d = to_f32(*reinterpret_cast<const bf16x4*>(&s_row[buf][k][L.n * ROW_LD + piece]));
            dxx += d * c;
            dxd += d;
            if constexpr (KEEP) {
                const f32x4 dc = d * xxv;
                vbeta[k] += dc;
                const bf16x4 dcT = transpose(to_bf16(dc), eye);   // F(dc^T) lane = channel, reg = token
                // F(bmid_k^T), F(dpre_k^T) halves: lane = mid index 32hh + dmap(jj, n), reg = token
#pragma unroll
                for (int hh = 0; hh < HH; hh++) {
                    accR[k][2 * hh] = mma(accR[k][2 * hh], transpose(__builtin_shufflevector(bm[hh], bm[hh], 0, 1, 2, 3), eye), dcT);   // + F(dc^T bmid_k)
                    accR[k][2 * hh + 1] = mma(accR[k][2 * hh + 1], transpose(__builtin_shufflevector(bm[hh], bm[hh], 4, 5, 6, 7), eye), dcT);
                    accL[k][2 * hh] = mma(accL[k][2 * hh], aT, transpose(__builtin_shufflevector(dp[hh], dp[hh], 0, 1, 2, 3), eye));    // + F(dpre_k^T a)
                    accL[k][2 * hh + 1] = mma(accL[k][2 * hh + 1], aT, transpose(__builtin_shufflevector(dp[hh], dp[hh], 4, 5, 6, 7), eye));
                }
            }
        }
        dxx += da * al;
        dxd += da;
        f32x4 o;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float rot = row_rot<1>(dxx[r]);   // token n+1's term; lane 15 gets the tile's first token
            o[r] = dxd[r] - dxx[r] + (L.n < TOK - 1 ? rot : carry[r]);
            carry[r] = chain ? rot : 0.f;
        }
        if constexpr (KEEP) {
            *reinterpret_cast<bf16x4*>(dx + (tile * TOK + L.n) * C + cl) = to_bf16(o);
            valpha += da * xxv;
        }
    };
    int tpos = (int)((unsigned)(hi - 1) % ((unsigned)T / TOK)) * TOK;
    const bool warm = hi < ntiles && tpos + TOK != T;   // the token after the range continues the sequence
    // Iteration i works on image i&1 while the registers hold the tile after it, fetched during iteration i-1; they
    // are written to the other image (last read before the previous barrier) and refilled for the tile after that.
    long next = warm ? hi : hi - 1;   // the tile the registers are fetched for
    const bool active = G == 1 || lo < hi;
    if (active) {
        fetch(next);
        park(0);
        fetch(--next);
    }
    __syncthreads();
    int it = 0;
    if (active && warm) {
        park(1);
        fetch(--next);
        body(hi, tpos + TOK, 0, std::false_type{});
        __syncthreads();
        it = 1;
    }
    for (long tile = hi - 1; tile >= lo; tile--, it++) {
        park((it + 1) & 1);
        fetch(--next);
        body(tile, tpos, it & 1, std::true_type{});
        __syncthreads();
        tpos = tpos >= TOK ? tpos - TOK : T - TOK;
    }
    if constexpr (G > 1) {
        for (; it < tiles_per_split + 1; it++) __syncthreads();   // the same number of barriers for every group
        static_assert(G == 2 && sizeof(lds.ex) <= sizeof(lds.s), "");
        f32x4* const ex = &lds.ex[w][0][lane];
        if (group == 1) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
#pragma unroll
                for (int j = 0; j < 2 * HH; j++) {
                    ex[(4 * HH * k + j) * WAVE] = accR[k][j];
                    ex[(4 * HH * k + 2 * HH + j) * WAVE] = accL[k][j];
                }
                ex[(16 * HH + k) * WAVE] = vbeta[k];
            }
            ex[(16 * HH + 4) * WAVE] = valpha;
        }
        __syncthreads();
        if (group == 1) return;
#pragma unroll
        for (int k = 0; k < 4; k++) {
#pragma unroll
            for (int j = 0; j < 2 * HH; j++) {
                accR[k][j] += ex[(4 * HH * k + j) * WAVE];
                accL[k][j] += ex[(4 * HH * k + 2 * HH + j) * WAVE];
            }
            vbeta[k] += ex[(16 * HH + k) * WAVE];
        }
        valpha += ex[(16 * HH + 4) * WAVE];
    }
    // this block's partial record: dR [4][64][D], dL [4D][64], dbeta [4][64], dalpha [64]
    float* out = partial + ((long)blockIdx.y * gridDim.x + blockIdx.x) * P::TOTAL;
    const int jw = 16 * w;   // first channel of this wavefront inside the block
#pragma unroll
    for (int k = 0; k < 4; k++) {
#pragma unroll
        for (int j = 0; j < 2 * HH; j++) {
            const int hh = j / 2, jj = j % 2;
            *reinterpret_cast<f32x4*>(out + (k * 64 + jw + L.n) * D + 32 * hh + dmap(jj, 4 * L.g)) = accR[k][j];
            *reinterpret_cast<f32x4*>(out + P::DR + (k * D + 32 * hh + dmap(jj, L.n)) * 64 + jw + 4 * L.g) = accL[k][j];
        }
        f32x4 sb;
#pragma unroll
        for (int r = 0; r < 4; r++) sb[r] = row_sum(vbeta[k][r]);
        if (L.n == 0) *reinterpret_cast<f32x4*>(out + P::DR + P::DL + k * 64 + jw + 4 * L.g) = sb;
    }
    f32x4 sa;
#pragma unroll
    for (int r = 0; r < 4; r++) sa[r] = row_sum(valpha[r]);
    if (L.n == 0) *reinterpret_cast<f32x4*>(out + P::DR + P::DL + P::DBETA + jw + 4 * L.g) = sa;
}

// Sums the partial records over the token splits and scatters them to dR [4][C][D], dL [4D][C], dbeta [4][C], dalpha [C] (all
// fp32): a thread has four elements of the record and an eighth of the records; the order of the additions is fixed.  (All
// records to a thread, four at a time: the same time at few records, 75 us instead of 8 for the 512 of 65536 tokens x 64.)
constexpr int REDUCE_SHARES = 8, REDUCE_COLS = 256 / REDUCE_SHARES;
template <int D>
__global__ __launch_bounds__(256) void ddlerp_param_reduce_kernel(int C, int nsplit, const float* __restrict__ partial,
                                                                  float* __restrict__ dR, float* __restrict__ dL,
                                                                  float* __restrict__ dbeta,
                                                                  float* __restrict__ dalpha) {
    using P = ParamPartial<D>;
    __shared__ f32x4 part[REDUCE_SHARES][REDUCE_COLS];
    const int ncb = C / 64;
    const int cblk = blockIdx.y;
    const int c0 = cblk * 64;
    const int col = threadIdx.x % REDUCE_COLS, share = threadIdx.x / REDUCE_COLS;
    const int e = 4 * (blockIdx.x * REDUCE_COLS + col);
    f32x4 s = zero4();
    if (e < P::TOTAL) {
        const float* src = partial + (long)cblk * P::TOTAL + e;
        const long pitch = (long)ncb * P::TOTAL;
#pragma unroll 4
        for (int sp = share; sp < nsplit; sp += REDUCE_SHARES) s += *reinterpret_cast<const f32x4*>(src + sp * pitch);
    }
    part[share][col] = s;
    __syncthreads();
    if (share != 0 || e >= P::TOTAL) return;
#pragma unroll
    for (int i = 1; i < REDUCE_SHARES; i++) s += part[i][col];
    float* dst;
    if (e < P::DR) {
        const int d = e % D, c = (e / D) % 64, k = e / (64 * D);
        dst = dR + ((long)k * C + c0 + c) * D + d;
    } else if (e < P::DR + P::DL) {
        const int f = e - P::DR;
        const int c = f % 64, j = f / 64;
        dst = dL + (long)j * C + c0 + c;
    } else if (e < P::DR + P::DL + P::DBETA) {
        const int f = e - P::DR - P::DL;
        dst = dbeta + (long)(f / 64) * C + c0 + f % 64;
    } else {
        dst = dalpha + c0 + e - P::DR - P::DL - P::DBETA;
    }
    *reinterpret_cast<f32x4*>(dst) = s;
}

// ------------------------------------------------------------------------------------------------
// The four streams of ONE token per sequence whose predecessor is carried from an earlier call, in fp32 on the parameters
// as they are (the kernels above round them, and the hidden activation, to bf16; a piece's first token decides what every
// later token of a continued sequence meets, and is not rounded twice).  Bound by the launches: 128 x 768 + 4 x 768 x 32
// weights spread over 32 and 12 blocks per sequence, 64 lanes on one row of L, then a channel per lane and a stream per
// wavefront: 3.1 + 3.3 us at two sequences.  Elements one by one: parameters of any alignment.
// ------------------------------------------------------------------------------------------------
template <class X, class P>   // element types of the tokens and of the parameters
__global__ __launch_bounds__(256) void first_mid_kernel(int C, int D4, const X* __restrict__ x, long x_seq, const X* __restrict__ x_prev,
                                                        const P* __restrict__ alpha, const P* __restrict__ Lw, float* __restrict__ mid) {
    const int lane = threadIdx.x & 63, m = blockIdx.y * 4 + (threadIdx.x >> 6), b = blockIdx.x;   // a wavefront per hidden unit
    const X *xr = x + (long)b * x_seq, *pr = x_prev + (long)b * C;
    const P* lr = Lw + (long)m * C;
    float acc = 0.f;
#pragma unroll 6
    for (int c = lane; c < C; c += 64) {
        const float cur = (float)xr[c];
        acc += (cur + ((float)pr[c] - cur) * (float)alpha[c]) * (float)lr[c];
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
    if (lane == 0) mid[(long)b * D4 + m] = tanhf(acc);
}
template <class X, class P, int D>
__global__ __launch_bounds__(256) void first_streams_kernel(int C, const X* __restrict__ x, long x_seq, const X* __restrict__ x_prev,
                                                            const P* __restrict__ R, const P* __restrict__ beta, const float* __restrict__ mid,
                                                            __bf16* __restrict__ y, long y_stream, long y_seq) {
    const int c = blockIdx.y * 64 + (threadIdx.x & 63), b = blockIdx.x;
    const int k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const P* r = R + ((long)k * C + c) * D;
    const float* h = mid + ((long)b * 4 + k) * D;   // (the same for all lanes)
    const float cur = (float)x[(long)b * x_seq + c], prev = (float)x_prev[(long)b * C + c];
    float coeff = (float)beta[(long)k * C + c];
#pragma unroll
    for (int j = 0; j < D; j++) coeff += h[j] * (float)r[j];
    y[k * y_stream + (long)b * y_seq + c] = (__bf16)(cur + (prev - cur) * coeff);
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
namespace {
constexpr size_t A256(size_t x) { return (x + 255) / 256 * 256; }
// Token ranges of the second backward pass: two groups per compute unit of an MI355X (256) over the channel
// blocks, at least eight tiles each (every group spends one more tile on its carry, and a block writes a 66 KiB record
// that the reduction reads back).
int param_splits(long M, int ncb) {
    const long ntiles = M / TOK;
    long s = ntiles / 8;
    const long cap = 2 * compute_units() / ncb > 0 ? 2 * compute_units() / ncb : 1;
    if (s > cap) s = cap;
    if (s < 1) s = 1;
    return (int)s;
}
// token-tile ranges of forward 2: as many blocks over the channel blocks as the machine holds at once (at rank 32 LDS and
// registers allow three per compute unit), at least four tiles (one per wavefront) each.  Two streams' rows in LDS, two blocks
// per compute unit, in one round / in two: 14.4 / 15.9 us instead of 13.6 at 8192 tokens x 768 channels
struct StreamSplit {
    int nsplit, tiles_per_split;
};
StreamSplit stream_splits(long M, int ncb, int slots) {
    const long ntiles = M / TOK;
    long s = slots / ncb > 0 ? slots / ncb : 1;
    if (s > ntiles / 4) s = ntiles / 4;
    if (s < 1) s = 1;
    return {(int)s, (int)((ntiles + s - 1) / s)};
}
}  // namespace

bool ddlerp_rank_supported(int D) { return D == 32 || D == 64; }

size_t ddlerp_bwd_workspace_bytes(long M, int C, int D) {
    const int ncb = C / 64;
    const size_t dpre = A256((size_t)M * 4 * D * 2);
    const size_t record = D == 64 ? ParamPartial<64>::TOTAL : ParamPartial<32>::TOTAL;
    const size_t partial = A256((size_t)param_splits(M, ncb) * ncb * record * 4);
    return dpre + partial;
}

namespace {
// up to two blocks per compute unit of the kernel for few tokens; us, that one / the other: 768 channels, 256 tokens 7.3 / 10.3,
// 1024 7.5 / 10.4, 4096 10.9 / 10.7; 2048 channels, 4096 18.7 / 21.5
bool few_tokens(long ntiles) { return (ntiles + 1) / 2 * 4 <= 2 * compute_units(); }
template <int D>
void forward_rank(long M, int T, int C, const void* x, const void* alpha, const void* Lw, const void* R, const void* beta,
                  void* bmid, void* bder, void* y, hipStream_t stream) {
    auto c = [](const void* p) { return static_cast<const __bf16*>(p); };
    // four tiles per block when that still gives every compute unit a block, else two; us at 768 channels, four / two: 16384
    // tokens 17.5 / 17.0, 32768 28.5 / 31.8.  (Backward 1 takes two at any size: 35.4 / 34.5 and 81 / 77, 65536 x 64 21.5 / 18.7.)
    const long ntiles = M / TOK;
    if (few_tokens(ntiles))
        hipLaunchKernelGGL((ddlerp_fwd_mid_few_kernel<D, 4, 2>), dim3((unsigned)((ntiles + 1) / 2), 4), dim3(256), 0, stream, M, T, C, c(x),
                           c(alpha), c(Lw), static_cast<__bf16*>(bmid), static_cast<__bf16*>(bder));
    else if (ntiles >= 4 * 256)
        hipLaunchKernelGGL((ddlerp_fwd_mid_kernel<D, 4>), dim3((unsigned)((ntiles + 3) / 4)), dim3(256), 0, stream, M, T, C,
                           c(x), c(alpha), c(Lw), static_cast<__bf16*>(bmid), static_cast<__bf16*>(bder));
    else
        hipLaunchKernelGGL((ddlerp_fwd_mid_kernel<D, 2>), dim3((unsigned)((ntiles + 1) / 2)), dim3(256), 0, stream, M, T, C,
                           c(x), c(alpha), c(Lw), static_cast<__bf16*>(bmid), static_cast<__bf16*>(bder));
    const StreamSplit sp = stream_splits(M, C / 64, 3 * compute_units());
    hipLaunchKernelGGL(ddlerp_fwd_out2_kernel<D>, dim3(C / 64, sp.nsplit), dim3(256), 0, stream, M, T, C, sp.tiles_per_split,
                       c(x), c(R), c(beta), c(bmid), static_cast<__bf16*>(y));
}

template <int D>
void backward_rank(long M, int T, int C, const void* x, const void* alpha, const void* Lw, const void* R, const void* beta,
                   const void* bmid, const void* bder, const void* const dy4[4], void* dx, void* dalpha, void* dL, void* dR,
                   void* dbeta, void* workspace, hipStream_t stream) {
    auto c = [](const void* p) { return static_cast<const __bf16*>(p); };
    const Dy4 dy{{c(dy4[0]), c(dy4[1]), c(dy4[2]), c(dy4[3])}};
    const int ncb = C / 64;
    char* p = static_cast<char*>(workspace);
    __bf16* dpre = reinterpret_cast<__bf16*>(p); p += A256((size_t)M * 4 * D * 2);
    float* partial = reinterpret_cast<float*>(p);
    const int tiles_per_split = (int)((M / TOK + param_splits(M, ncb) - 1) / param_splits(M, ncb));
    const int nsplit = (int)((M / TOK + tiles_per_split - 1) / tiles_per_split);   // no empty range: every block writes a record

    hipLaunchKernelGGL((ddlerp_bwd_mid_kernel<D, 2>), dim3((unsigned)((M / TOK + 1) / 2)), dim3(256), 0, stream, M, T, C, c(x), dy,
                       c(R), c(bder), dpre);
    // Two groups to a block where two would share a compute unit anyway (registers allow it at rank 32): half the records.  Second
    // pass + sums, us, two / one: 8192 tokens x 768 channels 39.1 / 42.6, 4096 x 768 29.8 / 32.3; where a group would have a compute
    // unit to itself, or the blocks are more than a round, two to a block are slower: 1024 x 768 26.2 / 20.5, 8192 x 1536 77 / 59
    const bool two = D == 32 && (long)ncb * nsplit > compute_units() && (long)ncb * ((nsplit + 1) / 2) <= compute_units();
    const int records = two ? (nsplit + 1) / 2 : nsplit;
    if constexpr (D == 32) {
        if (two)
            hipLaunchKernelGGL((ddlerp_bwd_main_kernel<D, 2>), dim3(ncb, records), dim3(512), 0, stream, M, T, C, tiles_per_split, c(x), dy,
                               c(alpha), c(Lw), c(R), c(beta), c(bmid), dpre, static_cast<__bf16*>(dx), partial);
    }
    if (!two)
        hipLaunchKernelGGL((ddlerp_bwd_main_kernel<D, 1>), dim3(ncb, records), dim3(256), 0, stream, M, T, C, tiles_per_split, c(x), dy,
                           c(alpha), c(Lw), c(R), c(beta), c(bmid), dpre, static_cast<__bf16*>(dx), partial);
    hipLaunchKernelGGL(ddlerp_param_reduce_kernel<D>, dim3((ParamPartial<D>::TOTAL / 4 + REDUCE_COLS - 1) / REDUCE_COLS, ncb), dim3(256), 0,
                       stream, C, records, partial,
                       static_cast<float*>(dR), static_cast<float*>(dL), static_cast<float*>(dbeta),
                       static_cast<float*>(dalpha));
}
}  // namespace

namespace {
template <class X, class P, int D>
void first_tokens(int B, int C, const FirstTokens& t, void* y, float* mid, hipStream_t stream) {
    auto x = [](const void* p) { return static_cast<const X*>(p); };
    auto w = [](const void* p) { return static_cast<const P*>(p); };
    hipLaunchKernelGGL((first_mid_kernel<X, P>), dim3(B, D), dim3(256), 0, stream, C, 4 * D, x(t.x), t.x_seq, x(t.x_prev), w(t.alpha), w(t.Lw), mid);
    hipLaunchKernelGGL((first_streams_kernel<X, P, D>), dim3(B, C / 64), dim3(256), 0, stream, C, x(t.x), t.x_seq, x(t.x_prev), w(t.R), w(t.beta),
                       mid, static_cast<__bf16*>(y), t.y_stream, t.y_seq);
}
template <int D>
void first_tokens_rank(int B, int C, const FirstTokens& t, void* y, float* mid, hipStream_t stream) {
    if (t.x_f32 && t.param_f32) first_tokens<float, float, D>(B, C, t, y, mid, stream);
    else if (t.x_f32) first_tokens<float, __bf16, D>(B, C, t, y, mid, stream);
    else if (t.param_f32) first_tokens<__bf16, float, D>(B, C, t, y, mid, stream);
    else first_tokens<__bf16, __bf16, D>(B, C, t, y, mid, stream);
}
}  // namespace

// (the callers have checked ddlerp_rank_supported(D))
void launch_ddlerp_first(int B, int C, int D, const FirstTokens& t, void* y, void* workspace, hipStream_t stream) {
    if (D == 64) first_tokens_rank<64>(B, C, t, y, static_cast<float*>(workspace), stream);
    else first_tokens_rank<32>(B, C, t, y, static_cast<float*>(workspace), stream);
}

void launch_ddlerp_forward(long M, int T, int C, int D, const void* x, const void* alpha, const void* Lw, const void* R, const void* beta, void* bmid, void* bder, void* y, hipStream_t stream) {
    if (D == 64) forward_rank<64>(M, T, C, x, alpha, Lw, R, beta, bmid, bder, y, stream);
    else forward_rank<32>(M, T, C, x, alpha, Lw, R, beta, bmid, bder, y, stream);
}

void launch_ddlerp_backward(long M, int T, int C, int D, const void* x, const void* alpha, const void* Lw, const void* R,
                            const void* beta, const void* bmid, const void* bder, const void* const dy4[4], void* dx,
                            void* dalpha,
                            void* dL, void* dR, void* dbeta, void* workspace, hipStream_t stream) {
    if (D == 64) backward_rank<64>(M, T, C, x, alpha, Lw, R, beta, bmid, bder, dy4, dx, dalpha, dL, dR, dbeta, workspace, stream);
    else backward_rank<32>(M, T, C, x, alpha, Lw, R, beta, bmid, bder, dy4, dx, dalpha, dL, dR, dbeta, workspace, stream);
}

}  // namespace wkv
