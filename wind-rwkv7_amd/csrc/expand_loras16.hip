// expand_loras at rank 16, the rank of the time mixer's four LoRAs: forward for heads of 64 channels, backward for heads of any
// size.  Same mathematics as expand_loras.hip; a file of its own because it is compiled with matrix results in ordinary
// registers, an option that crashes this compiler release on the kernels there.
#include "device_info.hpp"
#include "expand_loras_tile.hpp"

namespace wkv {

namespace {
constexpr int TOK = LORA_TOK;
constexpr int D = 16;
constexpr int REC = 4 * HEAD * D + 4 * HEAD;   // floats of a partial record: dW [4][64][16], then dbias [4][64]
}  // namespace

// ------------------------------------------------------------------------------------------------
// forward: block = (head, range of token tiles).  The head's weights and biases are staged in LDS once and each wavefront
// walks its tiles with the next tile's inputs already in flight; tiles move as whole lines through the wavefront's part of LDS
// (row_lines.hpp).
// 16 rows per instruction and two rounds of two blocks per compute unit took 20.9, 22.1, 47 us at 7056, 8192, 16384 tokens x 768
// channels, 49.5 at 8192 x 1536; whole lines and three blocks per compute unit in one round 16.9, 17.9, 35.9, 36.4 (two rounds of
// either two or three: 18.9 and 19.6 at 7056).  The bytes are 13, 15, 30, 30 at the rate of a copy, the instructions, a fifth of
// them transcendental, 11 at 8192 x 768.  Stored through the L2 (store_through_at) 10.0 instead of 11.2 us in a prompt of 2016 tokens, 16.4 instead
// of 20.0 in a block of 8192.
// ------------------------------------------------------------------------------------------------
// PADDED: a sequence's last chunk belongs to the tokens behind its whole chunks (`kept`, [3][sequences][16][C], takes its w, k and b) and
// gets what leaves the recurrence's state as it is instead: decay 1, k = b = 0.  (As a launch of its own behind this one a prompt of
// 2 x 1003 tokens took 113.9 us, so 111.8.)
struct PaddedRows {
    int chunks;   // of a sequence
    long plane;
    __bf16* kept;
};
template <bool PADDED>
__global__ __launch_bounds__(256) void expand_loras_fwd16_kernel(long M, int C, int tiles_per_split,
                                                                 const __bf16* __restrict__ w_in,
                                                                 const __bf16* __restrict__ k_in, LoraIn in, LoraW lw,
                                                                 __bf16* __restrict__ w_out, __bf16* __restrict__ k_out,
                                                                 __bf16* __restrict__ kk_out, __bf16* __restrict__ b_out,
                                                                 const PaddedRows padded) {
    __shared__ bf16x4 sW[4 * NBLK][WAVE];    // F(W_i[c0 + 16cb .., :])    lane = channel, reg = rank index
    __shared__ __attribute__((aligned(16))) float sBias[4][HEAD];
    __shared__ bf16x8 s_tile[4][2][TOK * 8];
    const int lane = threadIdx.x & 63, l8 = lane >> 3, piece = lane & 7;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane L;
    const int h = blockIdx.x, split = blockIdx.y;
    const int c0 = h * HEAD;
    const long ntiles = M / TOK;
    const long tile_begin = (long)split * tiles_per_split;
    const long tile_end = tile_begin + tiles_per_split < ntiles ? tile_begin + tiles_per_split : ntiles;
    const unsigned row_bytes = 2 * C, lane_bytes = l8 * row_bytes + 16 * piece, act_bytes = 2 * (D * L.n + 4 * L.g);
    auto(&buf)[2][TOK * 8] = s_tile[wave];

    struct TileIn {
        bf16x8 wi[2], ki[2];
        bf16x4 act[4];
    };
    auto fetch = [&](long tile) {
        TileIn t;
        const long m0 = tile * TOK;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            t.wi[i] = piece_at(w_in + (m0 * C + c0), lane_bytes + 8 * i * row_bytes);
            t.ki[i] = piece_at(k_in + (m0 * C + c0), lane_bytes + 8 * i * row_bytes);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) t.act[i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const char*>(in.p[i] + m0 * D) + act_bytes);
        return t;
    };
    long tile = tile_begin + wave;
    TileIn nxt;
    if (tile < tile_end) nxt = fetch(tile);
    // channel blocks follow the interleaved order of chan16 (frag.hpp): nothing here depends on which 16 channels form a block
#pragma unroll
    for (int cb = 0; cb < NBLK; cb++)
        sW[wave * NBLK + cb][lane] = *reinterpret_cast<const bf16x4*>(lw.W[wave] + (long)(c0 + chan16(cb, L.n)) * D + 4 * L.g);
    sBias[wave][lane] = (float)lw.bias[wave][c0 + lane];
    __syncthreads();
    auto bias4 = [&](int i, int cb) { return *reinterpret_cast<const f32x4*>(&sBias[i][chan16(cb, 4 * L.g)]); };
    bool last = false;   // PADDED: this tile is a sequence's last chunk
    long kept_at = 0;
    auto put = [&](__bf16* p, unsigned bytes, int plane, bf16x8 v) {   // plane: w, k, b, or negative
        if (PADDED && last && plane >= 0) {
            store_through_at(padded.kept + (plane * padded.plane + kept_at), bytes, v);
            const __bf16 none = (__bf16)(plane == 0 ? -80.f : 0.f);
            v = (bf16x8){none, none, none, none, none, none, none, none};
        }
        store_through_at(p, bytes, v);
    };
    auto store = [&](__bf16* p0, const TileB& t0, int plane0, __bf16* p1, const TileB& t1, int plane1, long off) {   // two tiles
#pragma unroll
        for (int pr = 0; pr < 2; pr++) {
            buf[0][piece_slot(L.n, 4 * pr + L.g)] = join(t0.f[2 * pr], t0.f[2 * pr + 1]);
            buf[1][piece_slot(L.n, 4 * pr + L.g)] = join(t1.f[2 * pr], t1.f[2 * pr + 1]);
        }
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < 2; i++) {
            put(p0 + off, lane_bytes + 8 * i * row_bytes, plane0, buf[0][piece_slot(l8 + 8 * i, piece)]);
            put(p1 + off, lane_bytes + 8 * i * row_bytes, plane1, buf[1][piece_slot(l8 + 8 * i, piece)]);
        }
        wave_lds_order();
    };
    for (; tile < tile_end; tile += 4) {
        const long off = tile * TOK * C + c0;
        if constexpr (PADDED) {
            const int sequence = (int)tile / padded.chunks;
            last = (int)tile - sequence * padded.chunks == padded.chunks - 1;
            kept_at = (long)sequence * TOK * C + c0;
        }
        bf16x4 act[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            buf[0][piece_slot(l8 + 8 * i, piece)] = nxt.wi[i];
            buf[1][piece_slot(l8 + 8 * i, piece)] = nxt.ki[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) act[i] = nxt.act[i];
        wave_lds_order();
        TileB wi, ki;
#pragma unroll
        for (int cb = 0; cb < NBLK; cb++) {
            wi.f[cb] = half_of(buf[0][piece_slot(L.n, 4 * (cb >> 1) + L.g)], cb & 1);
            ki.f[cb] = half_of(buf[1][piece_slot(L.n, 4 * (cb >> 1) + L.g)], cb & 1);
        }
        wave_lds_order();
        nxt = fetch(tile + 4 < tile_end ? tile + 4 : tile);   // past the end: the current tile again (never used)
        bf16x4 tz;
        {
            f32x4 t = to_f32(act[0]);
#pragma unroll
            for (int q = 0; q < 4; q++) t[q] = tanhf_(t[q]);
            tz = to_bf16(t);
        }
        TileF z, a;
        TileB wo, ko;
        float ss = 0.f;
#pragma unroll
        for (int cb = 0; cb < NBLK; cb++) {
            const f32x4 kin = to_f32(ki.f[cb]);
            z.f[cb] = mma(kin, sW[0 * NBLK + cb][lane], tz);
            const f32x4 pa = mma(bias4(1, cb), sW[1 * NBLK + cb][lane], act[1]);
            const f32x4 pma = mma(bias4(2, cb), sW[2 * NBLK + cb][lane], act[2]);
            const f32x4 pmk = mma(bias4(3, cb), sW[3 * NBLK + cb][lane], act[3]);
            const f32x4 u = bias4(0, cb) + to_f32(wi.f[cb]);
            f32x4 w, k;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float av = sigmoidf_(pa[q]), mav = sigmoidf_(pma[q]), mkv = sigmoidf_(pmk[q]);
                // -softplus(-u) - 0.5 = log(sigmoid(u)) - 0.5, evaluated without overflow
                w[q] = -(fmaxf(-u[q], 0.f) + log1pexp_(u[q])) - 0.5f;
                k[q] = kin[q] * (mav + av - mav * av) * __expf(w[q] * mkv);
                a.f[cb][q] = av;
                ss += z.f[cb][q] * z.f[cb][q];
            }
            wo.f[cb] = to_bf16(w);
            ko.f[cb] = to_bf16(k);
        }
        store(w_out, wo, 0, k_out, ko, 1, off);
        const float inorm = rsqrtf(fmaxf(group_sum(ss), 1e-12f));
        TileB kko, bo;
#pragma unroll
        for (int cb = 0; cb < NBLK; cb++) {
            const f32x4 kk = z.f[cb] * inorm;
            kko.f[cb] = to_bf16(kk);
            bo.f[cb] = to_bf16(-kk * a.f[cb]);
        }
        store(kk_out, kko, -1, b_out, bo, 2, off);
    }
}

// ------------------------------------------------------------------------------------------------
// backward: block = (head, range of token tiles), a tile per PAIR of wavefronts, each with 32 of the head's 64 channels.  Per
// tile the forward is computed again; dw_in, dk_in and this head's share of the four d*_in ([M, H, D], summed over heads
// afterwards: each head contributes to every rank channel) are written, and the head's weight and bias gradients accumulate in
// registers, combined over the block's two pairs at the end.  The two halves of a head meet three times per tile, through LDS:
// for the norm of z, for its backward's dot product, and for the sum of their shares of d*_in, which waits for the next tile's
// first barrier.
// A wavefront with all 64 channels holds 470 registers, alone on its SIMD, and stood still for 56 % of its time
// (instructions waiting for the results before them 34 %, memory 22 %; two such on a SIMD spilled and gained nothing): 45.9, 53.8,
// 94 us at 7056, 8192, 16384 tokens x 768 channels, 99 at 8192 x 1536.  Two wavefronts of 32 channels on a SIMD, inputs as 16 rows
// per instruction: 38.0 and 43.3 at 7056 and 8192, the vector cache busy for 62 % of the time; inputs as whole lines through LDS
// and four results of a tile in one store: 30.9, 34.2 .. 36, 62.5, 69.8.  (Three on a SIMD spill 26 registers: 55.)  8192 x 768 has 6144
// (tile, head)s for 1024 pairs of wavefronts, but 512 tiles of a head for 84 of them, seven rounds; the vector instructions
// of those take 22 us, the bytes 20.
// ------------------------------------------------------------------------------------------------
template <bool STATS>
__global__ __launch_bounds__(256, 2) void expand_loras_bwd16_kernel(long M, int C, int tiles_per_split,
                                                                 const __bf16* __restrict__ w_in,
                                                                 const __bf16* __restrict__ k_in, LoraIn in, LoraW lw,
                                                                 LoraDy dy, __bf16* __restrict__ dw_in,
                                                                 __bf16* __restrict__ dk_in, __bf16* __restrict__ din,
                                                                 float* __restrict__ partial,
                                                                 const HeadStat* __restrict__ stats, int HS) {
    constexpr int NB = NBLK / 2;   // channel blocks of a wavefront
    struct Weights {
        bf16x4 W[4][NBLK][WAVE];    // F(W_i[c0 + 16cb .., :])    lane = channel, reg = rank index
        bf16x4 WT[4][NBLK][WAVE];   // F(W_i[c0 + 16cb .., :]^T)  lane = rank index, reg = channel
        float bias[4][HEAD];
    };
    __shared__ __attribute__((aligned(16))) union {
        Weights w;
        float comb[REC];            // the second pair's sums, at the end
    } lds;
    __shared__ bf16x8 s_tile[2][2][6][TOK * 8];              // [pair][tile & 1]: w_in, k_in, dy 0 .. 3
    __shared__ f32x4 s_dact[2][2][2][WAVE];                 // [pair][half]: what the other half sums
    __shared__ float s_norm[2][2][TOK], s_dot[2][2][TOK];   // [pair][half]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), pair = wave >> 1, half = wave & 1;
    const Lane L;
    const int H = C / HEAD;
    const int h = blockIdx.x, split = blockIdx.y;
    const int c0 = h * HEAD;
    const long ntiles = M / TOK;
    const long tile_begin = (long)split * tiles_per_split;
    const long tile_end = tile_begin + tiles_per_split < ntiles ? tile_begin + tiles_per_split : ntiles;
    const bf16x4 eye = identity_bf16(L);

    // wavefront i stages LoRA i
    // channel blocks follow the interleaved order of chan16 (frag.hpp) so that tiles move with 16-byte accesses
#pragma unroll
    for (int cb = 0; cb < NBLK; cb++) {
        const bf16x4 f = *reinterpret_cast<const bf16x4*>(lw.W[wave] + (long)(c0 + chan16(cb, L.n)) * D + 4 * L.g);
        lds.w.W[wave][cb][lane] = f;
        lds.w.WT[wave][cb][lane] = transpose(f, eye);
    }
    lds.w.bias[wave][lane] = (float)lw.bias[wave][c0 + lane];
    __syncthreads();
    const int cb0 = NB * half;
    auto bias4 = [&](int i, int cb) { return *reinterpret_cast<const f32x4*>(&lds.w.bias[i][chan16(cb0 + cb, 4 * L.g)]); };
    auto weight = [&](int i, int cb) { return lds.w.W[i][cb0 + cb][lane]; };

    f32x4 dW[4][NB];   // F(dW_i[c0+16cb.., :])  lane = channel, reg = rank index
    // The four bias gradients of a channel block are token sums of du, pre_1, pre_2, pre_3.  One accumulator
    // holds all four: contract the transposed tiles, laid side by side along the token axis, with selector
    // fragments sel_i[col][t] = (col == i); column i of the result is sum_t x_i[t][c].
    f32x4 dB[NB];      // lane = channel, columns 0..3 (the lanes with g = 0) = the four bias gradients
#pragma unroll
    for (int cb = 0; cb < NB; cb++) {
        dB[cb] = zero4();
#pragma unroll
        for (int i = 0; i < 4; i++) dW[i][cb] = zero4();
    }
    bf16x4 sel[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float v = (L.n == i) ? 1.f : 0.f;
        sel[i] = to_bf16(f32x4{v, v, v, v});
    }

    // Either half fetches eight whole rows of a tile for both (six tensors of 16 bytes per lane, registers until the tile before
    // is done with).  A lane's 16 bytes of a row of results: row n, channels 32 half + 8g ..
    const int row8 = 8 * half + (lane >> 3), piece = lane & 7, slot8 = piece_slot(row8, piece);
    const unsigned in_bytes = 2 * ((unsigned)row8 * C + 8 * piece), out_bytes = 2 * ((unsigned)L.n * C + HEAD / 2 * half + 8 * L.g);
    const unsigned act_bytes = 2 * (D * L.n + 4 * L.g), din_bytes = 2 * ((unsigned)L.n * H * 4 * D + 32 * half + 8 * L.g);
    bf16x8 nxt[6];
    auto fetch = [&](long tile) {
        const long off = tile * TOK * C + c0;
        nxt[0] = piece_at(w_in + off, in_bytes);
        nxt[1] = piece_at(k_in + off, in_bytes);
#pragma unroll
        for (int i = 0; i < 4; i++) nxt[2 + i] = piece_at(dy.p[i] + off, in_bytes);
    };
    auto park = [&](int buf) {
#pragma unroll
        for (int t = 0; t < 6; t++) s_tile[pair][buf][t][slot8] = nxt[t];
    };
    bf16x4 act[4];
    auto fetch_act = [&](long tile) {
#pragma unroll
        for (int i = 0; i < 4; i++) act[i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const char*>(in.p[i] + tile * TOK * D) + act_bytes);
    };
    // a tile's d*_in of both halves, two of the four for either: own[e] of i = 2 half + e
    f32x4 own[2];
    auto flush = [&](long tile) {
        const f32x4 a = own[0] + s_dact[pair][1 - half][0][lane], b = own[1] + s_dact[pair][1 - half][1][lane];
        piece_at(din + (tile * TOK * H + h) * (4 * D), din_bytes) = join(to_bf16(a), to_bf16(b));
    };
    // Two barriers per round, the same number for both pairs: a pair without a tile in the last round only meets them.
    const int rounds = tile_end > tile_begin ? (int)((tile_end - tile_begin + 1) / 2) : 0;
    const long first = tile_begin + pair;
    const int mine = tile_end > first ? (int)((tile_end - first + 1) / 2) : 0;
    if (mine > 0) {
        fetch(first);
        fetch_act(first);
        park(0);
    }
    lds_barrier();
    long tile = first;
    for (int it = 0; it < mine; it++, tile += 2) {
        asm volatile("" ::: "memory");   // (the weights are read from LDS where they are used: kept in registers they leave no room for a second wavefront)
        const long off = tile * TOK * C + c0;
        const long next = it + 1 < mine ? tile + 2 : tile;   // past the end: the current one again (never used)
        fetch(next);
        auto tile_at = [&](int t) { return s_tile[pair][it & 1][t][piece_slot(L.n, 4 * half + L.g)]; };
        const bf16x8 wi = tile_at(0), ki = tile_at(1);
        // rank-space operands: tanh(z_in) and the transposed inputs (lane = rank index, reg = token)
        bf16x4 tz;
        {
            f32x4 t = to_f32(act[0]);
#pragma unroll
            for (int q = 0; q < 4; q++) t[q] = tanhf_(t[q]);
            tz = to_bf16(t);
        }
        // pass 1: z and the head norm
        float inorm = 0.f, proj = 0.f;
        if constexpr (STATS) {   // (a lane's 8 contiguous channels lie in one head whatever its size)
            const HeadStat hs = stats[(tile * TOK + L.n) * (C / HS) + (c0 + HEAD / 2 * half + 8 * L.g) / HS];
            inorm = hs.inorm;
            proj = hs.proj;
        }
        f32x4 z[NB];
        float ss = 0.f;
#pragma unroll
        for (int cb = 0; cb < NB; cb++) {
            z[cb] = mma(to_f32(half_of(ki, cb)), weight(0, cb), tz);
            if constexpr (!STATS) {
#pragma unroll
                for (int q = 0; q < 4; q++) ss += z[cb][q] * z[cb][q];
            }
        }
        if constexpr (!STATS) {
            ss = group_sum(ss);
            if (L.g == 0) s_norm[pair][half][L.n] = ss;
        }
        lds_barrier();
        if (it > 0) flush(tile - 2);
        if constexpr (!STATS) inorm = rsqrtf(fmaxf(s_norm[pair][0][L.n] + s_norm[pair][1][L.n], 1e-12f));

        bf16x8 g[4];
#pragma unroll
        for (int i = 0; i < 4; i++) g[i] = tile_at(2 + i);
        // pass 2: everything that does not need the projection of dkk on z
        f32x4 dkk[NB], dkin[NB];
        f32x4 dact[4] = {zero4(), zero4(), zero4(), zero4()};   // F(d in_i)  lane = token, reg = rank index
        float dot = 0.f;
        bf16x4 du_b[NB];
#pragma unroll
        for (int cb = 0; cb < NB; cb++) {
            const f32x4 kin = to_f32(half_of(ki, cb));
            const f32x4 pa = mma(bias4(1, cb), weight(1, cb), act[1]);
            const f32x4 pma = mma(bias4(2, cb), weight(2, cb), act[2]);
            const f32x4 pmk = mma(bias4(3, cb), weight(3, cb), act[3]);
            const f32x4 u = bias4(0, cb) + to_f32(half_of(wi, cb));
            f32x4 a, ma, mk, w, e, su;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                a[q] = sigmoidf_(pa[q]);
                ma[q] = sigmoidf_(pma[q]);
                mk[q] = sigmoidf_(pmk[q]);
                w[q] = -(fmaxf(-u[q], 0.f) + log1pexp_(u[q])) - 0.5f;
                e[q] = __expf(w[q] * mk[q]);
                su[q] = sigmoidf_(-u[q]);
            }
            const f32x4 kk = z[cb] * inorm;
            const f32x4 gb = to_f32(half_of(g[3], cb));
            dkk[cb] = to_f32(half_of(g[2], cb)) - gb * a;
            f32x4 da = -gb * kk;
            const f32x4 mix = ma + a - ma * a;
            const f32x4 dk = to_f32(half_of(g[1], cb)) * e;   // d/d(k_in * mix)
            const f32x4 de = dk * kin * mix;                      // d/d(w*mk), already times e
            const f32x4 dw = to_f32(half_of(g[0], cb)) + de * mk;
            const f32x4 dmk = de * w;
            du_b[cb] = to_bf16(dw * su);
            bf16x4 pT[4];
            pT[0] = transpose(du_b[cb], eye);
            dkin[cb] = dk * mix;
            const f32x4 dma = dk * kin * (1.f - a);
            da += dk * kin * (1.f - ma);
            f32x4 pre[4];
            pre[1] = da * a * (1.f - a);
            pre[2] = dma * ma * (1.f - ma);
            pre[3] = dmk * mk * (1.f - mk);
            if constexpr (!STATS) {
#pragma unroll
                for (int q = 0; q < 4; q++) dot += dkk[cb][q] * z[cb][q];
            }
#pragma unroll
            for (int i = 1; i < 4; i++) {
                const bf16x4 pb = to_bf16(pre[i]);
                pT[i] = transpose(pb, eye);
                dW[i][cb] = mma(dW[i][cb], transpose(act[i], eye), pT[i]);     // + F(pre^T in)
                dact[i] = mma(dact[i], lds.w.WT[i][cb0 + cb][lane], pb);            // + F(pre W)
            }
            dB[cb] = mma2(dB[cb], sel[0], sel[1], pT[0], pT[1]);
            dB[cb] = mma2(dB[cb], sel[2], sel[3], pT[2], pT[3]);
        }
        piece_at(dw_in + off, out_bytes) = join(du_b[0], du_b[1]);
        fetch_act(next);
        park((it + 1) & 1);   // (last read before the barrier before this one)
        if constexpr (!STATS) {
            dot = group_sum(dot);
            if (L.g == 0) s_dot[pair][half][L.n] = dot;
        }
        lds_barrier();
        if constexpr (!STATS) {   // z below the clamp has a constant norm: no gradient through it
            dot = s_dot[pair][0][L.n] + s_dot[pair][1][L.n];
            proj = (inorm < 1e6f) ? dot * inorm * inorm * inorm : 0.f;
        }

        // pass 3: the z LoRA and dk_in
        const bf16x4 tzT = transpose(tz, eye);
        bf16x4 dk_b[NB];
#pragma unroll
        for (int cb = 0; cb < NB; cb++) {
            const f32x4 pre0 = dkk[cb] * inorm - proj * z[cb];
            dk_b[cb] = to_bf16(dkin[cb] + pre0);
            const bf16x4 pb = to_bf16(pre0);
            dW[0][cb] = mma(dW[0][cb], tzT, transpose(pb, eye));
            dact[0] = mma(dact[0], lds.w.WT[0][cb0 + cb][lane], pb);
        }
        piece_at(dk_in + off, out_bytes) = join(dk_b[0], dk_b[1]);
        {   // through tanh
            const f32x4 t = to_f32(tz);
            dact[0] = dact[0] * (1.f - t * t);
        }
#pragma unroll
        for (int e = 0; e < 2; e++) {
            own[e] = half ? dact[2 + e] : dact[e];
            s_dact[pair][half][e][lane] = half ? dact[e] : dact[2 + e];
        }
    }
    bool pending = mine > 0;
    for (int it = mine; it < rounds; it++) {   // (at most once)
        lds_barrier();
        if (pending) flush(tile - 2);
        pending = false;
        lds_barrier();
    }
    lds_barrier();
    if (pending) flush(tile - 2);

    // the second pair's sums through LDS, where the weights were (nobody reads them behind the last barrier)
    auto dw_at = [&](int i, int cb) { return (i * HEAD + chan16(cb0 + cb, L.n)) * D + 4 * L.g; };
    auto db_at = [&](int i, int cb) { return 4 * HEAD * D + i * HEAD + chan16(cb0 + cb, L.n); };
    if (pair == 1) {
#pragma unroll
        for (int cb = 0; cb < NB; cb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                *reinterpret_cast<f32x4*>(lds.comb + dw_at(i, cb)) = dW[i][cb];
                if (L.g == 0) lds.comb[db_at(i, cb)] = dB[cb][i];   // this lane's channel, bias gradients 0..3 in the four registers
            }
    }
    lds_barrier();
    if (pair == 0) {
        float* out = partial + ((long)split * gridDim.x + h) * REC;
#pragma unroll
        for (int cb = 0; cb < NB; cb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                *reinterpret_cast<f32x4*>(out + dw_at(i, cb)) = dW[i][cb] + *reinterpret_cast<const f32x4*>(lds.comb + dw_at(i, cb));
                if (L.g == 0) out[db_at(i, cb)] = dB[cb][i] + lds.comb[db_at(i, cb)];
            }
    }
}

// ------------------------------------------------------------------------------------------------
// What the backward kernel's blocks leave, summed in one launch: blocks below `din_blocks` the input gradients over the heads (a
// quarter of the heads per thread, 16 bytes of a token's 128 each), the others the records over the token splits (a sixteenth of
// them per thread, four floats each).  The order of the sums is fixed.  Bound by the latency of loads that few threads wait for
// one after the other: all heads and, four at a time, all splits to a thread took 6.3 us at 8192 tokens and 12 heads, 16 at 24
// heads, 41 at 65536 tokens of one head, 512 splits; this
// way 6.0, 7.3 and 12.2
// ------------------------------------------------------------------------------------------------
constexpr int REDUCE_SHARES = 16, REDUCE_COLS = 256 / REDUCE_SHARES;
__global__ __launch_bounds__(256) void expand_loras_reduce16_kernel(long M, int H, int nsplit, int din_blocks, int param_blocks,
                                                                    const __bf16* __restrict__ din, const float* __restrict__ partial,
                                                                    LoraReduceOut out) {
    const int t = threadIdx.x;
    if (blockIdx.x < (unsigned)din_blocks) {   // (M is a multiple of 16: whole blocks of 8 tokens)
        const long m = blockIdx.x * 8L + (t >> 5);
        const int p = t & 7, share = t >> 3 & 3;
        const __bf16* src = din + m * H * 64 + 8 * p;
        f32x4 acc[2] = {zero4(), zero4()};
#pragma unroll 4
        for (int h = share; h < H; h += 4) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(src + (long)h * 64);
            acc[0] += to_f32(half_of(v, 0));
            acc[1] += to_f32(half_of(v, 1));
        }
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                acc[e][q] += __shfl_xor(acc[e][q], 8);
                acc[e][q] += __shfl_xor(acc[e][q], 16);
            }
        if (share < 2) {   // i = 2 half + e: shares 0 and 1 write one of the piece's two
            const int i = 2 * (p >> 2) + share;
            __bf16* dst = i == 0 ? out.din[0] : i == 1 ? out.din[1] : i == 2 ? out.din[2] : out.din[3];
            const long ld = i == 0 ? out.ld[0] : i == 1 ? out.ld[1] : i == 2 ? out.ld[2] : out.ld[3];
            *reinterpret_cast<bf16x4*>(dst + m * ld + 4 * (p & 3)) = to_bf16(share ? acc[1] : acc[0]);
        }
        return;
    }
    __shared__ f32x4 part[REDUCE_SHARES][REDUCE_COLS];
    const int b = blockIdx.x - din_blocks, h = b / param_blocks;
    const int col = t % REDUCE_COLS, share = t / REDUCE_COLS;
    const int e = 4 * ((b - h * param_blocks) * REDUCE_COLS + col);
    const float* src = partial + (long)h * REC + e;
    const long pitch = (long)H * REC;
    f32x4 s = zero4();
#pragma unroll 4
    for (int sp = share; sp < nsplit; sp += REDUCE_SHARES) s += *reinterpret_cast<const f32x4*>(src + sp * pitch);
    part[share][col] = s;
    __syncthreads();
    if (share != 0) return;
#pragma unroll
    for (int i = 1; i < REDUCE_SHARES; i++) s += part[i][col];
    const int r = e < 4 * HEAD * D ? e : e - 4 * HEAD * D, per = e < 4 * HEAD * D ? HEAD * D : HEAD, i = r / per;
    float* const* dst = e < 4 * HEAD * D ? out.dW : out.db;
    float* o = (i == 0 ? dst[0] : i == 1 ? dst[1] : i == 2 ? dst[2] : dst[3]) + (long)h * per + r % per;   // (of any alignment)
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = s[q];
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
// Blocks of the backward kernel per head: two fit a compute unit, all of them in one round, at least one tile per pair of
// wavefronts each (fewer where the workspace has fewer records).
int lora16_splits(long M, int H) {
    const long ntiles = M / TOK;
    long s = 2 * compute_units() / H;
    if (s > ntiles / 2) s = ntiles / 2;
    if (s < 1) s = 1;
    return (int)s;
}

void launch_loras16_forward(long M, int C, const __bf16* w_in, const __bf16* k_in, const LoraIn& in, const LoraW& lw, __bf16* const outs[4],
                            hipStream_t stream, int padded_T, void* kept) {
    // three blocks fit a compute unit, all of them in one round; at least four token tiles (one per wavefront) each
    const int H = C / HEAD;
    const long ntiles = M / TOK;
    long nsplit = 3 * compute_units() / H;
    if (nsplit > ntiles / 4) nsplit = ntiles / 4;
    if (nsplit < 1) nsplit = 1;
    const int tiles_per_split = (int)((ntiles + nsplit - 1) / nsplit);
    const PaddedRows padded{padded_T / TOK, kept ? M / padded_T * TOK * C : 0, static_cast<__bf16*>(kept)};
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(H, (unsigned)nsplit), dim3(256), 0, stream, M, C, tiles_per_split, w_in, k_in, in, lw, outs[0],
                           outs[1], outs[2], outs[3], padded);
    };
    kept ? go(expand_loras_fwd16_kernel<true>) : go(expand_loras_fwd16_kernel<false>);
}

void launch_loras16_backward(long M, int C, const __bf16* w_in, const __bf16* k_in, const LoraIn& in, const LoraW& lw, const LoraDy& dy,
                             __bf16* dw_in, __bf16* dk_in, __bf16* din, float* partial, int nsplit, const HeadStat* stats, int HS,
                             hipStream_t stream) {
    const int H = C / HEAD;
    const int tiles_per_split = (int)((M / TOK + nsplit - 1) / nsplit);
    const dim3 grid(H, nsplit), block(256);
    if (stats)
        hipLaunchKernelGGL(expand_loras_bwd16_kernel<true>, grid, block, 0, stream, M, C, tiles_per_split, w_in, k_in, in, lw, dy, dw_in, dk_in,
                           din, partial, stats, HS);
    else
        hipLaunchKernelGGL(expand_loras_bwd16_kernel<false>, grid, block, 0, stream, M, C, tiles_per_split, w_in, k_in, in, lw, dy, dw_in,
                           dk_in, din, partial, stats, HS);
}

void launch_loras16_reduce(long M, int C, int nsplit, const __bf16* din, const float* partial, const LoraReduceOut& out, hipStream_t stream) {
    static_assert(REC % (4 * REDUCE_COLS) == 0, "whole blocks");
    const int H = C / HEAD, din_blocks = (int)(M / 8), param_blocks = REC / (4 * REDUCE_COLS);
    hipLaunchKernelGGL(expand_loras_reduce16_kernel, dim3(din_blocks + param_blocks * H), dim3(256), 0, stream, M, H, nsplit,
                       din_blocks, param_blocks, din, partial, out);
}

}  // namespace wkv
