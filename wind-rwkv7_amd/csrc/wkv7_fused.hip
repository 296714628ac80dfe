// WKV7 for gfx950: chunk preparation and the sequential state scan in ONE kernel, handing the per-chunk operands
// from producer wavefronts to the chain wavefronts through LDS instead of through memory.
//
// Replaces forward_kernel / the first half of backward_kernel of the reference (attn.cu:11-106, 131-326;
// mathematics rwkv7_attn_triton.py:27-69, 72-156).  The reference runs one block of four warps per (batch, head),
// every warp taking part in every product of a chunk (~60 block barriers per chunk).  Here a block per (batch, head)
// has two kinds of wavefronts:
//   * FUSE_P producer wavefronts.  Each takes every FUSE_P-th chunk and does ALL the state-independent algebra of it
//     alone (decays, the 16x16 products, the triangular inverse, U0 = Tinv AK V, Wm = Tinv wa, transposes), reading
//     the caller's tensors and writing the chunk's operands into a slot of an LDS ring.
//   * four chain wavefronts, each owning 16 value rows of the 64x64 fp32 state in its accumulators.  Per chunk:
//         U^T = U0^T + S Wm^T ;   S <- (S + V^T kwi + U^T bwi) diag(fw) ;   forward also Y = QK V + QB U + wq S^T
//     (kwi = k / P_t, bwi = b / P_t, fw = P_K the chunk's whole decay: S diag(fw) + V^T kf + U^T bf with the
//     decay applied once to the sum)
//     They read their operands from the ring and leave the checkpoint (the state entering the chunk, bf16), U^T and
//     y in a second LDS ring; they touch memory neither way.
//   * one store wavefront that copies what the chain left two steps ago to memory.  A store issued behind a
//     producer's eleven tile loads waits in the compute unit's memory pipeline until they are through, and on a chain
//     wavefront that wait is on the critical path of the step (measured at B=8, H=12 with the chain's stores taken out:
//     T=4096 forward 194 -> 144 us; with inputs that the last-level cache does not hold, T=1024 56 -> 46 us); the
//     store wavefront has the whole step to get its handful of stores accepted.
// All wavefronts run in lock step, one block barrier per chunk: a producer's work on a chunk is cut into FUSE_P
// segments with a barrier after each, producer p starts p steps late, so exactly one chunk is completed per step and
// the chain consumes it two steps later.  No flags, no polling: every wavefront executes the same number of barriers.
// Nothing of the operands (13.25 KiB per chunk forward, 10.25 KiB backward) touches memory.
//
// The backward direction runs the same chain in reverse over dS with its own producers:
//   producers:  D0 = Tinv^T (QB^T dY),  Bm = Tinv^T bf        chain:  dab_u = D0 + Bm dS^T ;
//                                                                     dS' = dS diag(fw) + dY^T wq + dab_u^T wa
// and leaves the dstate arriving at each chunk's end plus dab_u^T for bwd_grads_kernel.
#include "device_info.hpp"
#include "ln_epilogue.hpp"
#include "row_lines.hpp"
#include "wkv7_common.hpp"
#include "wkv7_kernels.hpp"

#include <type_traits>

namespace wkv {

// A producer's work on a chunk has twelve possible cut points (see the SEG() marks in the kernel); bit k of CUTS says
// whether mark k carries a step barrier.  Their number is the number of producer wavefronts: a chunk takes a producer
// that many steps, and one chunk must be completed per step.  Twelve producers (0xfff), one segment each, are not the
// fastest: a block's wavefronts go to the four SIMDs round robin, and what counts is how many share a SIMD with a
// chain wavefront, whose round is the critical path of a step.
// Ten, for two blocks per head (2 chain wavefronts; 14 wavefronts would put a chain wavefront and three producers on
// two of the SIMDs): the triangular products with the start of the inverse, U0 with Wm.  Measured at B=8, T=1024, H=12
// against twelve: forward 49.4 -> 48.0 us, reverse scan 44.4 -> 42.8 us; nine and eight are no better than ten.
constexpr int CUTS_TEN = 0xeef;
// Eight, for one block per head (a chain wavefront and two producers per SIMD; with attn_ln's epilogue wavefronts
// there is room for no more anyway): the decay blocks one each, products + start of the inverse, the rest of the
// inverse, U0 + Wm + first stores, second stores.  Measured against twelve at H=12, T=1024: B=16 254 -> 251 us per
// step, B=64 851 -> 840 us; attn_ln at B=64 against eight cut as "decay blocks in pairs, the inverse in two parts"
// (0xeda): 1260 -> 1252 us.
constexpr int CUTS_EIGHT_EVEN = 0xcaf;
constexpr int fused_producers(int cuts) { return __builtin_popcount(cuts); }
// attn_ln adds three wavefronts that take turns applying the epilogue (GroupNorm, bonus, gate) to the chunk the chain
// finished a step ago: one step of work, two idle steps in which the tiles of the wavefront's next chunk arrive
// (measured: one such wavefront, with a step between request and use, 122 us at B8 T1024 H12 against 86 us; the work
// cut in two steps over four wavefronts 109 us - the statistics held across the barrier spill)
constexpr int LN_WAVES = 3;
// PREPARE: no ring and no chain; a block of one producer wavefront leaves one chunk's operands in memory, for
// wkv7_records_scan_kernel.
// VS: blocks per (batch, head), each owning 4 / VS of the four value blocks (16 value rows each) of the state
// (MAP: two sets of chain wavefronts and nothing to store)
constexpr int fused_threads(int cuts, bool ln, int vs = 1, bool map = false, bool prepare = false) {
    if (prepare) return 64;
    return ((map ? 2 : 1) * (4 / vs) + fused_producers(cuts) + (ln ? LN_WAVES : 0) + (map ? 0 : 1)) * 64;
}
constexpr int FUSE_SLOTS = 4;                   // ring slots; a producer stores in its last two segments only
// slot layout (bytes): six fragment pairs of the chain, the chunk decay, the four private (U0^T, V^T) pairs, and
// forward only the three pairs of the output (wq as two pairs, then (QK, QB))
constexpr int SL_J = 0, SL_FW = 6 * 1024, SL_I = SL_FW + 256, SL_Y = SL_I + 4 * 1024;
constexpr int SLOT_FWD = SL_Y + 3 * 1024, SLOT_BWD = SL_Y;
// The chain's results on their way to memory: per chain wavefront the kept state (2 KiB), U^T (512 B), y (512 B) and
// the output's centres (64 B), each laid out as its place in memory so that the store wavefront copies 16 bytes per
// lane.  Chunk st sits in slot st % OUT_SLOTS; the store wavefront takes it two steps after the chain's round, which
// is when the chain's LDS writes are known to have landed without the chain ever waiting for them (its next round
// waits for operands it requested after them, and a wavefront's LDS accesses complete in order).
constexpr int OUT_SLOTS = 4;
constexpr int out_ck(int) { return 0; }
constexpr int out_ut(int nch) { return nch * 2048; }
constexpr int out_y(int nch) { return out_ut(nch) + nch * 512; }
constexpr int out_cen(int nch) { return out_y(nch) + nch * 512; }
constexpr int out_slot(int nch) { return out_cen(nch) + nch * 64; }

struct FusedArgs {
    int T, H, NC, BH;
    int s_in_f32, s_out_f32;
    const __bf16 *w, *q, *k, *v, *a, *b, *dy;   // forward: w q k v a b; backward: w q a b dy
    __bf16* saved;                              // forward: per chunk checkpoint + U^T (Saved); backward: SavedPair
    const void* s_in;
    void* s_out;
    __bf16* y;                                  // forward only
    // attn_ln forward: gate, parameters [3][H*64] and where the plain WKV7 output is kept for the backward pass
    const __bf16* g;
    const float* params;
    __bf16* y_wkv;
    // attn_ln: where the per-block centres of the kept WKV7 output go (see Centred in ln_epilogue.hpp).  Also set for the
    // plain forward when its y is that kept output (the epilogue then runs as a kernel of its own): y is written centred.
    float* centers;
    int paired;                                 // a state per pair of chunks (SavedPair) or per chunk (Saved)
    // attn_ln backward, optional: the last 3 H blocks of the grid reduce the parameter-gradient partials that the
    // backward epilogue left (dparams_reduce_block) on compute units the scan does not fill
    const float* dparams_part;
    float* dparams;
    int B;
    int ds_run;                                 // backward, paired: see SavedPair::ds_kept
    // Long sequences on few heads: a (batch, head)'s NC chunks as PER + 1 segments, PER of them at a time, a block each.
    // The state entering segment 0 is known, and nobody needs the map of the last one.  So a first pass (PASS = 1) runs segment 0
    // as the kernel proper does and leaves the affine map (S_out = S_in M + N) of segments 1 .. PER - 1 in `maps`,
    // segment_carry_kernel composes them from the state that segment 0 left in entry 0 of s_seg into those entering the
    // segments after it, and the second pass (PASS = 2) starts segments 1 .. PER from their entries.
    // PASS = 0, PER = 1: the whole sequence in one block.
    int PER, L0;                                // L0: chunks of segment 0 (the rest is divided evenly)
    float* maps;                                // first pass: [B*H*PER][2][64][64], N in fragment order and M transposed
    unsigned char* records;                     // PREPARE and wkv7_records_scan_kernel: [B*H][NC] ring slots in processing order
};

#define STEP_BARRIER() step_barrier()
#define SEG(k) do { if constexpr (!PREPARE && ((CUTS >> (k)) & 1)) STEP_BARRIER(); } while (0)
// (the scheduling barriers keep each segment's arithmetic inside its step: the compiler would otherwise move it
// freely across the barrier, which only orders LDS traffic, and unbalance the steps)
__device__ __forceinline__ void step_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);
}

// The barrier of a wavefront that only READS the ring: it has nothing to publish, so it does not wait for its own
// outstanding LDS reads (the operands of its next round); they arrive during the barrier and the round's first
// instructions, and each is waited for where it is used.  (A fence would make the compiler wait for all of them
// here; the memory clobber keeps every access on its side of the barrier.)
__device__ __forceinline__ void reader_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void lds_pair(unsigned char* p, int lane, bf16x4 u, bf16x4 v) {
    *reinterpret_cast<bf16x8*>(p + lane * 16) = __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7);
}

constexpr int fused_ring(bool fwd, bool ln) { return FUSE_SLOTS * (fwd ? SLOT_FWD : SLOT_BWD) + (ln ? 2 * 4096 : 0); }
constexpr int fused_lds(bool fwd, bool ln, int vs) { return fused_ring(fwd, ln) + OUT_SLOTS * out_slot(4 / vs); }

template <bool FWD, bool SAVE, bool LN, int CUTS, int VS, bool MAP, bool PREPARE, int PASS>
__device__ __forceinline__ void fused_block(const FusedArgs& A, unsigned char* const ring) {
    static_assert(!PREPARE || (!SAVE && !LN && !MAP && VS == 1 && CUTS == 0xc00), "one wavefront, no steps to cut the work into");
    static_assert(!MAP || (!SAVE && !LN && PASS == 1), "the map form keeps and writes nothing but the maps");
    static_assert(PASS == 0 || (!LN && !PREPARE), "the one-kernel attn_ln form is for many heads");
    static_assert((CUTS >> 10 & 3) == 3, "the two storing segments are separate steps (ring slots are sized for that)");
    static_assert(!LN || FWD, "the epilogue belongs to the forward direction");
    static_assert(VS == 1 || (VS == 2 && !LN), "the epilogue needs the whole head in one block");
    constexpr int NCH = 4 / VS;                 // value blocks of this block = chain wavefronts of a set
    constexpr int NCW = (MAP ? 2 : 1) * NCH;    // chain wavefronts: MAP runs a second set on the homogeneous recurrence
    constexpr int SLOT = FWD ? SLOT_FWD : SLOT_BWD;
    constexpr int P = fused_producers(CUTS);
    constexpr int YRING = FUSE_SLOTS * SLOT;    // attn_ln: two slots of 4 KiB, the chain's fp32 output of one chunk each
    constexpr int ORING = fused_ring(FWD, LN), OSLOT = out_slot(NCH);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Two blocks per head: blocks i and i + 8 are the two halves of one head, so that (blocks going to the eight XCDs
    // round robin) both read the head's key-side tensors through the same L2; ids past the last head do nothing.
    if constexpr (!FWD) {
        const int extra = A.dparams != nullptr ? 3 * A.H : 0, scan_blocks = (int)gridDim.x - extra;
        if ((int)blockIdx.x >= scan_blocks) {   // (the whole block, before any step barrier)
            const int e = (int)blockIdx.x - scan_blocks;
            dparams_reduce_block(A.B, A.H, A.NC, A.dparams_part, A.dparams, e % A.H, e / A.H, reinterpret_cast<float*>(ring),
                                 (int)blockDim.x / 16);
            return;
        }
    }
    // PREPARE: block ids in turn over the (batch, head)s rounded up to eight, so that a record is written on the XCD that reads it
    const int heads8 = (A.BH + 7) & ~7;
    const int unit = PREPARE ? (int)blockIdx.x % heads8 : VS == 1 ? (int)blockIdx.x : 8 * (int)(blockIdx.x >> 4) + (int)(blockIdx.x & 7);   // (batch, head, segment)
    const int vb0 = VS == 1 ? 0 : (int)((blockIdx.x >> 3) & 1) * NCH;    // first value block of this block
    if ((VS == 2 || PREPARE) && unit >= A.BH * A.PER) return;   // (the whole block, before any barrier)
    const int NC = A.NC;            // chunks of the sequence: what the kept arrays are indexed with
    int bh = unit, seg = 0, first = 0, LS = NC;   // this block walks LS chunks from `first` on
    if constexpr (PASS != 0) {
        auto segment_start = [&](int k) { return k == 0 ? 0 : A.L0 + (k - 1) * (NC - A.L0) / A.PER; };
        bh = unit / A.PER;
        seg = unit - bh * A.PER + (PASS == 2 ? 1 : 0);
        first = segment_start(seg);
        LS = segment_start(seg + 1) - first;
    }
    const int STEPS = LS + P + 2;   // barriers every wavefront executes
    const Lane L;
    // processing order: forward walks the chunks up, backward down; segments are numbered in that order too
    auto chunk_of = [&](int st) -> int { return FWD ? first + st : NC - 1 - (first + st); };
    if constexpr (PASS == 1 && !MAP) {   // (the launch has the map form's wavefronts)
        if (wave >= fused_threads(CUTS, LN, VS, MAP, PREPARE) / 64) {
            for (int k = 0; k < STEPS; k++) STEP_BARRIER();
            return;
        }
    }

    // Buffer loads: a tile is addressed as (descriptor of the tensor's rows of this (batch, head), wave-uniform chunk
    // offset, one 32-bit byte offset per lane that never changes), so no 64-bit address lives in vector registers;
    // reads past the head's last row would return zero instead of faulting.
    const int voff = (L.n * A.H * HEAD + 8 * L.g) * 2;
    const long head0 = ((long)(bh / A.H) * A.T * A.H + (bh % A.H)) * HEAD;                // elements
    const unsigned extent = (unsigned)((((long)A.T - 1) * A.H * HEAD + HEAD) * 2);      // bytes from head0
    // (a descriptor of zero extent for the fetch after a producer's last chunk: same instructions, no memory access)
    auto rsrc = [&](const __bf16* base, unsigned bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(base + head0), 0, bytes, 0x00020000);
    };
    using Rsrc = decltype(rsrc(A.w, 0u));
    auto tile = [&](Rsrc r, int soff) {
        TileB t;
#pragma unroll
        for (int pr = 0; pr < NBLK / 2; pr++) {
            const bf16x8 v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 64 * pr, soff, 0));
            t.f[2 * pr] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
            t.f[2 * pr + 1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
        }
        return t;
    };

    // the value-side tile (v, backward dY): this block's NCH value blocks only, as blocks 0 .. NCH-1
    auto tile_v = [&](Rsrc r, int soff) {
        TileB t;
#pragma unroll
        for (int pr = 0; pr < NCH / 2; pr++) {
            const bf16x8 v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 64 * (vb0 / 2 + pr), soff, 0));
            t.f[2 * pr] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
            t.f[2 * pr + 1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
        }
        return t;
    };

    if constexpr (LN) {
        if (wave >= NCW + P && wave < NCW + P + LN_WAVES) {
            // ------------------------------------------------------------------------------------------------
            // epilogue wavefront e (attn_ln, attn_ln.cu:11-37): chunks e, e + 3, ...; chunk st in step st + P + 2, one
            // step after the chain left its fp32 output in the y ring (the statistics are taken on the fp32 values).
            // The tiles of its next chunk are requested when a chunk is done and have two idle steps to arrive.
            // ------------------------------------------------------------------------------------------------
            const int e = wave - (NCW + P);
            struct Ep {
                TileB q, k, v, g;
            };
            auto fetch_ep = [&](int st) {
                const unsigned bytes = st < LS ? extent : 0u;
                const int soff = st < LS ? chunk_of(st) * (CHUNK * HEAD * 2) * A.H : 0;
                Ep t;
                t.q = tile(rsrc(A.q, bytes), soff);
                t.k = tile(rsrc(A.k, bytes), soff);
                t.v = tile(rsrc(A.v, bytes), soff);
                t.g = tile(rsrc(A.g, bytes), soff);
                return t;
            };
            const LnParams prm = load_ln_params(A.params, bh % A.H, A.H, L);
            const long ld = (long)A.H * HEAD;
            Ep cur = fetch_ep(e);
            int done = 0;
            for (; done < P + 2 + e && done < STEPS; done++) STEP_BARRIER();
            for (int st = e; st < LS; st += LN_WAVES) {
                const unsigned char* ys = ring + YRING + (st & 1) * 4096;
                TileF yf;
#pragma unroll
                for (int i = 0; i < NBLK; i++) yf.f[i] = *reinterpret_cast<const f32x4*>(ys + i * 1024 + lane * 16);
                const long row0 = head0 + (long)chunk_of(st) * CHUNK * ld;
                if constexpr (SAVE) {
                    Centred kept;
                    store_rows16(A.y + row0, ld, L, ln_forward(yf, cur.q, cur.k, cur.v, cur.g, prm, &kept));
                    store_rows16(A.y_wkv + row0, ld, L, kept.y);
                    if (L.g == 0) *reinterpret_cast<f32x4*>(A.centers + 4 * (((long)(bh / A.H) * A.T + chunk_of(st) * CHUNK + L.n) * A.H + bh % A.H)) = kept.c;
                } else {
                    store_rows16(A.y + row0, ld, L, ln_forward(yf, cur.q, cur.k, cur.v, cur.g, prm));
                }
                cur = fetch_ep(st + LN_WAVES);
#pragma unroll
                for (int i = 0; i < LN_WAVES; i++) {
                    if (done < STEPS) {
                        STEP_BARRIER();
                        done++;
                    }
                }
            }
            for (; done < STEPS; done++) STEP_BARRIER();
            return;
        }
    }
    if (PREPARE || (wave >= NCW && wave < NCW + P)) {
        // ------------------------------------------------------------------------------------------------
        // producer p: chunks p, p + P, ... in processing order; segment k of chunk st runs in step st + k
        // ------------------------------------------------------------------------------------------------
        const int p = PREPARE ? (int)blockIdx.x / heads8 : wave - NCW;
        struct In {
            TileB w, q, k, v, a, b;   // backward: v holds dy, k unused
        };
        auto fetch = [&](int st) {
            const unsigned bytes = st < LS ? extent : 0u;
            const int soff = st < LS ? chunk_of(st) * (CHUNK * HEAD * 2) * A.H : 0;
            In t;
            t.w = tile(rsrc(A.w, bytes), soff);
            t.q = tile(rsrc(A.q, bytes), soff);
            t.a = tile(rsrc(A.a, bytes), soff);
            t.b = tile(rsrc(A.b, bytes), soff);
            t.v = tile_v(rsrc(FWD ? A.v : A.dy, bytes), soff);
            if constexpr (FWD) t.k = tile(rsrc(A.k, bytes), soff);
            else t.k = t.v;
            return t;
        };
        In nxt = fetch(p);
        int done = 0;
        if constexpr (!PREPARE)
            for (; done < p; done++) STEP_BARRIER();
        for (int st = p; st < LS; st += P) {
            unsigned char* const slot = PREPARE ? A.records + ((long)unit * NC + st) * SLOT : ring + (st % FUSE_SLOTS) * SLOT;
            auto hand_on = [&](unsigned char* to, int l, bf16x4 u, bf16x4 v) {   // (records through the L2: 2 x 992 tokens x 12 heads 10.4 -> 9.2 us)
                if constexpr (PREPARE) store_through_at(to, 16 * l, join(u, v));
                else lds_pair(to, l, u, v);
            };
            const In cur = nxt;
            const bf16x4 eye = identity_bf16(L);
            // ---- segments 0, 1: decay factors and the scaled operands, two blocks of 16 key channels each ----
            // (see chunk_decay in wkv7_common.hpp for the factors; kept per block here so that only the bf16 operands
            // live on across the step barriers)
            TileB wq, wa, bwi, bf, kwi;   // (bf backward only, kwi forward only)
            float fw1 = 0.f;   // the chunk decay is the same in all 16 token lanes: lane n keeps entry n of its group's 16
#pragma unroll
            for (int i = 0; i < NBLK; i++) {
                constexpr float LOG2E = 1.4426950408889634f, LOG2_LOG2E = 0.5287663729448977f;
                const f32x4 wf = to_f32(cur.w.f[i]);
                const f32x4 qf = to_f32(cur.q.f[i]), af = to_f32(cur.a.f[i]), bfl = to_f32(cur.b.f[i]);
                f32x4 kfl;
                if constexpr (FWD) kfl = to_f32(cur.k.f[i]);
                float wq_[4], wa_[4], bwi_[4], bf_[4], kwi_[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // exp(w) log2(e) as one exponential: 2^(w log2(e) + log2(log2(e))); the prefix sum is then the base-2 log decay
                    const float lc2 = row_prefix_sum(-__builtin_amdgcn_exp2f(fmaf(wf[r], LOG2E, LOG2_LOG2E)));
                    const float P = __builtin_amdgcn_exp2f(lc2);        // decay from the chunk start through token n
                    const float Pi = __builtin_amdgcn_exp2f(-lc2);
                    const float Px = __builtin_bit_cast(                // ... up to but excluding token n
                        float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, P), 0x111, 0xf, 0xf, false));
                    const float fw = row_bcast_last(P);                  // the whole chunk's decay
                    fw1 = (L.n == 4 * i + r) ? fw : fw1;
                    wq_[r] = qf[r] * P;                                 // q * P_t
                    wa_[r] = af[r] * Px;                                // a * P_{t-1}
                    bwi_[r] = bfl[r] * Pi;                              // b / P_t
                    if constexpr (FWD) kwi_[r] = kfl[r] * Pi;
                    else bf_[r] = bwi_[r] * fw;                         // b * P_K / P_t
                }
                wq.f[i] = pack_bf16(wq_[0], wq_[1], wq_[2], wq_[3]);
                wa.f[i] = pack_bf16(wa_[0], wa_[1], wa_[2], wa_[3]);
                bwi.f[i] = pack_bf16(bwi_[0], bwi_[1], bwi_[2], bwi_[3]);
                if constexpr (FWD) kwi.f[i] = pack_bf16(kwi_[0], kwi_[1], kwi_[2], kwi_[3]);
                else bf.f[i] = pack_bf16(bf_[0], bf_[1], bf_[2], bf_[3]);
                if ((CUTS >> i) & 1) STEP_BARRIER();   // cut points 0-3 (the loop is unrolled)
            }
            // ---- segment 2: transposes of V (dY) and the strictly triangular 16x16 products ----
            TileB XT;   // forward: V^T; backward: dY^T   (lane = value ch, reg = token)
#pragma unroll
            for (int ib = 0; ib < NCH; ib++) XT.f[ib] = transpose(cur.v.f[ib], eye);
            const f32x4 AB = mask_lower_strict(tile_xyT(wa, bwi), L);   // [t][s] = wa_t . bwi_s, s < t
            const f32x4 ABT = mask_upper_strict(tile_xyT(bwi, wa), L);
            bf16x4 AK_b, QBT;
            if constexpr (FWD) AK_b = to_bf16(mask_lower_strict(tile_xyT(wa, kwi), L));
            else QBT = to_bf16(mask_upper_incl(tile_xyT(bwi, wq), L));  // [s][t] = wq_t . bwi_s, s <= t
            SEG(4);
            // ---- segments 3, 4: the triangular inverse (matrix instructions in one long dependent chain); the
            //      output's inclusive products ride in the second one ----
            f32x4 Tinv, TinvT;
            tri_inverse_begin(AB, ABT, L, Tinv, TinvT);
            tri_inverse_level<2>(AB, L, Tinv, TinvT);
            SEG(5);
            tri_inverse_level<4>(AB, L, Tinv, TinvT);
            SEG(6);
            tri_inverse_level<8>(AB, L, Tinv, TinvT);
            const bf16x4 Tm = to_bf16(FWD ? Tinv : TinvT);
            bf16x4 QKB0, QKB1;
            if constexpr (FWD && !MAP) {
                QKB0 = to_bf16(mask_lower_incl(tile_xyT(wq, kwi), L));  // QK[t][s] = wq_t . kwi_s, s <= t
                QKB1 = to_bf16(mask_lower_incl(tile_xyT(wq, bwi), L));  // QB
            }
            SEG(7);
            // ---- segment 5: the private operands (forward U0 = Tinv AK V; backward D0 = Tinv^T QB^T dY) and
            //      forward Wm = Tinv wa, backward Bm = Tinv^T bf ----
            TileB ZT;
#pragma unroll
            for (int ib = 0; ib < NCH; ib++) {
                const f32x4 RT = mma(zero4(), FWD ? AK_b : QBT, XT.f[ib]);
                ZT.f[ib] = to_bf16(mma(zero4(), Tm, to_bf16(RT)));
            }
            SEG(8);
            bf16x4 Mm[NBLK];
#pragma unroll
            for (int jb = 0; jb < NBLK; jb++) {
                const bf16x4 xT = transpose(FWD ? wa.f[jb] : bf.f[jb], eye);   // lane = key ch, reg = token
                Mm[jb] = to_bf16(mma(zero4(), xT, Tm));                        // lane = token, reg = key ch
            }
            SEG(9);
            // ---- segment 6: first half of the stores; the next chunk's tiles set out (not earlier: a fetch issued
            //      in segments 2-5 measured 0.4 us slower per step) ----
#pragma unroll
            for (int ib = 0; ib < NCH; ib++) hand_on(slot + SL_I + ib * 1024, lane, ZT.f[ib], XT.f[ib]);
            if constexpr (FWD && !MAP) {
                hand_on(slot + SL_Y, lane, wq.f[0], wq.f[1]);
                hand_on(slot + SL_Y + 1024, lane, wq.f[2], wq.f[3]);
                hand_on(slot + SL_Y + 2048, lane, QKB0, QKB1);
            }
            *reinterpret_cast<float*>(slot + SL_FW + (16 * (L.n >> 2) + 4 * L.g + (L.n & 3)) * 4) = fw1;
            if constexpr (!PREPARE) nxt = fetch(st + P);
            SEG(10);
            // ---- segment 7: the shared operands of the chain ----
#pragma unroll
            for (int jb = 0; jb < NBLK; jb++) {
                if constexpr (FWD)
                    hand_on(slot + SL_J + (2 + jb) * 1024, lane, transpose(kwi.f[jb], eye), transpose(bwi.f[jb], eye));
                else
                    hand_on(slot + SL_J + (2 + jb) * 1024, lane, transpose(wq.f[jb], eye), transpose(wa.f[jb], eye));
            }
            hand_on(slot + SL_J, lane, Mm[0], Mm[1]);
            hand_on(slot + SL_J + 1024, lane, Mm[2], Mm[3]);
            SEG(11);
            if constexpr (PREPARE) return;
            done += P;
        }
        for (; done < STEPS; done++) STEP_BARRIER();
        return;
    }

    if constexpr (PREPARE) return;
    if (!MAP && wave == NCW + P + (LN ? LN_WAVES : 0)) {
        // ------------------------------------------------------------------------------------------------
        // store wavefront: after its barrier number P + 3 + st the results of chunk st are in their out slot
        // ------------------------------------------------------------------------------------------------
        unsigned char* const saved = reinterpret_cast<unsigned char*>(A.saved);
        const long row_ld = (long)A.H * HEAD;
        const long y_head = (long)(bh / A.H) * A.T * row_ld + (long)(bh % A.H) * HEAD;   // elements
        for (int k = 1; k <= STEPS; k++) {
            STEP_BARRIER();
            const int st = k - (P + 3);
            if (st < 0 || st >= LS) continue;
            const int c = chunk_of(st);
            const unsigned char* o = ring + ORING + (st % OUT_SLOTS) * OSLOT;
            auto piece = [&](int off) { return *reinterpret_cast<const bf16x8*>(o + off + lane * 16); };
            if constexpr (SAVE) {
                long ck, ut;   // byte offsets of this block's part of the kept state and of U^T
                bool keep;
                if (A.paired) {
                    const long pid = (long)bh * SavedPair::pairs(NC) + (c >> 1);
                    ck = SavedPair::ds(pid, vb0) * 2, ut = (SavedPair::ut(pid, c) + vb0 * FRAG_ELEMS) * 2;
                    keep = FWD ? !(c & 1) : SavedPair::keeps(c, NC) && SavedPair::ds_kept(pid, c >> 1, SavedPair::pairs(NC), A.ds_run);
                } else {
                    const long cid = (long)bh * NC + c;
                    ck = Saved::ckpt(cid, vb0) * 2, ut = (Saved::ut(cid) + vb0 * FRAG_ELEMS) * 2;
                    keep = true;
                }
                if (keep) {
#pragma unroll
                    for (int i = 0; i < 2 * NCH; i++) store_streamed(saved + ck + i * 1024 + lane * 16, piece(out_ck(NCH) + i * 1024));
                }
                if constexpr (NCH == 4) {
#pragma unroll
                    for (int i = 0; i < 2; i++) store_streamed(saved + ut + i * 1024 + lane * 16, piece(out_ut(NCH) + i * 1024));
                } else {
                    store_streamed(saved + ut + lane * 16, piece(out_ut(NCH)));
                }
            }
            if constexpr (FWD && !LN) {
                // y by rows: a lane's 16 bytes are the fragments of value blocks 2p and 2p + 1 (8 contiguous channels)
                if constexpr (NCH == 4) {   // whole lines: eight lanes a row
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int row = 8 * i + (lane >> 3), pc = lane & 7;
                        store_streamed(A.y + y_head + (long)(c * CHUNK + row) * row_ld + 8 * pc,
                                       *reinterpret_cast<const bf16x8*>(o + out_y(NCH) + (pc >> 2) * 1024 + (16 * (pc & 3) + row) * 16));
                    }
                } else {
                    store_streamed(A.y + y_head + (long)(c * CHUNK + L.n) * row_ld + 32 * (vb0 / 2) + 8 * L.g, piece(out_y(NCH)));
                }
                if (A.centers != nullptr && lane < 16) {   // token `lane`: the centres of this block's value blocks
                    float* dst = A.centers + 4 * (((long)(bh / A.H) * A.T + c * CHUNK + lane) * A.H + bh % A.H) + vb0;
                    const float* src = reinterpret_cast<const float*>(o + out_cen(NCH)) + lane * NCH;
                    if constexpr (NCH == 4) *reinterpret_cast<f32x4*>(dst) = *reinterpret_cast<const f32x4*>(src);
                    else *reinterpret_cast<float2*>(dst) = *reinterpret_cast<const float2*>(src);
                }
            }
        }
        return;
    }
    // ----------------------------------------------------------------------------------------------------
    // chain wavefront ib: value rows 16 ib .. 16 ib + 15 of the state
    // ----------------------------------------------------------------------------------------------------
    // MAP: set 0 runs the recurrence from a zero state (-> N), set 1 the homogeneous recurrence (no V, no U0; backward
    // no dY, no D0) from the identity (-> M); both take the shared operands from the one ring
    const int part = MAP ? wave / NCH : 0;
    const int iw = MAP ? wave % NCH : wave;   // value block within this block (its slot in the ring)
    const int ib = vb0 + iw;                  // value block within the head
    // the chain is the critical path of every step: its wavefronts win the SIMD's issue arbitration against the two
    // producers they share it with, which fill the gaps
    __builtin_amdgcn_s_setprio(3);
    struct Operands {   // read from the ring one step ahead of their use
        bf16x8 j[6];
        bf16x8 iv;
    };
    auto read_ops = [&](Operands& o, int st) {
        const unsigned char* base = ring + (st % FUSE_SLOTS) * SLOT;
#pragma unroll
        for (int i = 0; i < 6; i++) o.j[i] = *reinterpret_cast<const bf16x8*>(base + SL_J + i * 1024 + lane * 16);
        o.iv = *reinterpret_cast<const bf16x8*>(base + SL_I + iw * 1024 + lane * 16);
    };
    // Off the chain: the chunk decay and, forward, the output's operands.  Their producer stored them two steps before
    // the round that uses them, so they too are requested at the end of the round before (into the registers that round
    // has just finished with) and no round starts by waiting for LDS.
    struct Early {
        f32x4 fw[NBLK];
        bf16x8 yp[3];
    };
    auto read_early = [&](Early& e, int st) {
        const unsigned char* base = ring + (st % FUSE_SLOTS) * SLOT;
#pragma unroll
        for (int jb = 0; jb < NBLK; jb++) e.fw[jb] = *reinterpret_cast<const f32x4*>(base + SL_FW + jb * 64 + L.g * 16);
        if constexpr (FWD && !MAP) {
#pragma unroll
            for (int i = 0; i < 3; i++) e.yp[i] = *reinterpret_cast<const bf16x8*>(base + SL_Y + i * 1024 + lane * 16);
        }
    };
    f32x4 S[NBLK];
#pragma unroll
    for (int jb = 0; jb < NBLK; jb++) {
        if constexpr (MAP) {   // zero, or the rows 16 ib .. + 15 of the identity (fragment order on both sides, as the maps are kept)
#pragma unroll
            for (int r = 0; r < 4; r++) S[jb][r] = (part == 1 && 16 * ib + L.n == 16 * jb + 4 * L.g + r) ? 1.f : 0.f;
        } else {
            S[jb] = load_state_frag(A.s_in, A.s_in_f32, PASS == 2 ? unit : bh, ib, jb, L);
        }
    }

    Early early;
    auto round = [&](int st, const Operands& op, Operands& next) {
        const int c = chunk_of(st);
        const f32x4(&fw)[NBLK] = early.fw;
        const bf16x8(&yp)[3] = early.yp;
        const bf16x4 b0 = to_bf16(S[0]), b1 = to_bf16(S[1]), b2 = to_bf16(S[2]), b3 = to_bf16(S[3]);
        const bf16x8 s01 = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
        const bf16x8 s23 = __builtin_shufflevector(b2, b3, 0, 1, 2, 3, 4, 5, 6, 7);
        bf16x8 iv = op.iv;
        if constexpr (MAP) {
            const bf16x8 none = {};
            if (part) iv = none;
        }
        const bf16x4 U0 = __builtin_shufflevector(iv, iv, 0, 1, 2, 3);
        const f32x4 Ua = mma8(to_f32(U0), op.j[0], s01);   // + F(S_ib Wm^T), two independent halves
        const f32x4 Uc = mma8(zero4(), op.j[1], s23);
        f32x4 y;
        if constexpr (FWD && !MAP) {   // F(Y_ib): lane = token, reg = value channel.  wq S_ib^T does not wait for U
            y = mma8(zero4(), s01, yp[0]);
            y = mma8(y, s23, yp[1]);
        }
        const bf16x4 u = to_bf16(Ua + Uc);
        const bf16x8 VU = __builtin_shufflevector(iv, __builtin_shufflevector(u, u, 0, 1, 2, 3, 0, 1, 2, 3), 4, 5, 6, 7, 8, 9, 10, 11);
#pragma unroll
        for (int jb = 0; jb < NBLK; jb++) {
            // forward: (S + V_ib^T kwi_jb + U_ib^T bwi_jb) diag(fw), the chunk decay applied to the sum (the producers
            // then need no separately scaled copies of k and b); backward: dS diag(fw) + dY_ib^T wq_jb + dab_u_ib^T wa_jb
            if constexpr (FWD) S[jb] = mma8(S[jb], op.j[2 + jb], VU) * fw[jb];
            else S[jb] = mma8(S[jb] * fw[jb], op.j[2 + jb], VU);
        }
        unsigned char* const out = ring + ORING + (st % OUT_SLOTS) * OSLOT;
        if constexpr (SAVE) {
            // forward: the state only where a pair of chunks begins (the gradient kernel advances it across the pair's
            // first chunk); backward: the dstate only where a pair ends (SavedPair); every chunk when a state per chunk is kept
            bool keep = !A.paired || (FWD ? !(c & 1) : SavedPair::keeps(c, NC));
            if constexpr (!FWD) {
                const int NP = SavedPair::pairs(NC);
                if (A.paired) keep = keep && SavedPair::ds_kept((long)bh * NP + (c >> 1), c >> 1, NP, A.ds_run);
            }
            if (keep) {
                bf16x8* q = reinterpret_cast<bf16x8*>(out + out_ck(NCH) + iw * 2048 + lane * 32);
                q[0] = s01;
                q[1] = s23;
            }
            *reinterpret_cast<bf16x4*>(out + out_ut(NCH) + iw * 512 + lane * 8) = u;
        }
        if constexpr (FWD && !MAP) {
            const f32x4 yo = mma8(y, VU, yp[2]);             // + QK V_ib + QB U_ib
            if constexpr (LN) *reinterpret_cast<f32x4*>(ring + YRING + (st & 1) * 4096 + iw * 1024 + lane * 16) = yo;
            else {
                bf16x4* yq = reinterpret_cast<bf16x4*>(out + out_y(NCH) + ((iw >> 1) * 64 + lane) * 16 + (iw & 1) * 8);
                if (A.centers != nullptr) {   // y is attn_ln's kept output: centred per block (all four lanes of a token hold the same centre)
                    const float cen = row_sum16_bf16(yo) * (1.f / 16);
                    *yq = to_bf16(yo - cen);
                    if (L.g == 0) *reinterpret_cast<float*>(out + out_cen(NCH) + (L.n * NCH + iw) * 4) = cen;
                } else *yq = to_bf16(yo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // the next round's operand reads stay behind these writes (see OUT_SLOTS)
        read_ops(next, st + 1);   // complete since the end of the step before this one
        read_early(early, st + 1);
        if constexpr (LN) STEP_BARRIER();   // (publishes the y ring)
        else reader_barrier();
    };

    for (int i = 0; i < P; i++) STEP_BARRIER();
    Operands op0, op1;
    read_ops(op0, 0);
    read_early(early, 0);
    STEP_BARRIER();
    int st = 0;
    for (; st + 2 <= LS; st += 2) {
        round(st, op0, op1);
        round(st + 1, op1, op0);
    }
    if (st < LS) round(st, op0, op1);
    STEP_BARRIER();   // the last round's results are in LDS; the epilogue wavefronts' and the store wavefront's last step
    if constexpr (MAP) {
        float* dst = A.maps + ((long)unit * 2 + part) * HEAD * HEAD;
#pragma unroll
        for (int jb = 0; jb < NBLK; jb++) {
            if (part == 0) {
                *reinterpret_cast<f32x4*>(dst + (16 * ib + L.n) * HEAD + 16 * jb + 4 * L.g) = S[jb];
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) dst[(16 * jb + 4 * L.g + r) * HEAD + 16 * ib + L.n] = S[jb][r];
            }
        }
    } else if (PASS != 2 || seg == A.PER) {   // the first segment in a pass of its own; the one walked last: the sequence's final state
#pragma unroll
        for (int jb = 0; jb < NBLK; jb++) store_state_frag(A.s_out, A.s_out_f32, PASS == 1 ? unit : bh, ib, jb, L, S[jb]);
    }
}

template <bool FWD, bool SAVE, bool LN, int CUTS, int VS = 1, bool PREPARE = false, int PASS = 0>
__global__ __launch_bounds__(fused_threads(CUTS, LN, VS, false, PREPARE)) void wkv7_fused_kernel(const FusedArgs A) {
    __shared__ __attribute__((aligned(16))) unsigned char ring[PREPARE ? 16 : fused_lds(FWD, LN, VS)];
    fused_block<FWD, SAVE, LN, CUTS, VS, false, PREPARE, PASS>(A, ring);
}

// The first pass over segments: the first one of each (batch, head) as above, the maps of the others.  Bound as those forms are: a
// chunk of a map takes the producers 0.8 us, one of the kernel proper as long while the rest of the chip writes nothing.
// Against the maps of PER equal segments and then a scan of those (forward with states kept + backward with the gradient kernel, us):
// 1 x 16384 tokens x 32 heads 723 -> 687, 1 x 8192 x 64 720 -> 655, 4 x 8192 x 12 579 -> 540, 1 x 4096 x 12 154 -> 150.
template <bool FWD, bool SAVE, int CUTS, int VS>
__global__ __launch_bounds__(fused_threads(CUTS, false, VS, true)) void wkv7_first_pass_kernel(const FusedArgs A) {
    static_assert(fused_threads(CUTS, false, VS, true) >= fused_threads(CUTS, false, VS), "the maps take more wavefronts");
    __shared__ __attribute__((aligned(16))) unsigned char ring[fused_lds(FWD, false, VS)];
    const int unit = VS == 1 ? (int)blockIdx.x : 8 * (int)(blockIdx.x >> 4) + (int)(blockIdx.x & 7);
    if (unit % A.PER == 0) fused_block<FWD, SAVE, false, CUTS, VS, false, false, 1>(A, ring);
    else fused_block<FWD, false, false, CUTS, VS, true, false, 1>(A, ring);
}

// ------------------------------------------------------------------------------------------------
// The chain over records in memory: few (batch, head)s, where one block each (or two) would leave most of the chip idle and a
// step of the one-kernel form, 0.556 us, is the time its producers take, ten wavefronts on one compute unit.  There the chunks are
// prepared first, each by a wavefront of its own all over the chip (the PREPARE form above: the ring slot of a chunk, 13.25 KiB forward,
// 10.25 KiB backward, goes to memory), and this kernel walks them with nothing but the chain: 0.21 us a chunk.
// A block per value block (16 rows of the state), so four per (batch, head), of two wavefronts on two SIMDs:
//   * the chain wavefront reads its operands straight into registers, RECORDS_AHEAD records ahead (7.25 KiB each, whole lines; 8 ahead
//     is no faster), multiplies, and leaves the state and U^T of the chunk in LDS.  It waits for nobody but the barrier of a round.
//   * the output wavefront takes them a round later: forward Y, and every store, of which none stands behind the chain's loads.
// What bounds a round is the chain's own dependent instructions: two matrix instructions, a sum, four matrix instructions, the decay.
// Measured, whole call (forward keeping a state per pair / backward with the gradient kernel, us; one kernel -> records), 64-channel
// heads: 2 x 992 tokens x 12 heads 41.7 -> 26.8 / 58.8 -> 44.8, 1 x 256 x 4 17.4 -> 10.5 / 31.8 -> 25.7, 1 x 1024 x 64 44 -> 36 / 79 -> 71.
// The same bits as the one-kernel form: the same instructions on the same operands.  Other forms, forward at 2 x 992 x 12: records through LDS rings
// by loader wavefronts, two value blocks to a block 31.4 (what the wavefronts read from LDS is its time), four 39.8; one wavefront
// doing the output and the stores as well 32.9.
// ------------------------------------------------------------------------------------------------
constexpr int RECORDS_AHEAD = 4;

// x times entry 4 JB + R of the sixteen that a row of sixteen lanes holds
template <int K>
__device__ __forceinline__ float times_row_lane(float x, float held) {
    return x * __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, held), 0x150 + K, 0xf, 0xf, true));
}
template <int JB>
__device__ __forceinline__ f32x4 times_decay(f32x4 x, float held) {
    return (f32x4){times_row_lane<4 * JB>(x[0], held), times_row_lane<4 * JB + 1>(x[1], held), times_row_lane<4 * JB + 2>(x[2], held),
                   times_row_lane<4 * JB + 3>(x[3], held)};
}

// the barrier of a wavefront whose own LDS accesses are done
__device__ __forceinline__ void done_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <bool FWD, bool SAVE, bool CENTRED>
__global__ __launch_bounds__(128) void wkv7_records_scan_kernel(const FusedArgs A) {
    constexpr int RECORD = FWD ? SLOT_FWD : SLOT_BWD, AHEAD = RECORDS_AHEAD;
    constexpr int OUT = 2048 + 512;   // the chain's results of a chunk: the state before it (bf16), U^T
    __shared__ __attribute__((aligned(16))) unsigned char outs[2 * OUT];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (!FWD) {
        const int extra = A.dparams != nullptr ? 3 * A.H : 0, scan_blocks = (int)gridDim.x - extra;
        if ((int)blockIdx.x >= scan_blocks) {   // (the whole block, before any barrier)
            const int e = (int)blockIdx.x - scan_blocks;
            dparams_reduce_block(A.B, A.H, A.NC, A.dparams_part, A.dparams, e % A.H, e / A.H, reinterpret_cast<float*>(outs), (int)blockDim.x / 16);
            return;
        }
    }
    // the four value blocks of a (batch, head) are 8 block ids apart: the same XCD, whose L2 brings a record in once
    const int bh = 8 * (int)(blockIdx.x >> 5) + (int)(blockIdx.x & 7), ib = (int)(blockIdx.x >> 3) & 3;
    if (bh >= A.BH) return;   // (the whole block, before any barrier)
    const int NC = A.NC;      // barriers of either wavefront: the chain's results of round st are in LDS behind barrier st + 1
    const Lane L;
    auto chunk_of = [&](int st) -> int { return FWD ? st : NC - 1 - st; };
    const int NP = SavedPair::pairs(NC);
    auto keeps = [&](int c) {   // forward the state only where a pair of chunks begins, backward the dstate only where one ends and a run starts
        if (!A.paired) return true;
        return FWD ? !(c & 1) : SavedPair::keeps(c, NC) && SavedPair::ds_kept((long)bh * NP + (c >> 1), c >> 1, NP, A.ds_run);
    };
    // Everything in memory by descriptors on this (batch, head)'s part and 32-bit offsets
    auto rsrc = [](const void* base, long bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (unsigned)bytes, 0x00020000); };
    const auto rec = rsrc(A.records + (long)bh * NC * RECORD, (long)NC * RECORD);
    auto record = [&](int st) { return min(st, NC - 1) * RECORD; };   // (behind the last one: that one again)
    auto piece = [&](int st, int off) {
        return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rec, lane * 16, record(st) + off, 0));
    };
    // fetch(i, st): record st into register set i; round(i, st)
    auto walk = [&](auto&& fetch, auto&& round) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            fetch(i, i);
            __builtin_amdgcn_sched_barrier(0);   // (in the loop's order: what is waited for there is counted)
        }
        int st = 0;
        for (; st + AHEAD <= NC; st += AHEAD) {
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                round(i, st + i);
                __builtin_amdgcn_sched_barrier(0);   // (a round's operands are waited for in that round)
                fetch(i, st + i + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            if (st + i < NC) round(i, st + i);
    };

    if (wave == 1) {
        // output wavefront: forward Y = QK V + QB U + wq S^T; the kept state and U^T; all stores
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        // A store that is not to be is one to an offset behind the end: no branch, so the number of accesses behind a load is
        // known where the compiler waits for it.
        constexpr unsigned NOWHERE = 0x40000000;
        const long per_head = A.paired ? (long)NP * SavedPair::BYTES : (long)NC * Saved::BYTES;
        const auto saved = rsrc(reinterpret_cast<unsigned char*>(A.saved) + (SAVE ? bh * per_head : 0), SAVE ? per_head : 0);
        const int row = A.H * HEAD * 2;                                  // bytes
        const long token0 = (long)(bh / A.H) * A.T * A.H + bh % A.H;     // of this (batch, head), in heads
        const auto y_to = rsrc(A.y + (FWD ? token0 * HEAD : 0), FWD ? (long)A.T * row : 0);
        const auto cen_to = rsrc(A.centers + (CENTRED ? token0 * 4 : 0), CENTRED ? (long)A.T * A.H * 16 : 0);
        const unsigned y_lane = L.n * row + (32 * (ib / 2) + 8 * L.g + 4 * (ib % 2)) * 2;
        const unsigned cen_lane = L.g == 0 ? (L.n * A.H * 4 + ib) * 4 : NOWHERE;
        struct {
            bf16x8 iv, yp[3];
        } op[AHEAD];
        walk(
            [&](int i, int st) {
                if constexpr (FWD) {
                    op[i].iv = piece(st, SL_I + ib * 1024);
#pragma unroll
                    for (int k = 0; k < 3; k++) op[i].yp[k] = piece(st, SL_Y + k * 1024);
                }
            },
            [&](int i, int st) {
                done_barrier();
                const int c = chunk_of(st);
                const unsigned char* const o = outs + (st & 1) * OUT;
                const bf16x8 s01 = reinterpret_cast<const bf16x8*>(o + lane * 32)[0], s23 = reinterpret_cast<const bf16x8*>(o + lane * 32)[1];
                const bf16x4 u = *reinterpret_cast<const bf16x4*>(o + 2048 + lane * 8);
                if constexpr (SAVE) {
                    // bytes from this (batch, head)'s first: this value block's part of the kept state and of U^T
                    const unsigned ck = (A.paired ? SavedPair::ds(c >> 1, ib) : Saved::ckpt(c, ib)) * 2;
                    const unsigned ut = ((A.paired ? SavedPair::ut(c >> 1, c) : Saved::ut(c)) + ib * FRAG_ELEMS) * 2;
                    const unsigned to = keeps(c) ? ck + lane * 32 : NOWHERE;
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s01), saved, to, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s23), saved, to + 16, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, u), saved, lane * 8, ut, 0);
                }
                if constexpr (FWD) {
                    const bf16x8 VU = __builtin_shufflevector(op[i].iv, __builtin_shufflevector(u, u, 0, 1, 2, 3, 0, 1, 2, 3), 4, 5, 6, 7, 8, 9, 10, 11);
                    f32x4 y = mma8(zero4(), s01, op[i].yp[0]);   // F(Y_ib): lane = token, reg = value channel
                    y = mma8(y, s23, op[i].yp[1]);
                    y = mma8(y, VU, op[i].yp[2]);
                    if constexpr (CENTRED) {   // (see the fused kernel: attn_ln's kept output, centred per block)
                        const float cen = row_sum16_bf16(y) * (1.f / 16);
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, cen), cen_to, cen_lane, c * CHUNK * A.H * 16, 0);
                        y = y - cen;
                    }
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, to_bf16(y)), y_to, y_lane, c * CHUNK * row, 0);
                }
            });
        return;
    }
    // chain wavefront: value rows 16 ib .. 16 ib + 15 of the state
    __builtin_amdgcn_s_setprio(3);
    f32x4 S[NBLK];
#pragma unroll
    for (int jb = 0; jb < NBLK; jb++) S[jb] = load_state_frag(A.s_in, A.s_in_f32, bh, ib, jb, L);
    struct {
        bf16x8 j[6], iv;
        float fw;
    } ops[AHEAD];
    walk(
        [&](int i, int st) {
            auto& op = ops[i];
#pragma unroll
            for (int k = 0; k < 2; k++) op.j[k] = piece(st, SL_J + k * 1024);
            op.iv = piece(st, SL_I + ib * 1024);
#pragma unroll
            for (int k = 2; k < 6; k++) op.j[k] = piece(st, SL_J + k * 1024);
            op.fw = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rec, (16 * (L.n >> 2) + 4 * L.g + (L.n & 3)) * 4, record(st) + SL_FW, 0));
        },
        [&](int i, int st) {
            const auto& op = ops[i];
            const bf16x4 b0 = to_bf16(S[0]), b1 = to_bf16(S[1]), b2 = to_bf16(S[2]), b3 = to_bf16(S[3]);
            const bf16x8 s01 = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
            const bf16x8 s23 = __builtin_shufflevector(b2, b3, 0, 1, 2, 3, 4, 5, 6, 7);
            const bf16x4 U0 = __builtin_shufflevector(op.iv, op.iv, 0, 1, 2, 3);
            const f32x4 Ua = mma8(to_f32(U0), op.j[0], s01);   // + F(S_ib Wm^T), two independent halves
            const f32x4 Uc = mma8(zero4(), op.j[1], s23);
            unsigned char* const o = outs + (st & 1) * OUT;
            reinterpret_cast<bf16x8*>(o + lane * 32)[0] = s01;
            reinterpret_cast<bf16x8*>(o + lane * 32)[1] = s23;
            auto decay = [&] { S[0] = times_decay<0>(S[0], op.fw), S[1] = times_decay<1>(S[1], op.fw), S[2] = times_decay<2>(S[2], op.fw), S[3] = times_decay<3>(S[3], op.fw); };
            if constexpr (!FWD) decay();
            const bf16x4 u = to_bf16(Ua + Uc);
            const bf16x8 VU = __builtin_shufflevector(op.iv, __builtin_shufflevector(u, u, 0, 1, 2, 3, 0, 1, 2, 3), 4, 5, 6, 7, 8, 9, 10, 11);
            *reinterpret_cast<bf16x4*>(o + 2048 + lane * 8) = u;
#pragma unroll
            for (int jb = 0; jb < NBLK; jb++) S[jb] = mma8(S[jb], op.j[2 + jb], VU);
            if constexpr (FWD) decay();
            done_barrier();
        });
#pragma unroll
    for (int jb = 0; jb < NBLK; jb++) store_state_frag(A.s_out, A.s_out_f32, bh, ib, jb, L, S[jb]);
}

// ------------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------------
namespace {
// grid of a launch over `units` (batch, head, segment)s: one block each, or two (halves 8 block ids apart)
inline unsigned fused_grid(int units, int vs) { return vs == 1 ? units : 16 * ((units + 7) / 8); }
inline bool fused_split(int units) { return 2 * units <= compute_units(); }

FusedArgs fused_args(int B, int T, int H, int state_f32, int per) {
    FusedArgs A{};
    A.T = T, A.H = H, A.NC = T / CHUNK, A.BH = B * H, A.B = B;
    A.s_in_f32 = A.s_out_f32 = state_f32;
    A.PER = per, A.L0 = first_segment_chunks(A.NC, per);
    A.ds_run = 1;
    return A;
}

// Long sequences on few heads (ScanPlan::segments > 1): the first pass, then the states entering the segments of the second.  After
// this A.s_in is the per-segment array and the kernel proper can be launched over the B*H*PER units of the second pass.
template <bool FWD>
void first_pass(FusedArgs& A, bool save, void* seg_ws, hipStream_t stream) {
    const int units = A.BH * A.PER;
    float* maps = static_cast<float*>(seg_ws);
    float* s_seg = maps + (size_t)units * 2 * HEAD * HEAD;
    FusedArgs M = A;
    M.maps = maps, M.s_out = s_seg, M.s_out_f32 = 1;
    M.dparams = nullptr, M.dparams_part = nullptr;
    auto go = [&](auto kernel, int vs, int threads) { hipLaunchKernelGGL(kernel, dim3(fused_grid(units, vs)), dim3(threads), 0, stream, M); };
    if (fused_split(units)) {
        constexpr int THREADS = fused_threads(CUTS_TEN, false, 2, true);
        if (save) go(wkv7_first_pass_kernel<FWD, true, CUTS_TEN, 2>, 2, THREADS);
        else if constexpr (FWD) go(wkv7_first_pass_kernel<FWD, false, CUTS_TEN, 2>, 2, THREADS);
    } else {
        constexpr int THREADS = fused_threads(CUTS_EIGHT_EVEN, false, 1, true);
        if (save) go(wkv7_first_pass_kernel<FWD, true, CUTS_EIGHT_EVEN, 1>, 1, THREADS);
        else if constexpr (FWD) go(wkv7_first_pass_kernel<FWD, false, CUTS_EIGHT_EVEN, 1>, 1, THREADS);
    }
    launch_segment_carry(A.BH, A.PER, maps, s_seg, stream);
    A.s_in = s_seg, A.s_in_f32 = 1;
}

// The chunks' records, then the chain over them.
template <bool FWD>
void by_records(FusedArgs A, bool save, void* ws, unsigned extra, hipStream_t stream) {
    A.records = static_cast<unsigned char*>(ws);
    FusedArgs P = A;
    P.dparams = nullptr, P.dparams_part = nullptr;
    constexpr int CUTS = 0xc00;
    hipLaunchKernelGGL((wkv7_fused_kernel<FWD, false, false, CUTS, 1, true>), dim3((unsigned)((A.BH + 7) & ~7) * A.NC), dim3(64), 0, stream, P);
    const dim3 grid(32 * ((A.BH + 7) / 8) + extra), block(128);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, stream, A); };
    if constexpr (!FWD) go(wkv7_records_scan_kernel<false, true, false>);
    else if (A.centers) save ? go(wkv7_records_scan_kernel<true, true, true>) : go(wkv7_records_scan_kernel<true, false, true>);
    else save ? go(wkv7_records_scan_kernel<true, true, false>) : go(wkv7_records_scan_kernel<true, false, false>);
}
}  // namespace

size_t scan_record_bytes(bool fwd) { return fwd ? SLOT_FWD : SLOT_BWD; }

void launch_fused_forward(int B, int T, int H, int state_f32, const void* w, const void* q, const void* k, const void* v,
                          const void* a, const void* b, const void* s_in, void* s_out, void* y, void* saved,
                          int paired, hipStream_t stream, const void* g, const void* params, void* y_wkv, float* centers,
                          void* ws, size_t ws_bytes) {
    auto c = [](const void* p) { return static_cast<const __bf16*>(p); };
    const ScanPlan plan = params ? ScanPlan{false, 1} : scan_plan(B, T, H, ws_bytes, saved ? SCAN_FORWARD : SCAN_PREFILL);   // (the one-kernel attn_ln forward is for many heads)
    const int nseg = plan.segments;
    FusedArgs A = fused_args(B, T, H, state_f32, nseg);
    A.w = c(w), A.q = c(q), A.k = c(k), A.v = c(v), A.a = c(a), A.b = c(b);
    A.saved = static_cast<__bf16*>(saved), A.s_in = s_in, A.s_out = s_out, A.y = static_cast<__bf16*>(y);
    A.g = c(g), A.params = static_cast<const float*>(params), A.y_wkv = static_cast<__bf16*>(y_wkv), A.centers = centers;
    A.paired = paired;
    if (plan.records) {
        by_records<true>(A, saved != nullptr, ws, 0, stream);
        return;
    }
    if (nseg > 1) first_pass<true>(A, saved != nullptr, ws, stream);
    const int units = B * H * nseg;
    auto go = [&](auto kernel, int threads, int vs = 1) {
        hipLaunchKernelGGL(kernel, dim3(fused_grid(units, vs)), dim3(threads), 0, stream, A);
    };
    // Two blocks per (batch, head), two value blocks each, while every block still gets a compute unit of its own: the
    // chain's and the value-side producers' work is halved per block at the price of repeating the key-side producers.
    const bool split = !params && fused_split(units);
    if (params) {
        constexpr int CUTS = CUTS_EIGHT_EVEN;
        if (saved) go(wkv7_fused_kernel<true, true, true, CUTS>, fused_threads(CUTS, true));
        else go(wkv7_fused_kernel<true, false, true, CUTS>, fused_threads(CUTS, true));
    } else {
        auto pass = [&](auto which) {
            constexpr int PASS = decltype(which)::value;
            if (split) {
                constexpr int CUTS2 = CUTS_TEN;
                if (saved) go(wkv7_fused_kernel<true, true, false, CUTS2, 2, false, PASS>, fused_threads(CUTS2, false, 2), 2);
                else go(wkv7_fused_kernel<true, false, false, CUTS2, 2, false, PASS>, fused_threads(CUTS2, false, 2), 2);
            } else {
                constexpr int CUTS1 = CUTS_EIGHT_EVEN;
                if (saved) go(wkv7_fused_kernel<true, true, false, CUTS1, 1, false, PASS>, fused_threads(CUTS1, false));
                else go(wkv7_fused_kernel<true, false, false, CUTS1, 1, false, PASS>, fused_threads(CUTS1, false));
            }
        };
        if (nseg > 1) pass(std::integral_constant<int, 2>());
        else pass(std::integral_constant<int, 0>());
    }
}

bool fused_backward_scan_takes_dparams(int B, int T, int H, size_t ws_bytes) {
    const ScanPlan plan = scan_plan(B, T, H, ws_bytes, SCAN_BACKWARD);
    // Beside a scan by records there is room everywhere, but its blocks have two wavefronts, and the more sequences a head has the
    // longer theirs take: 32 x 128 tokens x 2 heads 38.0 -> 37.6 us, 64 x 512 tokens x 1 head 75 in the scan, 66 on their own.
    if (plan.records) return B <= 32;
    const int units = B * H * plan.segments;
    const int scan_blocks = (int)fused_grid(units, fused_split(units) ? 2 : 1);
    return scan_blocks + 3 * H <= compute_units();
}

void launch_fused_backward_scan(int B, int T, int H, int state_f32, const void* w, const void* q, const void* a,
                                const void* b, const void* dy, const void* ds_in, void* ds_out, void* saved,
                                int paired, hipStream_t stream, const float* dparams_part, float* dparams, void* ws, size_t ws_bytes) {
    auto c = [](const void* p) { return static_cast<const __bf16*>(p); };
    const ScanPlan plan = scan_plan(B, T, H, ws_bytes, SCAN_BACKWARD);
    const int nseg = plan.segments;
    FusedArgs A = fused_args(B, T, H, state_f32, nseg);
    A.w = c(w), A.q = c(q), A.a = c(a), A.b = c(b), A.dy = c(dy);
    A.saved = static_cast<__bf16*>(saved), A.s_in = ds_in, A.s_out = ds_out;
    A.paired = paired, A.ds_run = paired ? dstate_run(B, T, H) : 1;
    A.dparams_part = dparams_part, A.dparams = dparams;
    const unsigned extra = dparams ? 3 * H : 0;
    if (plan.records) {
        by_records<false>(A, true, ws, extra, stream);
        return;
    }
    if (nseg > 1) first_pass<false>(A, true, ws, stream);
    const int units = B * H * nseg;
    auto pass = [&](auto which) {
        constexpr int PASS = decltype(which)::value;
        if (fused_split(units))
            hipLaunchKernelGGL((wkv7_fused_kernel<false, true, false, CUTS_TEN, 2, false, PASS>), dim3(fused_grid(units, 2) + extra),
                               dim3(fused_threads(CUTS_TEN, false, 2)), 0, stream, A);
        else
            hipLaunchKernelGGL((wkv7_fused_kernel<false, true, false, CUTS_EIGHT_EVEN, 1, false, PASS>), dim3(fused_grid(units, 1) + extra),
                               dim3(fused_threads(CUTS_EIGHT_EVEN, false)), 0, stream, A);
    };
    if (nseg > 1) pass(std::integral_constant<int, 2>());
    else pass(std::integral_constant<int, 0>());
}

}  // namespace wkv
