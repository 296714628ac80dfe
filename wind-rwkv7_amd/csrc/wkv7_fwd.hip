// WKV7 for gfx950, what runs beside the one-kernel organisation of wkv7_fused.hip in the forward direction:
//   * the composition of the segments' affine maps for long sequences on few heads (the states entering the segments),
//   * the attn_ln epilogue as a kernel of its own (GroupNorm + bonus + gate on the kept WKV7 output; attn_ln.cu:11-37),
//     used where the plain forward kernel runs two blocks per (batch, head) and cannot host it,
//   * the rule that says when a sequence is cut into segments.
#include "ln_epilogue.hpp"
#include "device_info.hpp"
#include "wkv7_common.hpp"
#include "wkv7_kernels.hpp"

#include <algorithm>

namespace wkv {

// ------------------------------------------------------------------------------------------------
// Composes the segment maps in processing order: S(g) = S(g-1) M_g + N_g for g = 1 .. PER - 1, all in fp32 (fp32
// matrix instructions).  maps: as written by wkv7_first_pass_kernel ([pair][g]; g = 0 is not there); s_seg: [pair][g][64][64]
// floats, the state leaving segment g: entry 0 is there.
// The value rows of a state go through the maps independently, so a block takes 16 of them (four blocks per (batch,
// head)) and its four wavefronts a block of 16 key columns each: 16 matrix instructions per wavefront and segment,
// then the row block's four fragments change hands through LDS.  All maps a wavefront needs (PER <= MOST: MOST - 1 times
// 20 registers) are requested before the first product, and what is requested is read whether there or not: eight segments through the
// form for twelve took 10.9 us instead of 7.9.  (One block per (batch, head), a wavefront per 16 rows doing
// all four column blocks: 64 dependent-by-fours matrix instructions per segment, 2.8 us each, 23 us at 8 segments.)
// ------------------------------------------------------------------------------------------------
constexpr int CARRY_MAX_SEG = 12;
template <int MOST>
__global__ __launch_bounds__(256) void segment_carry_kernel(int PER, const float* __restrict__ maps, float* s_seg) {
    __shared__ f32x4 xch[2][NBLK][WAVE];
    const int jb = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int bh = blockIdx.x >> 2, ib = blockIdx.x & 3;
    const Lane L;
    f32x4 S[NBLK];
#pragma unroll
    for (int kb = 0; kb < NBLK; kb++) S[kb] = load_state_frag(s_seg, 1, bh * PER, ib, kb, L);
    f32x4 n[MOST - 1], mt[MOST - 1][NBLK];
#pragma unroll
    for (int g = 0; g < MOST - 1; g++) {
        const long e = (long)bh * PER + (g < PER - 1 ? g + 1 : PER - 1);   // (past the end: a valid map, not used)
        const float* N = maps + (e * 2 + 0) * HEAD * HEAD;
        const float* MT = maps + (e * 2 + 1) * HEAD * HEAD;
        n[g] = *reinterpret_cast<const f32x4*>(N + (16 * ib + L.n) * HEAD + 16 * jb + 4 * L.g);
#pragma unroll
        for (int kb = 0; kb < NBLK; kb++)   // A operand of S[ib][kb] M[kb][jb]: F(M[kb][jb]^T) = the (jb, kb) block of MT
            mt[g][kb] = *reinterpret_cast<const f32x4*>(MT + (16 * jb + L.n) * HEAD + 16 * kb + 4 * L.g);
    }
#pragma unroll
    for (int g = 0; g < MOST - 1; g++) {
        if (g < PER - 1) {   // (uniform; no load inside)
            f32x4 a0 = mma_f32(n[g], mt[g][0], S[0]), a1 = mma_f32(zero4(), mt[g][1], S[1]);
            a0 = mma_f32(a0, mt[g][2], S[2]);
            a1 = mma_f32(a1, mt[g][3], S[3]);
            const f32x4 T = a0 + a1;
            store_state_frag(s_seg, 1, bh * PER + g + 1, ib, jb, L, T);
            xch[g & 1][jb][lane] = T;
            __syncthreads();
#pragma unroll
            for (int kb = 0; kb < NBLK; kb++) S[kb] = xch[g & 1][kb][lane];
        }
    }
}


// ------------------------------------------------------------------------------------------------
// attn_ln epilogue: one wavefront per chunk applies GroupNorm + bonus + gate to the WKV7 output the scan
// left in y_wkv (kept, bf16, for the backward pass; centred per block when `centers` is given, see ln_epilogue.hpp).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ln_epilogue_kernel(const LnForwardArgs A, int nchunks) {
    const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= nchunks) return;
    ln_forward_chunk(A, A.H >= 16 ? head_major_chunk(wid, nchunks, A.T) : wid, Lane());   // (long rows: see head_major_chunk)
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
// Segments per (batch, head) and pass for long sequences on few heads (the whole sequence is one more): four up to 8 or 12, as many as the
// (batch, head)s leave compute units and no more than a fortieth of the chunks; 1 = the whole sequence in one block (or two).  It is cut in
// one more than that, the first one 0.8 of the others: 200 chunks at 5 are 27 and 34 or 35, 480 at 12 30 and 37 or 38.
// A segmented pass is two launches of the one-kernel organisation (wkv7_fused.hip: the first segment and the others' affine maps,
// then the scan proper from the composed entering states) with the carry between them, so it costs twice a launch's fixed
// 11-14 us, the carry's 3 us per segment, and 1.2 us per chunk and segment instead of 0.55: below four segments
// it does not pay (measured forward+backward, 12 heads: 1024 tokens 133 us in two segments against 103 in one block).
// Four segments fit up to a quarter of the compute units' worth of (batch, head) pairs (64: 8192 tokens 876 -> 768 us,
// 60 pairs: 4096 tokens 459 -> 425 us, 2048 tokens 242 -> 246 us against the unsegmented kernel).
// scan_segments_least: 4 or 8 of them where that divides the chunks and leaves each 32; what a call with scratch for no more than that
// runs.  (Segments need not divide the chunks; the condition says how much scratch a call has to bring, which is not to grow.)
// scan_segments_most: any number.  Forward + backward, us, least -> most: 40 heads x 16384 tokens 1070 (4) -> 920 (6), 48 pairs x 8192 540 (4) ->
// 507 (5), 40 x 3200 244 -> 224 (5).  Past eight where a segment has one block and not two: 24 x 16384 618 (8) -> 572 (10), 20 x 8192
// 306 -> 276 (12), 17 x 16384 514 -> 429 (12).  Odd numbers of chunks, which keep a state per chunk: 32 x 16368 1423 (1) -> 810 (8), 24 x 8176 678 -> 341
// (10), 12 x 12272 840 -> 336 (8), 30 x 4112 336 -> 242 (6), 64 x 4080 467 -> 406 (4), 64 x 2608 299 -> 276 (4).
static int scan_segments_least(int B, int T, int H) {
    const int BH = B * H, NC = T / CHUNK;
    int g = 1;
    while (g < 8 && BH * g * 2 <= compute_units() && NC % (g * 2) == 0 && NC / (g * 2) >= 32) g *= 2;
    return g >= 4 ? g : 1;
}
static int scan_segments_most(int B, int T, int H) {
    const int BH = B * H, NC = T / CHUNK, least = scan_segments_least(B, T, H);
    const int g = std::min({2 * 8 * BH > compute_units() ? CARRY_MAX_SEG : 8, compute_units() / BH, NC / 40});
    return g >= 4 && g > least ? g : least;
}
// Chunks of the segment that the first pass walks while it makes the maps of the others.  Its stores make its step longer than
// theirs.  Forward + backward, us, at 0.7 / 0.8 / 0.9 / 1 of another segment's chunks: 1 x 16384 tokens x 32 heads 692 / 687 / 692 / 698,
// 4 x 8192 x 12 545 / 540 / 542 / 542.
int first_segment_chunks(int NC, int per) { return (int)(NC * 0.8 / (per + 0.8)); }
// By records where they are the fastest (forward, keeping a state per pair / whole backward, us; one launch or segments -> records):
//   * four blocks per (batch, head) have a compute unit each: 64 pairs x 1024 tokens 44 -> 36 / 80 -> 71, 80 44.8 -> 49.2 / 91 -> 87,
//     96 45.0 -> 53.4 / 95 -> 100;
//   * from eight chunks on (without kept states: 1 pair x 128 tokens 11.6 -> 8.2; below, four chunks 8.4 -> 7.6, the gain is not worth
//     the scratch).  A training pass has two launches more then, and a short one waits for its launches: eager forward + backward
//     of attn on a host that takes 88-95 us for it, 4 x 512 tokens x 12 heads 88-91 -> 92-95, 4 x 768 99 -> 83, 1 x 1024 x 4 95 -> 95,
//     4 x 1024 x 12 116 -> 95, of attn_ln 1 x 1024 x 4 115 -> 120.  So there from 96 chunks on, or 48 and 2048 in all;
//   * up to 6144 chunks in all, 80 MiB of records, behind which writing and reading them is what counts (96 x 1024 above);
//   * less far where the sequence runs as segments otherwise, and not at all where those are six or more.  Forward keeping a state
//     per pair / whole backward, us, segments -> records, four: 24 heads x 3072 tokens 65 -> 64 / 113 -> 108, 40 x 2048 (5120 chunks) 59 -> 56 / 106 ->
//     104, 32 x 2560 60 -> 59 / 109 -> 108, 32 x 2576 60 -> 66, 48 x 2048 59 -> 64 / 114 -> 105, 32 x 3072 65 -> 77 / 119 -> 115; five: 16 x 3200 (3200 chunks)
//     61 -> 60 / 95 -> 88, 20 x 3200 61 -> 64 / 98 -> 92, 24 x 3200 61 -> 66 / 110 -> 112; six: 12 x 3840 62 -> 69 / 95 -> 94, 24 x 3840 71 -> 84 / 118 -> 126;
//     eight: 8 x 4096 55 -> 68 / 73 -> 84, 4 x 8192 85 -> 127 / 102 -> 132.
static bool scan_by_records(int B, int T, int H, ScanUse use) {
    const long BH = (long)B * H, NC = T / CHUNK, least = use == SCAN_PREFILL ? 8 : BH * NC >= 2048 ? 48 : 96;
    const int segments = scan_segments_most(B, T, H);
    const long most = segments > 5 ? 0 : segments == 1 || use == SCAN_BACKWARD ? 6144 : segments == 4 ? 5120 : 3584;
    return NC >= least && 4 * BH <= compute_units() && BH * NC <= most;
}
static size_t records_bytes(int B, int T, int H, bool fwd) { return (size_t)B * H * (T / CHUNK) * scan_record_bytes(fwd); }
// N, M^T and the entering state per segment
static size_t segments_bytes(int B, int H, int g) { return g == 1 ? 0 : (size_t)B * H * g * 3 * HEAD * HEAD * sizeof(float); }
ScanPlan scan_plan(int B, int T, int H, size_t ws_bytes, ScanUse use) {
    if (scan_by_records(B, T, H, use) && ws_bytes >= records_bytes(B, T, H, use != SCAN_BACKWARD)) return {true, 1};
    const int most = scan_segments_most(B, T, H);
    return {false, ws_bytes >= segments_bytes(B, H, most) ? most : scan_segments_least(B, T, H)};
}
size_t scan_workspace_bytes(int B, int T, int H, ScanUse use) {
    return scan_by_records(B, T, H, use) ? records_bytes(B, T, H, use != SCAN_BACKWARD) : segments_bytes(B, H, scan_segments_most(B, T, H));
}
size_t scan_workspace_least_bytes(int B, int T, int H) { return segments_bytes(B, H, scan_segments_least(B, T, H)); }

void launch_segment_carry(int BH, int per, const float* maps, float* s_seg, hipStream_t stream) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(4 * BH), dim3(256), 0, stream, per, maps, s_seg); };
    per <= 8 ? go(segment_carry_kernel<8>) : go(segment_carry_kernel<CARRY_MAX_SEG>);
}

void launch_ln_epilogue(int B, int T, int H, const void* y_wkv, const float* centers, const void* q, const void* k,
                        const void* v, const void* g, const void* params, void* y, hipStream_t stream) {
    const int nchunks = B * H * (T / CHUNK);
    auto c = [](const void* p) { return static_cast<const __bf16*>(p); };
    const LnForwardArgs A{T, H, c(y_wkv), centers, c(q), c(k), c(v), c(g), static_cast<const float*>(params), static_cast<__bf16*>(y)};
    hipLaunchKernelGGL(ln_epilogue_kernel, dim3((nchunks + 3) / 4), dim3(256), 0, stream, A, nchunks);
}

}  // namespace wkv
