// Projections y = x W^T (and input gradients dx = dy W, on the transposed weight) of a block, several in one launch.
//
// The reference leaves every product of the block to the BLAS library (time_mixer.py:120-131, :167).  The block has six
// first-half products on four inputs, two second-half ones, the output projection, and as many input gradients: most are
// too small to fill the chip on their own, each library call costs 10-15 us of host time, and the library knows neither
// that two products add up to one input gradient nor that a concatenated output is cut into columns (some through tanh)
// right after.  Here a launch takes up to nine problems on the same M tokens (eight through the C interface).  A problem is
//     D[m][n] = sum over up to two segments of  sum_k A[m][k] W[n][k]
// with D's columns going to up to four tensors, each as it is, through tanh, or times 1 - aux^2 (the derivative).
//
// Both operands lie with the contraction index fastest, so a tile goes from memory to LDS without passing registers
// (buffer_load ... lds) and from LDS into v_mfma_f32_32x32x16_bf16 as it lies: eight consecutive k of one row per lane and
// 16-byte read.  The pieces of 16 bytes of a row are permuted by the number of its pair of rows on the way into LDS (by choosing
// which piece a lane fetches), which keeps those reads out of each other's banks.  A block of four wavefronts (2 x 2) computes
// 64 TMB tokens x 64 TNB columns; what bounds it is the LDS read rate against the matrix rate: 32 x 32 blocks TMB x TNB
// per wavefront need TMB + TNB reads of 1 KB for TMB TNB instructions of 32 cycles.  Two blocks share a compute unit, so
// one's matrix work covers the other's barriers and last loads.
//
// Measured (us; in brackets the library's kernels for the same, replayed without host time): six first-half products of a
// 768-channel block with their tanh and cut columns at 2006 / 8192 / 32768 tokens 19.5 (49) / 50 (69) / 170 (203); three input
// gradients with one second segment at 8192 38 (55); a single 768 x 768 product at 512 / 8192 / 65536 tokens 7.3 (6.4) / 15.5 (16) /
// 82-90 (70).  Of the 54 us of six on inputs out of memory the matrix instructions alone take 28 (their rate on these numbers, not on
// zeros, is 1.3 PFLOP/s), with the LDS reads 32, with the loads 39; the output is the rest.  Blocks that stay and fetch the next tile's
// first stage while they write this one's output: 54.  Stages of
// 32 (half lines): 14 % slower at 65536 tokens; 256 x 192 tiles, one block per compute unit, a whole stage's operands in
// registers: 13 % slower (768 contraction indices are twelve stages, too few to amortise its start and end alone);
// walking the contraction from different places per tile: 5-15 % slower.
#include "linear_kernels.hpp"
#include "device_info.hpp"

#include "frag.hpp"

#include <cstddef>

namespace wkv {
namespace {

// tanh by the hardware's exponential: (1 - t) / (1 + t) with t = exp(-2 |x|), and where the difference loses digits the series to x^5 (its next
// term, 17/315 x^7, is 5e-8 of the value at 0.1): 1e-6 of the value at most.  The result is rounded to bf16: of every finite
// bf16 argument the nearest to its tanh in 64 bits, as by the library's, which takes three times the instructions, sixty-four times a lane.
__device__ __forceinline__ float tanh_of(float x) {
    const float a = fabsf(x), t = __builtin_amdgcn_exp2f(a * -2.8853900817779268f);   // 2 log2(e)
    const float x2 = a * a, small = a * fmaf(x2, fmaf(x2, 2.f / 15, -1.f / 3), 1.f);
    return copysignf(a < 0.1f ? small : (1.f - t) * __builtin_amdgcn_rcpf(1.f + t), x);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int problem_words16 __attribute__((ext_vector_type(16), aligned(8)));   // (as a LinearProblem lies)
typedef int problem_words4 __attribute__((ext_vector_type(4), aligned(8)));
static_assert(alignof(problem_words16) <= alignof(LinearProblem) && alignof(problem_words4) <= alignof(LinearProblem), "what is read as such");
using Rsrc = __amdgpu_buffer_rsrc_t;

constexpr int BK = 64;           // contraction indices per stage: whole 128-byte lines of a row
constexpr int MAX_PROBLEMS = LINEAR_GROUP_MAX;

template <int TMB, int TNB>
struct Tile {
    static constexpr int BM = 64 * TMB, BN = 64 * TNB;
    static constexpr int STAGE_BYTES = (BM + BN) * BK * 2;
};

struct GroupArgs {
    // what a block finds its tile by: of problem j its tiles (0 past the last problem), and 4 times those in a row of blocks + TNB
    i32x16 tiles, columns;   // tiles[15]: M
    LinearProblem p[MAX_PROBLEMS];
};

// STAGES in LDS: two where blocks share a compute unit; four in launches that have less than a block per compute unit, where
// nothing but a block's own loads in flight covers their latency (512 x 768 x 768: 10.5 -> 8.9 us).
template <int TMB, int TNB, int STAGES>
__device__ __forceinline__ void gemm_tile(unsigned char* lds, const LinearProblem& p, const int M, const int m0, const int n0) {
    using S = Tile<TMB, TNB>;
    // (what the first loads need, at once: see linear_group_kernel)
    struct Operands {
        const __bf16 *A[2], *W[2];
        long lda[2], ldw[2];
    };
    struct Lengths {
        int K[2], N, npieces;
    };
    static_assert(offsetof(LinearProblem, lda) == offsetof(Operands, lda) && offsetof(LinearProblem, K) == sizeof(Operands) &&
                  offsetof(LinearProblem, npieces) == sizeof(Operands) + offsetof(Lengths, npieces), "the head of a LinearProblem");
    problem_words16 operand_words = *reinterpret_cast<const problem_words16*>(&p);
    problem_words4 length_words = *reinterpret_cast<const problem_words4*>(p.K);
    asm volatile("" : "+s"(operand_words), "+s"(length_words));
    const Operands o = __builtin_bit_cast(Operands, operand_words);
    const Lengths len = __builtin_bit_cast(Lengths, length_words);
    constexpr int CPR = BK / 8;                      // 16-byte pieces per row
    constexpr int RPP = 256 / CPR;                   // rows per pass of the block
    constexpr int QA = S::BM / RPP, QB = S::BN / RPP, LOADS = QA + QB;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = tid / CPR;                      // this thread's row in a pass
    // (LDS answers sixteen lanes' 16-byte reads at a time, 256 bytes: two rows a line, so the pieces are permuted by pairs of
    // rows.  By single rows, 47 % of the cycles that LDS was busy were conflicts, now 5 %; six products of the sizes of a 768-channel
    // block, each to one tensor as it is, 42.4 -> 41.8 us, 65536 x 768 x 768 91 -> 90: LDS is busy 16 % of the time.)
    auto swizzle = [](int row) { return (row >> 1) & 7; };
    static_assert(CPR == 8, "a row of a stage is one 128-byte line");
    const int piece = (tid % CPR) ^ swizzle(lrow);   // the piece of the row it fetches (RPP is a multiple of 8: the same in every pass)

    f32x16 acc[TMB][TNB];
#pragma unroll
    for (int mb = 0; mb < TMB; mb++)
#pragma unroll
        for (int nb = 0; nb < TNB; nb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[mb][nb][r] = 0.f;

    // stages of both segments in a row
    const int nk0 = (len.K[0] + BK - 1) / BK, nk = nk0 + (len.K[1] + BK - 1) / BK;
    Rsrc ra, rb;
    unsigned aoff[QA], boff[QB];
    int kseg = 0;
    auto enter_segment = [&](int g) {   // descriptors at the tile's first rows; rows past the ends repeat the last
        ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(o.A[g] + (long)m0 * o.lda[g]), 0, 0x7fffffff, 0x00020000);
        rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(o.W[g] + (long)n0 * o.ldw[g]), 0, 0x7fffffff, 0x00020000);
#pragma unroll
        for (int q = 0; q < QA; q++) aoff[q] = (unsigned)min(lrow + RPP * q, M - 1 - m0) * (unsigned)o.lda[g] * 2;
#pragma unroll
        for (int q = 0; q < QB; q++) boff[q] = (unsigned)min(lrow + RPP * q, len.N - 1 - n0) * (unsigned)o.ldw[g] * 2;
        kseg = len.K[g];
    };
    auto k_of = [&](int kt) { return BK * (kt >= nk0 ? kt - nk0 : kt); };
    auto issue = [&](int kt) {
        if (kt == nk0) enter_segment(1);
        const int k0 = k_of(kt);
        const int c = k0 + 8 * piece < kseg ? k0 + 8 * piece : k0;   // (past the segment's end: a piece that is not used)
        unsigned char* dst = lds + (kt % STAGES) * S::STAGE_BYTES + wave * 1024;
#pragma unroll
        for (int q = 0; q < QA; q++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst + q * 4096, 16, aoff[q] + 2 * c, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < QB; q++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst + S::BM * BK * 2 + q * 4096, 16, boff[q] + 2 * c, 0, 0, 0);
    };
    // operand reads: lane = row (lane % 32) of a 32-row block, k = 16 ks + 8 (lane / 32) ..
    const int r32 = lane & 31, half = lane >> 5;
    int rd[BK / 16];
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) rd[ks] = r32 * (BK * 2) + (((2 * ks + half) ^ swizzle(r32)) << 4);
    const int a_base = wm * TMB * 32 * BK * 2, b_base = S::BM * BK * 2 + wn * TNB * 32 * BK * 2;

    // a stage of every wavefront has arrived when at most `after` stages behind it are on their way, and nobody reads the one
    // before it any more (own LDS reads are waited for: their consumers could be scheduled behind the barrier)
    auto arrived = [&](int after) {
        if (STAGES > 3 && after >= 3)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(3 * LOADS) : "memory");
        else if (STAGES > 2 && after == 2)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * LOADS) : "memory");
        else if (after == 1)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    enter_segment(0);
    // Operands of a 16-wide step are read from LDS while the step before multiplies, across stages too: the barrier for
    // stage kt + 1 stands before the last step of stage kt, whose operands are in registers by then, so that stage's place
    // is free for stage kt + STAGES right there.
    constexpr int KS = BK / 16;
    bf16x8 a[2][TMB], b[2][TNB];
    auto read = [&](int set, int kt, int ks) {
        const unsigned char* st = lds + (kt % STAGES) * S::STAGE_BYTES;
#pragma unroll
        for (int mb = 0; mb < TMB; mb++) a[set][mb] = *reinterpret_cast<const bf16x8*>(st + a_base + mb * 32 * BK * 2 + rd[ks]);
#pragma unroll
        for (int nb = 0; nb < TNB; nb++) b[set][nb] = *reinterpret_cast<const bf16x8*>(st + b_base + nb * 32 * BK * 2 + rd[ks]);
        if (ks > 0 && 16 * ks >= len.K[kt >= nk0 ? 1 : 0] - k_of(kt)) {   // past a segment's end: zeros
#pragma unroll
            for (int mb = 0; mb < TMB; mb++) a[set][mb] = bf16x8{};
#pragma unroll
            for (int nb = 0; nb < TNB; nb++) b[set][nb] = bf16x8{};
        }
    };
#pragma unroll
    for (int st = 0; st < STAGES; st++)
        if (st < nk) issue(st);
    // (where a single tensor takes the output, while the operands are on their way)
    __bf16* out0 = p.out[0];
    long ld_out0 = p.ld_out[0];
    int op0 = p.op[0];
    asm volatile("" : "+s"(out0), "+s"(ld_out0), "+s"(op0));
    arrived(min(nk - 1, STAGES - 1));
    read(0, 0, 0);
    for (int kt = 0; kt < nk; kt++) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks < KS - 1) {
                read((ks + 1) & 1, kt, ks + 1);
            } else if (kt + 1 < nk) {
                arrived(min(nk - 2 - kt, STAGES - 2));
                if (kt + STAGES < nk) issue(kt + STAGES);
                read((ks + 1) & 1, kt + 1, 0);
            }
#pragma unroll
            for (int mb = 0; mb < TMB; mb++)
#pragma unroll
                for (int nb = 0; nb < TNB; nb++)
                    acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[ks & 1][nb], a[ks & 1][mb], acc[mb][nb], 0, 0, 0);
        }
    }
    // Register r of lane l of block (mb, nb): token 32 mb + l % 32, column 32 nb + 8 (r / 4) + 4 (l / 32) + r % 4.  Eight columns lie in one
    // output tensor, so what is done to the registers 4 q .. 4 q + 3 is the same for the whole wavefront: tanh and its derivative
    // are applied here, to the sums as bf16, as they leave, with all of the derivative's operands requested at once.  (Row by row on the way
    // out, each lane finding its tensor and waiting for its operand: the two gradients through tanh of a 768-channel block at 32768 tokens 40.6 us, now
    // 35.6; six first halves at 512 tokens 13.9, now 13.5.)
    const int m_first = m0 + 32 * TMB * wm, n_first = n0 + 32 * TNB * wn;
    const bool plain = len.npieces == 1 && op0 == LINEAR_PLAIN;
    auto tensor_of = [&](int col) {
        int t = 0;
#pragma unroll
        for (int k = 1; k < LinearProblem::PIECES; k++) t += k < len.npieces && col >= p.start[k] ? 1 : 0;
        return t;
    };
    auto of = [&](int t, auto f) {
        auto r = f(0);
#pragma unroll
        for (int k = 1; k < LinearProblem::PIECES; k++) r = t == k ? f(k) : r;
        return r;
    };
    if (!plain) {
        bf16x4 y[TMB][TNB][4];
#pragma unroll
        for (int nb = 0; nb < TNB; nb++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int col = n_first + 32 * nb + 8 * q, t = tensor_of(col);
                const bool wanted = of(t, [&](int k) { return p.op[k]; }) == LINEAR_TANH_GRAD && col < len.N;
                const int width = of(t, [&](int k) { return p.width[k]; });
                const __bf16* const aux = of(t, [&](int k) { return p.aux[k]; }) + (col - of(t, [&](int k) { return p.start[k]; }) + 4 * half);
#pragma unroll
                for (int mb = 0; mb < TMB; mb++) {
                    y[mb][nb][q] = bf16x4{};
                    if (wanted) y[mb][nb][q] = *reinterpret_cast<const bf16x4*>(aux + (long)min(m_first + 32 * mb + r32, M - 1) * width);
                }
            }
#pragma unroll
        for (int nb = 0; nb < TNB; nb++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int t = tensor_of(n_first + 32 * nb + 8 * q), op = of(t, [&](int k) { return p.op[k]; });
                if (op != LINEAR_PLAIN) {
#pragma unroll
                    for (int mb = 0; mb < TMB; mb++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float f = (float)(__bf16)acc[mb][nb][4 * q + e], g = (float)y[mb][nb][q][e];
                            acc[mb][nb][4 * q + e] = op == LINEAR_TANH ? tanh_of(f) : f * (1.f - g * g);
                        }
                }
            }
    }
    // Two lanes swap their halves so that a lane has eight consecutive columns of a token; the wavefront's tile then goes through
    // LDS and leaves in rows (as it lies in registers every store would touch 32 rows for 32 bytes each: 8192 x 768 x 64, which
    // is all output, 13 us instead of 9), through the L2: what the end of the kernel writes back of the output is a time in which
    // nothing else runs (one 768 x 768 product at 8192 tokens 17.9 -> 16.5 us, two second halves 10.3 -> 9.0, six first halves at 2006 tokens 21.4 -> 19.5;
    // past all caches faster still where the output is more than they hold, but the block, which reads it next, 615 -> 619).
    constexpr int CH = 4 * TNB, PITCH = 32 * TNB * 2 + 16;   // 16-byte pieces per row of the wavefront; its LDS row, bank-shifted
    static_assert(4 * 32 * TMB * PITCH <= STAGES * (64 * TMB + 64 * TNB) * BK * 2, "the output tile fits where the stages were");
    arrived(0);
    unsigned char* const mine = lds + wave * (32 * TMB * PITCH);
#pragma unroll
    for (int mb = 0; mb < TMB; mb++)
#pragma unroll
        for (int nb = 0; nb < TNB; nb++)
#pragma unroll
            for (int pr = 0; pr < 2; pr++) {
                const f32x16& x = acc[mb][nb];
                const u32x2 lo = __builtin_bit_cast(u32x2, pack_bf16(x[8 * pr], x[8 * pr + 1], x[8 * pr + 2], x[8 * pr + 3]));
                const u32x2 hi = __builtin_bit_cast(u32x2, pack_bf16(x[8 * pr + 4], x[8 * pr + 5], x[8 * pr + 6], x[8 * pr + 7]));
                // lanes below 32 take columns 0 .. 7 of the sixteen, the others 8 .. 15
                const auto s0 = __builtin_amdgcn_permlane32_swap(lo[0], hi[0], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(lo[1], hi[1], false, false);
                typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<u32x4*>(mine + (32 * mb + r32) * PITCH + (4 * nb + 2 * pr + half) * 16) = (u32x4){s0[0], s1[0], s0[1], s1[1]};
            }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (a wavefront reads what it wrote itself)
    auto rows_of = [&](int i, int& m, int& col) -> const bf16x8* {
        const int id = lane + 64 * i, row = id / CH, ch = id % CH;
        m = m0 + 32 * TMB * wm + row, col = n0 + 32 * TNB * wn + 8 * ch;
        return reinterpret_cast<const bf16x8*>(mine + row * PITCH + ch * 16);
    };
    if (plain) {
#pragma unroll
        for (int i = 0; i < 2 * TMB * TNB; i++) {
            int m, col;
            const bf16x8* v = rows_of(i, m, col);
            if (m < M && col < len.N) store_through(out0 + (long)m * ld_out0 + col, *v);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 2 * TMB * TNB; i++) {
        int m, col;
        const bf16x8* v = rows_of(i, m, col);
        if (m < M && col < len.N) {
            const int t = tensor_of(col);
            __bf16* const out = of(t, [&](int k) { return p.out[k]; }) + (long)m * of(t, [&](int k) { return p.ld_out[k]; });
            store_through(out + (col - of(t, [&](int k) { return p.start[k]; })), *v);
        }
    }
}

template <int TMB, int STAGES>
__global__ __launch_bounds__(256, STAGES == 2 ? 2 : 1) void linear_group_kernel(const GroupArgs G) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * Tile<TMB, 3>::STAGE_BYTES];
    // Blocks go to the eight XCDs in turn (block b to XCD b % 8), and each XCD has an L2 of its own.  An XCD takes a run of
    // consecutive tiles, i.e. some row blocks of a problem with all their column blocks: it reads each of its rows of the
    // input once and keeps the weight.
    // All of it in scalar registers before it is looked at, and so with a tile's operands and its output: left to the compiler these are
    // scalar loads where each is used, seven one after the other before the first load of an operand (77 x 8 x 8 3.9 -> 3.1 us, one
    // 768 x 768 product at 512 tokens 8.3 -> 7.3, at 2006 10.7 -> 9.5, two second halves at 2006 5.6 -> 4.9, four input gradients at 512 12.0 -> 10.7).
    i32x16 tiles = G.tiles, columns = G.columns;
    asm volatile("" : "+s"(tiles), "+s"(columns));
    const unsigned x = blockIdx.x % 8;
    unsigned rest = blockIdx.x / 8, tile = 0;
    int j = -1, of_row = 5;
#pragma unroll
    for (int k = 0; k < MAX_PROBLEMS; k++) {   // problem by problem: tiles of XCD x are [T x / 8, T (x+1) / 8) of each problem's T
        const unsigned T = tiles[k], lo = T * x / 8, here = T * (x + 1) / 8 - lo;
        const bool found = j < 0 && rest < here;
        j = found ? k : j, tile = found ? lo + rest : tile, of_row = found ? columns[k] : of_row;
        rest -= here;   // (not looked at any more once it is found)
    }
    if (j < 0) return;   // (whole block)
    const LinearProblem& p = G.p[j];
    const unsigned ncol = of_row >> 2, shape = of_row & 3;
    const int M = tiles[15], m0 = tile / ncol * (64 * TMB), n0 = tile % ncol * (64 * shape);
    switch (shape) {
        case 1: gemm_tile<TMB, 1, STAGES>(lds, p, M, m0, n0); break;
        case 2: gemm_tile<TMB, 2, STAGES>(lds, p, M, m0, n0); break;
        default: gemm_tile<TMB, 3, STAGES>(lds, p, M, m0, n0); break;
    }
}

}  // namespace

void launch_linear_group(int n, long M, const LinearProblem* problems, hipStream_t stream) {
    GroupArgs G{};
    static_assert(MAX_PROBLEMS < 15, "one place is left for M");
    G.tiles[15] = (int)M;
    // Columns per block (64 times this): as many of a problem's as the shape allows, since wide tiles read least per product.
    int all = 0;
    auto plan = [&](int rows, int widest) {
        all = 0;
        for (int j = 0; j < n; j++) {
            const int N = problems[j].N, blocks = (N + 63) / 64;
            const int shape = blocks < widest ? blocks : widest == 3 && N % 192 != 0 && N <= 256 ? 2 : widest, ncol = (blocks + shape - 1) / shape;
            G.columns[j] = 4 * ncol + shape;
            all += G.tiles[j] = (int)((M + rows - 1) / rows) * ncol;
        }
        return all;
    };
    for (int j = 0; j < n; j++) G.p[j] = problems[j];
    // 128 tokens x 192 columns where that gives every compute unit a block; else 64 tokens, and narrower until most have one
    const int enough = compute_units() * 3 / 4;
    const bool small = plan(128, 3) < compute_units();
    if (small && plan(64, 3) < enough && plan(64, 2) < enough) plan(64, 1);
    // the largest share of an XCD, times eight
    int most = 0;
    for (int x = 0; x < 8; x++) {
        int c = 0;
        for (int j = 0; j < n; j++) {
            const int T = G.tiles[j];
            c += T * (x + 1) / 8 - T * x / 8;
        }
        most = c > most ? c : most;
    }
    const dim3 grid(8 * most), block(256);
    if (!small) hipLaunchKernelGGL((linear_group_kernel<2, 2>), grid, block, 0, stream, G);
    else if (all > compute_units()) hipLaunchKernelGGL((linear_group_kernel<1, 2>), grid, block, 0, stream, G);
    else hipLaunchKernelGGL((linear_group_kernel<1, 4>), grid, block, 0, stream, G);
}

}  // namespace wkv
