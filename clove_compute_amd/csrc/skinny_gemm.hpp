// GEMM for few rows of A (M <= 128) against a large N-contiguous B on gfx950:
// the prefill/small-batch shapes of gemm_fp16 and gemm_int8, where the run
// time is streaming B (the weights) from HBM once.
//
//   acc[m, n] = sum_k A[m, k] * B[k, n]      fp16 -> fp32, or int8 -> int32
//
// Both operands go global -> LDS by LDS DMA (buffer_load_dwordx4 ... lds, no
// VGPR staging), several stages in flight.  B stays N-contiguous in LDS and
// its MFMA fragments come from the transposing LDS reads: within a 16-lane
// group, ds_read_b64_tr_b16 gives result lane j element r = source lane
// (4 r + j / 4) element (j % 4), and ds_read_b64_tr_b8 gives result lane j
// byte r = source lane (2 r + j / 8) byte (j % 8); with source lane s of a
// group pointing at 8 bytes of k-row kb + s / 4 (fp16; s / 2 for int8),
// columns of the group's 16, every result lane receives 4 (8) consecutive k
// of one column.  Two such reads make the 16-byte MFMA operand.
//
// LDS layout per stage (16-byte chunks XOR-swizzled so that every fragment
// read is bank-conflict free):
//   A  BM rows x 128 bytes of k:   chunk c of row m at c ^ (m & 7)
//   B  BK k-rows x BNB bytes of n: chunk c of row r at c ^ swz_b(r)
// MFMA: v_mfma_f32_32x32x16_f16 / v_mfma_i32_32x32x32_i8 with the B fragment
// as the "A" operand (rows = n) and the A fragment as "B" (cols = m): a lane
// holds one row m and 4-column runs of n.  A k-step consumes 32 bytes of k.
//
// Split-K over workgroups (whole K tiles) when the tile grid does not cover
// the CUs, with the shared publish / reduce (split order, deterministic;
// int32 partials for INT8, so the integer accumulator stays exact).
//
// K slices (KW > 1, FP16 only): the small products (short K, a 32x32 tile per
// CU or fewer) run 32x32 tiles whose four waves each take one of every K
// tile's four k-steps; after the K loop every wave stores its sums to LDS and
// each wave adds the four slices, in slice order, for a quarter of the tile's
// output runs.  Up to 32 rows on moderate weights run 32x64 tiles with two
// slices, which also split K over workgroups.
//
// Zero points (ZP, INT8): with
//   sum (a - za)(b - zb) = sum ab - zb rowsum(A) - za colsum(B) + k za zb
// the sums come from the MFMA operands already in registers: a fragment lane
// holds 16 k of one column (row), so four v_dot4 against ones per fragment and
// k-step add them up (VALU, beside an MFMA pipe that is mostly idle here: the
// kernel streams B), and the correction is applied to the split's
// accumulators before they are published (int32 wrap-around, exact).  A
// separate pass for the column sums would read the weights twice (with one, a
// thread per column, and the register-staged kernel behind it, 512 x 4096 x
// 4096 with an activation zero point took 1041 us; here it takes 22.6).
//
// Ragged K (K not a multiple of the K tile): the k-rows of B past K lie past
// the end of the operand and read as zero; A's chunks past K would read the
// next row, so for FP16 (whose stray bits could be NaN or infinity) their
// lanes take an offset past the end instead.
//
// Unaligned operands (UA): row strides or pointers that are not multiples of
// 16 bytes, which an LDS DMA cannot take.  The same chunks go global -> VGPR
// by 16-byte loads at element alignment (ordinary loads, which gfx950 takes at
// any byte address) -> the same LDS layout, P K tiles ahead in registers
// and two LDS stages.  A chunk of the last K tile is loaded from at most 16 bytes
// before the operand's end and shifted into place, and what lies past K is
// zeroed, so no access leaves an operand; chunks past M or N load row or
// column 0.  Stores and the loads of C take any alignment too.  Bound as the
// aligned form by operand bytes per CU, plus the LDS writes; measured against
// the generic kernel, whose loader gathers element by element (us per call):
// FP16 333 x 5001 x 2050 142 -> 31.5, 496 x 3512 x 3275 264 -> 38; INT8 with a
// zero point 1184 x 3392 x 6900 3538 -> 95, 1 x 1408 x 7922 1932 -> 9.
//
// Two B operands (NB = 2, FP16 only): B and B2 share A and the tile's
// columns; each stage holds A, then the B tile, then the B2 tile, and every
// wave keeps both accumulator sets.  The SwiGLU epilogue (kF16SwiGLU) then
// writes fp16(silu(fp16(A@B)) * fp16(A@B2)) -- gate and up of an MLP -- with
// neither projection reaching memory.  Each accumulator sums its k in the
// same order as the one-operand kernel with the same BM, BN and split plan,
// so gate and up are bit-identical to two separate GEMMs.
#pragma once

#include "common.hpp"
#include "f16_dma_gemm.hpp"
#include "skinny_plan.hpp"

namespace clove {
namespace sk {

using namespace hw;
using dma::dma16;
using dma::make_rsrc;
using dma::vmcnt_imm;

enum Out { kF16AlphaBeta = 0, kI8Tensor = 1, kI8RowCol = 2, kI8Acc32 = 3, kF16SwiGLU = 4 };

struct Args {
    const void* A;       // [batch][M, K]
    const void* B;       // [batch][K, N]
    const void* B2;      // [batch][K, N], second B operand (NB = 2)
    void* C;             // [batch][M, N]  fp16, or int32 for kI8Acc32
    const uint16_t* sa;  // [M] fp16 (kI8RowCol)
    const uint16_t* sb;  // [N] fp16 (kI8RowCol)
    float scale;         // kI8Tensor
    float alpha, beta;   // kF16AlphaBeta
    int za, zb, acc_add; // ZP: zero points of A and B; acc_add goes to every accumulator
    int M, N, K;
    int64_t sA, sB, sC;  // batch strides, elements
    int tiles_m, tiles_n, batch, nsplit, kps;  // kps: K per split (multiple of BK)
    float* part;
    unsigned* counters;
};

typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef int i32x2v __attribute__((vector_size(8)));
typedef short i16x4v __attribute__((vector_size(8)));
typedef __attribute__((address_space(3))) i32x2v lds_i32x2v;
typedef __attribute__((address_space(3))) i16x4v lds_i16x4v;

__device__ __forceinline__ u32x4 lds_read16(unsigned a) { return *reinterpret_cast<const lds_u32x4*>((size_t)a); }

template <bool I8>
__device__ __forceinline__ u32x2 lds_read_tr(unsigned a) {
    if constexpr (I8) {
        const i32x2v v = __builtin_amdgcn_ds_read_tr8_b64_v2i32(reinterpret_cast<lds_i32x2v*>((size_t)a));
        return u32x2{(unsigned)v[0], (unsigned)v[1]};
    } else {
        const i16x4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_i16x4v*>((size_t)a));
        return bitcast<u32x2>(v);
    }
}

// wait until stage t has landed, `ahead` later stages may stay in flight,
// then the workgroup barrier
// (ahead <= S - 2)
template <int S, int D, int A = S - 2>
__device__ __forceinline__ void stage_wait(int ahead) {
    if constexpr (A >= 1) {
        if (ahead >= A) {
            dma::stage_barrier<vmcnt_imm(A * D)>();
            return;
        }
        stage_wait<S, D, A - 1>(ahead);
    } else {
        dma::stage_barrier<vmcnt_imm(0)>();
    }
}

// how the operands reach LDS (see the header comment): by DMA with K a multiple
// of the K tile (any aligned K for INT8), by DMA with ragged K, through VGPRs.
// A kernel of its own for whole K tiles: with the ragged tail's branch beside
// every stage's DMAs, 128 x 4096 x 11008 took 32.7 instead of 32.1 us.
enum Feed { kWhole = 0, kRagged = 1, kUnaligned = 2 };

template <class CF, int OUT, bool ZP = false, Feed FEED = kWhole>
__global__ void __launch_bounds__(CF::NT) skinny_gemm(Args p) {
    static_assert(!ZP || CF::I8, "zero points: INT8 only");
    constexpr bool UA = FEED == kUnaligned;
    static_assert(FEED == kWhole || CF::NB == 1, "ragged or unaligned: one B operand");
    static_assert(FEED != kRagged || !CF::I8, "INT8 needs no ragged form: stray k of A meet zeros of B");
    constexpr int ES = CF::ES, NW = CF::NW, FM = CF::FM, FN = CF::FN, S = CF::S;
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, BNB = CF::BNB, SB = CF::SB;
    constexpr int D = CF::D;
    constexpr bool I8 = CF::I8;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / (CF::WM * CF::WN);  // k slice (0 unless KW > 1)
    const int wmn = wave - kw * (CF::WM * CF::WN);
    const int wm = wmn % CF::WM, wn = wmn / CF::WM;
    constexpr int NKS = CF::NKS;

    // ---- tile, split, K range ----
    // Workgroups are dealt to the 8 XCDs round-robin (workgroup b runs on XCD
    // b % 8) and each XCD has its own L2: the grid is renumbered so that every
    // XCD owns a contiguous run of logical workgroups.  Logical order is
    // split-major (the workgroups in flight together share K rows of B), and
    // within a split the tiles are walked in groups of 8 tile-rows, column by
    // column, so one XCD's run shares a few A row panels and B column panels
    // instead of touching every A panel.
    int bid = blockIdx.x;
    if ((gridDim.x & 7) == 0) bid = (bid & 7) * (int)(gridDim.x >> 3) + (bid >> 3);
    const int ntiles = p.tiles_m * p.tiles_n * p.batch;
    const int split = bid / ntiles;
    int tile = bid - split * ntiles;
    const int per_batch = p.tiles_m * p.tiles_n;
    const int batch = tile / per_batch;
    const int t_in = tile - batch * per_batch;
    constexpr int GM = 8;
    const int group = t_in / (GM * p.tiles_n);
    const int first_m = group * GM;
    const int gm = min(p.tiles_m - first_m, GM);
    const int in_group = t_in - group * GM * p.tiles_n;
    const int tm = first_m + in_group % gm, tn = in_group / gm;
    const int m0 = tm * BM, n0 = tn * BN;
    const int M = p.M, N = p.N, K = p.K;
    const int kbeg = split * p.kps;
    const int nkt = (min(K, kbeg + p.kps) - kbeg + BK - 1) / BK;

    const unsigned lds0 = __builtin_amdgcn_readfirstlane(
        (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem));

    const unsigned char* Ab = static_cast<const unsigned char*>(p.A) + batch * p.sA * ES;
    const unsigned char* Bb = static_cast<const unsigned char*>(p.B) + batch * p.sB * ES;
    const u32x4 ra = make_rsrc(Ab, (unsigned)M * K * ES);
    const u32x4 rb = make_rsrc(Bb, (unsigned)K * N * ES);
    const u32x4 rb2 = CF::NB == 2
        ? make_rsrc(static_cast<const unsigned char*>(p.B2) + batch * p.sB * ES, (unsigned)K * N * ES)
        : rb;

    // ---- per-lane DMA offsets (fixed over K; the K position is the soffset) ----
    int offa[CF::DA], offb[CF::DB];
#pragma unroll
    for (int i = 0; i < CF::DA; ++i) {
        const int row = 8 * (wave * CF::DA + i) + (lane >> 3);
        offa[i] = (m0 + row) * K * ES + 16 * ((lane & 7) ^ (row & 7));
    }
    constexpr int CPR = BNB / 16, RPI = 1024 / BNB;  // chunks per B row, rows per instruction
#pragma unroll
    for (int i = 0; i < CF::DB; ++i) {
        const int row = RPI * (wave * CF::DB + i) + lane / CPR;
        offb[i] = row * N * ES + n0 * ES + 16 * ((lane % CPR) ^ swz_b<BNB, I8>(row));
    }
    auto issue = [&](int t, int stage) {
        const int k0 = kbeg + t * BK;
        const unsigned st = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(stage * SB));
        if (FEED == kRagged && k0 + BK > K) {
            // ragged K: a lane whose chunk starts at or past K reads past the end, zero
            const bool past = k0 + 8 * ((lane & 7) ^ (lane >> 3)) >= K;
#pragma unroll
            for (int i = 0; i < CF::DA; ++i)
                dma16(ra, st + (wave * CF::DA + i) * 1024, past ? 0x7ffffff0 : offa[i], k0 * ES);
        } else {
#pragma unroll
            for (int i = 0; i < CF::DA; ++i) dma16(ra, st + (wave * CF::DA + i) * 1024, offa[i], k0 * ES);
        }
#pragma unroll
        for (int i = 0; i < CF::DB; ++i)
            dma16(rb, st + CF::A_BYTES + (wave * CF::DB + i) * 1024, offb[i], k0 * N * ES);
        if constexpr (CF::NB == 2) {
#pragma unroll
            for (int i = 0; i < CF::DB; ++i)
                dma16(rb2, st + CF::A_BYTES + CF::B_BYTES + (wave * CF::DB + i) * 1024, offb[i], k0 * N * ES);
        }
    };

    // ---- fragment addressing (relative to the stage) ----
    const int kh = lane >> 5, l32 = lane & 31;
    // A: row wm*32FM + 32j + l32, k-step t reads chunk (2t + kh) ^ (l & 7); tile j is +4096 j.
    // The wave's k-steps of a K tile are t = NKS kw + u, u < NKS.
    unsigned aoff[NKS];
#pragma unroll
    for (int u = 0; u < NKS; ++u) {
        const int t = NKS * kw + u;
        aoff[u] = (wm * 32 * FM + l32) * 128 + 16 * ((2 * t + kh) ^ (lane & 7));
    }
    // B: group g = l32 / 16 covers columns wn*32FN + 32i + 16g .. +15; source lane s = lane & 15
    // points at k-row (step rows) + s / RL and byte 8 (s % LR) of the group's columns
    constexpr int RL = I8 ? 2 : 4;        // lanes per k-row in one transposing read
    constexpr int RR = 16 / RL;           // k-rows per transposing read
    const int s16 = lane & 15, g = l32 >> 4;
    // (the swizzle mixes chunk bits that distinguish the tiles i, so every
    // tile has its own offsets)
    unsigned boff[NKS][2][FN];            // [k-step][read][tile]
#pragma unroll
    for (int u = 0; u < NKS; ++u)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < FN; ++i) {
                const int t = NKS * kw + u;
                const int row = t * (32 / ES) + kh * (16 / ES) + e * RR + s16 / RL;
                const int col = (wn * 32 * FN + 32 * i + 16 * g) * ES + 8 * (s16 % RL);
                boff[u][e][i] = CF::A_BYTES + row * BNB + 16 * ((col >> 4) ^ swz_b<BNB, I8>(row)) + (col & 15);
            }

    typedef typename std::conditional<I8, i32x16, f32x16>::type AccT;
    typedef typename std::conditional<I8, i32x4, f32x4>::type AccT4;
    constexpr int NB = CF::NB;
    static_assert((OUT == kF16SwiGLU) == (NB == 2), "the SwiGLU epilogue takes two B operands");
    AccT acc[NB][FN][FM];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[b][i][j][v] = 0;

    // ZP: this lane's partial sums of column 32 i + l32 (row 32 j + l32) of the
    // wave's tile, over the k of its lane half
    int csum[ZP ? FN : 1], rsum[ZP ? FM : 1];
    if constexpr (ZP) {
#pragma unroll
        for (int i = 0; i < FN; ++i) csum[i] = 0;
#pragma unroll
        for (int j = 0; j < FM; ++j) rsum[j] = 0;
    }
    auto ones_dot = [](const u32x4& f, int s) {
#pragma unroll
        for (int d = 0; d < 4; ++d) s = __builtin_amdgcn_sdot4((int)f[d], 0x01010101, s, false);
        return s;
    };

    // one K tile (k0 its first k) from the stage at LDS address st
    auto compute = [&](unsigned st, [[maybe_unused]] int k0) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            u32x4 af[FM];
            const unsigned ab = st + aoff[ks];
#pragma unroll
            for (int j = 0; j < FM; ++j) af[j] = lds_read16(ab + 4096 * j);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                u32x4 bf[FN];
#pragma unroll
                for (int i = 0; i < FN; ++i) {
                    const u32x2 lo = lds_read_tr<I8>(st + b * CF::B_BYTES + boff[ks][0][i]);
                    const u32x2 hi = lds_read_tr<I8>(st + b * CF::B_BYTES + boff[ks][1][i]);
                    bf[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
                }
                if constexpr (ZP) {
                    if (p.za != 0) {
#pragma unroll
                        for (int i = 0; i < FN; ++i) csum[i] = ones_dot(bf[i], csum[i]);
                    }
                    if (p.zb != 0) {
#pragma unroll
                        for (int j = 0; j < FM; ++j) {
                            const int r = ones_dot(af[j], rsum[j]);
                            // (aligned ragged K: chunks past K hold the next row)
                            rsum[j] = UA || k0 + 16 * (2 * ks + kh) < K ? r : rsum[j];
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < FN; ++i)
#pragma unroll
                    for (int j = 0; j < FM; ++j) {
                        if constexpr (I8)
                            acc[b][i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                                bitcast<i32x4>(bf[i]), bitcast<i32x4>(af[j]), acc[b][i][j], 0, 0, 0);
                        else
                            acc[b][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                bitcast<f16x8>(bf[i]), bitcast<f16x8>(af[j]), acc[b][i][j], 0, 0, 0);
                    }
            }
        }
    };

    if constexpr (!UA) {
#pragma unroll
        for (int t = 0; t < S - 1; ++t)
            if (t < nkt) issue(t, t);

        int stage = 0, stage_next = S - 1;
        for (int t = 0; t < nkt; ++t) {
            stage_wait<S, D>(min(S - 2, nkt - 1 - t));
            if (t + S - 1 < nkt) issue(t + S - 1, stage_next);
            const unsigned st = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(stage * SB));
            stage_next = stage;
            stage = stage + 1 == S ? 0 : stage + 1;
            if constexpr (I8) {
                compute(st, kbeg + t * BK);
            } else {
                // (the same as compute, written out: through the closure the compiler
                // schedules the 128x64 tiles' LDS reads around other waits, 128 x 4096 x
                // 11008 33.4 against 32.9 us, 100 x 8192 x 4096 23.1 against 22.4; INT8 is
                // ahead with it, 512 x 4096 x 4096 with a zero point 26.4 against 27.4)
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    u32x4 af[FM];
                    const unsigned ab = st + aoff[ks];
#pragma unroll
                    for (int j = 0; j < FM; ++j) af[j] = lds_read16(ab + 4096 * j);
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        u32x4 bf[FN];
#pragma unroll
                        for (int i = 0; i < FN; ++i) {
                            const u32x2 lo = lds_read_tr<I8>(st + b * CF::B_BYTES + boff[ks][0][i]);
                            const u32x2 hi = lds_read_tr<I8>(st + b * CF::B_BYTES + boff[ks][1][i]);
                            bf[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
                        }
#pragma unroll
                        for (int i = 0; i < FN; ++i)
#pragma unroll
                            for (int j = 0; j < FM; ++j)
                                acc[b][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                    bitcast<f16x8>(bf[i]), bitcast<f16x8>(af[j]), acc[b][i][j], 0, 0, 0);
                    }
                }
            }
        }
    } else {
        constexpr int P = CF::P;
        const unsigned a_end = (unsigned)M * K * ES, b_end = (unsigned)K * N * ES;  // bytes of A, of B
        unsigned ua[CF::DA], ub[CF::DB];  // this lane's chunks of K tile 0
#pragma unroll
        for (int i = 0; i < CF::DA; ++i) ua[i] = ua_chunk_a<CF>(m0, wave * CF::DA + i, lane, M, K);
#pragma unroll
        for (int i = 0; i < CF::DB; ++i) ub[i] = ua_chunk_b<CF>(n0, wave * CF::DB + i, lane, N);
        u32x4 rg[P][D];
        // a K tile whose every chunk lies inside (ua_whole_tiles)
        auto load_fast = [&](u32x4 (&r)[D], int t) {
            const int k0 = kbeg + t * BK;
            const unsigned char* at = Ab + (int64_t)k0 * ES;
            const unsigned char* bt = Bb + (int64_t)k0 * N * ES;
#pragma unroll
            for (int i = 0; i < CF::DA; ++i) r[i] = load_any16(at + ua[i]);
#pragma unroll
            for (int i = 0; i < CF::DB; ++i) r[CF::DA + i] = load_any16(bt + ub[i]);
        };
        auto load_careful = [&](u32x4 (&r)[D], int t) {
            const int k0 = kbeg + t * BK;
#pragma unroll
            for (int i = 0; i < CF::DA; ++i) {
                const unsigned off = ua[i] + (unsigned)k0 * ES, at = ua_inside(off, a_end);
                r[i] = keep_bytes(shift_bytes(load_any16(Ab + at), off - at), ua_keep_a<CF>(k0, lane, K));
            }
#pragma unroll
            for (int i = 0; i < CF::DB; ++i) {
                const unsigned off = ub[i] + (unsigned)k0 * N * ES, at = ua_inside(off, b_end);
                r[CF::DA + i] = shift_bytes(load_any16(Bb + at), off - at);  // (zero from the end on)
            }
        };
        auto put = [&](const u32x4 (&r)[D], int t) {
            const unsigned st = lds0 + (unsigned)((t & 1) * SB) + 16 * lane;
#pragma unroll
            for (int i = 0; i < CF::DA; ++i)
                *reinterpret_cast<lds_u32x4*>((size_t)(st + (wave * CF::DA + i) * 1024)) = r[i];
#pragma unroll
            for (int i = 0; i < CF::DB; ++i)
                *reinterpret_cast<lds_u32x4*>((size_t)(st + CF::A_BYTES + (wave * CF::DB + i) * 1024)) = r[CF::DA + i];
        };
        // One barrier per K tile: a wave that writes stage t % 2 again has passed
        // barrier t + 1, and every wave reached that one with its reads of tile t
        // complete.  The steady loop's loads are unconditional, so that the wait
        // before a tile's LDS writes leaves the P - 1 later tiles in flight.
        const int whole = ua_whole_tiles<CF>(kbeg, nkt, K);
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (u < nkt) load_careful(rg[u], u);
        int t = 0;
#pragma unroll 1
        for (; ua_steady<CF>(t, whole); t += P) {
#pragma unroll
            for (int u = 0; u < P; ++u) {
                put(rg[u], t + u);
                load_fast(rg[u], t + u + P);
                lds_barrier();
                compute(lds0 + (unsigned)(((t + u) & 1) * SB), kbeg + (t + u) * BK);
            }
        }
#pragma unroll 1
        for (; t < nkt; t += P) {
#pragma unroll
            for (int u = 0; u < P; ++u) {
                if (t + u < nkt) {
                    put(rg[u], t + u);
                    if (t + u + P < nkt) load_careful(rg[u], t + u + P);
                    lds_barrier();
                    compute(lds0 + (unsigned)(((t + u) & 1) * SB), kbeg + (t + u) * BK);
                }
            }
        }
        if (CF::KW > 1 || p.nsplit > 1) __syncthreads();  // (LDS is used again below)
    }

    // ---- zero points: the split's correction (both lane halves added, column
    // sums passed from the lane that holds a column to those that need it) ----
    if constexpr (ZP) {
        const unsigned za = (unsigned)p.za, zb = (unsigned)p.zb;
        const unsigned kzz = (unsigned)(min(K, kbeg + p.kps) - kbeg) * za * zb + (split == 0 ? (unsigned)p.acc_add : 0u);
        unsigned rcorr[FM];
#pragma unroll
        for (int j = 0; j < FM; ++j) rcorr[j] = kzz - zb * (unsigned)halves_sum2(rsum[j], rsum[j]);
#pragma unroll
        for (int i = 0; i < FN; ++i) {
            const int cs = halves_sum2(csum[i], csum[i]);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int src = 8 * (v >> 2) + 4 * kh + (v & 3);  // lane of this register's column
                const unsigned cc = p.za != 0 ? za * (unsigned)__builtin_amdgcn_ds_bpermute(4 * src, cs) : 0u;
#pragma unroll
                for (int j = 0; j < FM; ++j) acc[0][i][j][v] = (int)((unsigned)acc[0][i][j][v] + rcorr[j] - cc);
            }
        }
    }

    // ---- k slices: every wave stores its sums to LDS; wave kw then owns the
    // runs q with q / (4 / KW) == kw of every block and adds the KW slices in
    // slice order ----
    constexpr int NQ = 4 / CF::KW;  // runs of 4 columns per block owned by a wave
    if constexpr (CF::KW > 1) {
        const unsigned red = lds0 + (unsigned)((UA ? 2 : S) * SB);
        // wave tile wmn, slice s, block (b, i, j), run q: 1 KB, 16 lane-contiguous
        // bytes per lane
        auto slot = [&](int s, int b, int i, int j, int q) {
            return red +
                   (unsigned)(((((((wmn * CF::KW + s) * NB + b) * FN + i) * FM + j) * 4 + q) << 10) + 16 * lane);
        };
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<lds_u32x4*>((size_t)slot(kw, b, i, j, q)) = bitcast<u32x4>(
                            f32x4{acc[b][i][j][4 * q], acc[b][i][j][4 * q + 1], acc[b][i][j][4 * q + 2],
                                  acc[b][i][j][4 * q + 3]});
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (q / NQ != kw) continue;
                        f32x4 sum = bitcast<f32x4>(lds_read16(slot(0, b, i, j, q)));
#pragma unroll
                        for (int s = 1; s < CF::KW; ++s) {
                            const f32x4 v = bitcast<f32x4>(lds_read16(slot(s, b, i, j, q)));
                            sum = f32x4{sum[0] + v[0], sum[1] + v[1], sum[2] + v[2], sum[3] + v[3]};
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[b][i][j][4 * q + e] = sum[e];
                    }
    }

    // ---- split-K (with k slices: of the runs a wave owns) ----
    if (CF::KW < 4 && p.nsplit > 1) {
        constexpr int NC = NB * FN * FM * NQ;
        f32x4 v[NC];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (CF::KW > 1 && q / NQ != kw) continue;
                        v[((b * FN + i) * FM + j) * NQ + q % NQ] = bitcast<f32x4>(
                            AccT4{acc[b][i][j][4 * q], acc[b][i][j][4 * q + 1], acc[b][i][j][4 * q + 2],
                                  acc[b][i][j][4 * q + 3]});
                    }
        float* slabs = p.part + (size_t)tile * p.nsplit * NC * CF::NT * 4;
        splitk_publish<NC, CF::NT>(slabs + (size_t)split * NC * CF::NT * 4, tid, v);
        if (!splitk_arrive_is_last(p.counters + tile, (unsigned)p.nsplit, reinterpret_cast<int*>(smem)))
            return;
        splitk_reduce<NC, CF::NT, I8>(slabs, p.nsplit, split, tid, v);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (CF::KW > 1 && q / NQ != kw) continue;
                        const AccT4 w = bitcast<AccT4>(v[((b * FN + i) * FM + j) * NQ + q % NQ]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[b][i][j][4 * q + e] = w[e];
                    }
    }

    // ---- epilogue: lane row m, runs of 4 columns ----
    // Everything the epilogue reads (row / column scales, C for beta) is
    // loaded before the first store, from clamped addresses: a load issued
    // after a store to memory the compiler cannot tell apart waits for it, one
    // round trip per run of 4 columns.
    unsigned char* Cb = static_cast<unsigned char*>(p.C) + batch * p.sC * (OUT == kI8Acc32 ? 4 : 2);
    float sav[FM];
    float sbv[FN][4][4];
    u32x2 oldc[FM][FN][4];
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int mc = min(m0 + wm * 32 * FM + 32 * j + l32, M - 1);
        sav[j] = 1.0f;
        if constexpr (OUT == kI8RowCol) sav[j] = h2f(p.sa[mc]);
        if constexpr (OUT == kF16AlphaBeta) {
            if (p.beta != 0.0f) {
#pragma unroll
                for (int i = 0; i < FN; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (CF::KW > 1 && q / NQ != kw) continue;
                        const int n = n0 + wn * 32 * FN + 32 * i + 8 * q + 4 * kh;
                        const int nc = min(n, N - 4);
                        const uint16_t* src = reinterpret_cast<const uint16_t*>(Cb) + (int64_t)mc * N + nc;
                        if constexpr (UA) {
                            // (a run cut by N: the row's last four, shifted into place)
                            const u32x2 c = *reinterpret_cast<const u32x2u*>(src);
                            const uint64_t w = ((uint64_t)c.y << 32 | c.x) >> (16 * min(n - nc, 3));
                            oldc[j][i][q] = u32x2{(unsigned)w, (unsigned)(w >> 32)};
                        } else {
                            oldc[j][i][q] = *reinterpret_cast<const u32x2*>(src);
                        }
                    }
            }
        }
    }
    if constexpr (OUT == kI8RowCol) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wn * 32 * FN + 32 * i + 8 * q + 4 * kh;
#pragma unroll
                for (int e = 0; e < 4; ++e) sbv[i][q][e] = h2f(p.sb[min(n + e, N - 1)]);
            }
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int m = m0 + wm * 32 * FM + 32 * j + l32;
        if (m >= M) continue;
        const float sa = sav[j];
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (CF::KW > 1 && q / NQ != kw) continue;
                const int n = n0 + wn * 32 * FN + 32 * i + 8 * q + 4 * kh;
                if (n >= N) continue;  // aligned: N % 8 == 0, the run is whole
                if constexpr (OUT == kI8Acc32) {
                    int* dst = reinterpret_cast<int*>(Cb) + (int64_t)m * N + n;
                    if constexpr (UA) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < N) dst[e] = acc[0][i][j][4 * q + e];
                    } else {
                        *reinterpret_cast<i32x4*>(dst) = i32x4{acc[0][i][j][4 * q], acc[0][i][j][4 * q + 1],
                                                               acc[0][i][j][4 * q + 2], acc[0][i][j][4 * q + 3]};
                    }
                } else {
                    uint16_t* dst = reinterpret_cast<uint16_t*>(Cb) + (int64_t)m * N + n;
                    float r[4];
                    if constexpr (OUT == kF16AlphaBeta) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) r[e] = p.alpha * acc[0][i][j][4 * q + e];
                        if (p.beta != 0.0f) {
                            const u32x2 c = oldc[j][i][q];
                            r[0] = fmaf(p.beta, h2f(c.x & 0xffffu), r[0]);
                            r[1] = fmaf(p.beta, h2f(c.x >> 16), r[1]);
                            r[2] = fmaf(p.beta, h2f(c.y & 0xffffu), r[2]);
                            r[3] = fmaf(p.beta, h2f(c.y >> 16), r[3]);
                        }
                    } else if constexpr (OUT == kF16SwiGLU) {
                        // gate and up rounded to fp16 as two GEMM outputs would be
                        const uint16_t o0 = swiglu_h(f2h(acc[0][i][j][4 * q]), f2h(acc[NB - 1][i][j][4 * q]));
                        const uint16_t o1 = swiglu_h(f2h(acc[0][i][j][4 * q + 1]), f2h(acc[NB - 1][i][j][4 * q + 1]));
                        const uint16_t o2 = swiglu_h(f2h(acc[0][i][j][4 * q + 2]), f2h(acc[NB - 1][i][j][4 * q + 2]));
                        const uint16_t o3 = swiglu_h(f2h(acc[0][i][j][4 * q + 3]), f2h(acc[NB - 1][i][j][4 * q + 3]));
                        *reinterpret_cast<u32x2*>(dst) = u32x2{(unsigned)o0 | ((unsigned)o1 << 16),
                                                               (unsigned)o2 | ((unsigned)o3 << 16)};
                        continue;
                    } else if constexpr (OUT == kI8Tensor) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) r[e] = static_cast<float>(acc[0][i][j][4 * q + e]) * p.scale;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) r[e] = static_cast<float>(acc[0][i][j][4 * q + e]) * (sa * sbv[i][q][e]);
                    }
                    const u32x2 w = {pack2h(r[0], r[1]), pack2h(r[2], r[3])};
                    if constexpr (UA) {
                        if (n + 4 <= N) {
                            *reinterpret_cast<u32x2u*>(dst) = w;
                        } else {
#pragma unroll
                            for (int e = 0; e < 3; ++e)
                                if (n + e < N) dst[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
                        }
                    } else {
                        *reinterpret_cast<u32x2*>(dst) = w;
                    }
                }
            }
    }
}

}  // namespace sk
}  // namespace clove
