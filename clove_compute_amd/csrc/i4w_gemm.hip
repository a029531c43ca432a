// Host side of the INT4-weight MFMA GEMM (i4w_gemm.hpp): tile configuration,
// split-K plan, scratch, and the B transpose of group-wise INT4.
#include "dispatch.hpp"
#include "i4w_gemm.hpp"
#include "i4w_stream.hpp"

namespace clove {
namespace {

using namespace i4w;

// (WR, WC, FW, FX, stages): waves along weight rows x along X rows, 32x32
// tiles per wave in each direction
using CfgBig = Cfg<4, 1, 2, 4, 3>;  // 256 x 128, 4 waves of 64 x 128
// 128 x 64, one stage ahead (50 KB LDS: two workgroups per CU).  The
// prefill GEMMs are bound by the VALU and MFMA issue, not by their loads: a
// second stage in flight only made every workgroup's first stage wait behind
// a larger burst of the grid's prologue loads (W4A16 Llama-1B layer T = 512
// 125.6 -> 122.9 us, fused 114.9 -> 111.1 us against three stages)
using CfgC64 = Cfg<4, 1, 1, 2, 2>;
// the same with two stages ahead (75 KB), where the grid leaves a CU one
// workgroup: nothing else then covers a stage's round trip (W4A16, three
// operand sets in turn, T = 140 on 3328 x 7424 25.3 -> 23.0 us, 187 on 1920 x 11008
// 27.2 -> 23.4)
using CfgC64S3 = Cfg<4, 1, 1, 2, 3>;
// 128 x 32, three stages ahead (70 KB LDS: two workgroups per CU): few X rows
// or few tiles, where a workgroup's chain of stages is the time
using CfgC32 = Cfg<4, 1, 1, 1, 4>;
// 64 x 32, two waves, for few tiles over a long K: half the partial tile that the
// last workgroup of a tile adds up from every split
using CfgC32H = Cfg<2, 1, 1, 1, 4>;
// 256 x 64 (four waves of 64 x 64), one stage ahead (70 KB LDS: two workgroups
// per CU): the fused gate/up + SwiGLU from 512 X rows up, where each wave's two
// weight blocks (a gate and an up block per 32 outputs) share every X
// fragment it reads.  Measured against 128 x 64 / 256 x 128 on the Llama-1B
// and -7B MLPs (I x K = 8192 x 2048, 11008 x 4096; graph replays, cold
// weights), T = 512 (alternating blocks): 47.0-48.0 -> 45.0-45.2 and
// 119.3-119.8 -> 116.6-117.2 us, T = 1024: 94.8 -> 85.9 and 224.6 -> 217.2,
// T = 2048: 184.2 -> 166.2 and 470.8 -> 420.1; at T <= 256 it loses (T = 64:
// 14.6 -> 19.3)
using CfgS64 = Cfg<4, 1, 2, 2, 2>;
// 256 x 128 with eight waves of 64 x 64 (two per SIMD), one stage ahead
// (100 KB LDS, one workgroup per CU): the fused gate/up + SwiGLU once these
// tiles alone cover 3/4 of the CUs (never split: the kernel has no split-K
// path for eight waves).  Llama-1B MLP T = 512 (I x K = 8192 x 2048, graph-free
// timing of 30 calls, cold weights): 48.6 us with 256 x 64 -> 40.6 us; with
// two stages ahead 42.4.  The one-projection shapes measured slower on it
// (they need split K at T = 512)
using CfgS128 = Cfg<4, 2, 2, 2, 2>;

inline size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

struct Plan {
    int tiles_r, tiles_c, nsplit, gps;
};

// No split when the tiles cover 3/4 of the CUs; otherwise split K (whole
// groups, at least min_groups per split) until the grid reaches `target`
// workgroups (the number that can be resident at once).
template <class CF>
Plan make_plan(int R, int C, int G, int cus, int target, int min_groups) {
    Plan pl;
    pl.tiles_r = cdiv(R, CF::BR);
    pl.tiles_c = cdiv(C, CF::BC);
    const int tiles = pl.tiles_r * pl.tiles_c;
    int ns = 4 * tiles >= 3 * cus || CF::NW == 8 ? 1 : target / tiles;
    ns = max(1, min(ns, G / min_groups));
    pl.gps = cdiv(G, ns);
    pl.nsplit = cdiv(G, pl.gps);
    return pl;
}

// `prep(args, extra)` runs before the GEMM with `extra_bytes` of scratch
// (after the split-K partials) and may point args.X / args.xs into it.
// Where scratch is short: with `other` (the caller has another kernel, which
// needs none) the status says so; else short K, and grids that cover 3/8 of the
// CUs with 128-row tiles of few columns, run unsplit.
template <class CF, bool XS, int OUT, class Prep>
clove_status_t run(Args a, int cus, int target, int min_groups, size_t extra_bytes, hipStream_t stream,
                   Prep prep, bool other) {
    // OUT 2 (SwiGLU): a tile of BR weight rows makes BR/2 outputs
    const Plan pl = make_plan<CF>(OUT == 2 ? 2 * a.R : a.R, a.C, a.G, cus, target, min_groups);
    a.tiles_r = pl.tiles_r;
    a.tiles_c = pl.tiles_c;
    a.nsplit = pl.nsplit;
    a.gps = pl.gps;
    const int tiles = pl.tiles_r * pl.tiles_c;
    const size_t part_bytes =
        pl.nsplit > 1 ? round256((size_t)tiles * pl.nsplit * CF::NT * CF::FW * CF::FX * 16 * sizeof(float)) : 0;
    char* extra = nullptr;
    if (part_bytes + extra_bytes > 0) {
        Scratch s;
        const bool unsplit = extra_bytes == 0 && !other &&
                             (a.C <= 32 ? a.G < 20 || 4 * cdiv(OUT == 2 ? 2 * a.R : a.R, 64) >= 3 * cus : a.G < 16);
        const clove_status_t st =
            acquire_scratch(stream, part_bytes + extra_bytes, (size_t)tiles, &s, unsplit || other);
        if (unsplit && scratch_short(st)) {
            a.nsplit = 1;
            a.gps = a.G;
        } else if (st != CLOVE_OK) {
            return st;
        }
        a.part = s.partials;
        a.counters = s.counters;
        extra = reinterpret_cast<char*>(s.partials) + part_bytes;
    }
    const clove_status_t st = prep(a, extra);
    if (st != CLOVE_OK) return st;
    auto k = i4w_gemm<CF, XS, OUT>;
    constexpr int lds = CF::template lds_bytes<XS>();
    static_assert(lds <= 160 * 1024, "LDS");
    if (ensure_lds(reinterpret_cast<const void*>(k), lds) != CLOVE_OK)
        return CLOVE_ERR_LAUNCH;
    CLOVE_LAUNCH(k, dim3((unsigned)(tiles * a.nsplit)), dim3(CF::NT), lds, stream, a);
    return check_launch();
}

// Tile choice by the number of X rows C (us per call, 500 W4A16 and INT4 shapes,
// weights that rotate past the Infinity Cache unless three sets are named):
//   128 x 32 for C <= 32, and while these tiles fit the CUs once and tiles x
//   groups stay under 12 a CU (16 up to 20 groups), where a stage's latency and not
//   its MFMAs is the time (against 128 x 64, three sets: W4A16 T = 64 on 3072 x 2048
//   11.2 -> 8.0, 100 on 2432 x 1920 13.9 -> 9.3, 427 on 1920 x 1536 12.7 -> 10.2; INT4
//   1216 x 55 x 2560 18.7 -> 12.6; the fused SwiGLU of 63 on 6144 x 1920, 11 a CU, 17.6
//   -> 12.4; T = 397 on 2304 x 2176, 15, 14.7 -> 13.1; past it INT4 8320 x 43 x 3584, 14,
//   21.4 -> 26.3, W4A16 T = 45 on 5888 x 4480, 13, 14.6 -> 16.0).  For C <= 32 it
//   replaced 64 x 32 tiles of two waves (fused SwiGLU 22016 x 4096 T = 16 26.0 ->
//   19.6), which stay for few tiles over 40 groups or more (W4A16 T = 26 on 1536 x
//   10368 13.9 -> 11.8, INT4 1600 x 16 x 12416 18.5 -> 16.9; 2944 x 7808, 23 tiles x 61
//   groups, 13.2 -> 15.4)
//   128 x 64 with two stages ahead while those tiles cover less than 1/3 of the
//   CUs, split to one workgroup per CU (with two splits some CUs have none: 158 on
//   3840 x 5632, 90 tiles, 22.0 -> 23.7, INT4 11456 x 36 x 12672 50.0 -> 54.2)
//   otherwise 128 x 64 with two workgroups per CU, whose waves interleave
//   VALU (unpack, fold) with MFMA -- ahead of 128 x 128 by 15-25 % on the
//   INT4 N = 128 and W4A16 T = 512 shapes -- unless 256 x 128 tiles already
//   cover the CUs (large prefill); the fused SwiGLU from 512 X rows up: 256 x
//   128 with eight waves where those tiles cover 3/4 of the CUs, else 256 x 64
// Splits keep at least 4 groups each (8 where two workgroups share a CU).
template <bool XS, int OUT, class Prep>
clove_status_t by_shape(const Args& a, int cus, size_t extra_bytes, hipStream_t stream, Prep prep, bool other = false) {
    const int rows = OUT == 2 ? 2 * a.R : a.R;  // weight rows
    const int64_t t32 = (int64_t)cdiv(rows, CfgC32::BR) * cdiv(a.C, CfgC32::BC);
    if constexpr (OUT != 2) {
        if (a.C <= 32 && a.G >= 40 && 10 * t32 <= cus && t32 * a.G <= 5 * cus)
            return run<CfgC32H, XS, OUT>(a, cus, 3 * cus, 10, extra_bytes, stream, prep, other);
    }
    if (a.C <= 32 || (t32 <= cus && t32 * a.G <= (a.G <= 20 ? 16 : 12) * cus))
        return run<CfgC32, XS, OUT>(a, cus, cus, a.G > 44 ? 8 : 4, extra_bytes, stream, prep, other);
    if (3 * (int64_t)cdiv(rows, CfgC64::BR) * cdiv(a.C, CfgC64::BC) < cus)
        return run<CfgC64S3, XS, OUT>(a, cus, cus, 4, extra_bytes, stream, prep, other);
    if (OUT == 2 && a.C >= 512) {
        if (4 * cdiv(rows, CfgS128::BR) * cdiv(a.C, CfgS128::BC) >= 3 * cus)
            return run<CfgS128, XS, OUT>(a, cus, cus, 8, extra_bytes, stream, prep, other);
        return run<CfgS64, XS, OUT>(a, cus, 2 * cus, 8, extra_bytes, stream, prep, other);
    }
    // (SwiGLU tiles pair gate and up rows: the same outputs take twice the
    // weight rows, so the big tile waits for twice the grid)
    if (cdiv(rows, CfgBig::BR) * cdiv(a.C, CfgBig::BC) >= (OUT == 2 ? 2 : 1) * cus)
        return run<CfgBig, XS, OUT>(a, cus, cus, 8, extra_bytes, stream, prep, other);
    return run<CfgC64, XS, OUT>(a, cus, 2 * cus, 8, extra_bytes, stream, prep, other);
}

bool fits31(int64_t bytes) { return bytes < ((int64_t)1 << 31); }

// ---- the streaming kernel (i4w_stream.hpp) for C <= 32 X rows ----
template <int WF, int XF, int NG, int KS, bool XS, int OUT, int RAWB>
clove_status_t launch_stream(const Args& a, hipStream_t stream) {
    using SC = SCfg<WF, XF, NG, KS>;
    const int lds = SC::lds_bytes(a.G, XS, RAWB);
    auto k = i4w_stream<SC, XS, OUT, RAWB>;
    if (ensure_lds(reinterpret_cast<const void*>(k), lds) != CLOVE_OK)
        return CLOVE_ERR_LAUNCH;
    CLOVE_LAUNCH(k, dim3((unsigned)cdiv(a.R, SC::ROWS)), dim3(SC::NT), lds, stream, a);
    return check_launch();
}

// K slices: 4 or 8 waves of at most 11 groups.  Short slices: a wave's chain
// of groups is most of a small product's time (us per call, against the
// fewest waves that hold K: W4A16 T = 13 on 8128 x 1280 6.9 -> 5.2, INT4 N =
// 12 on 10496 x 1152 7.5 -> 5.8, N = 19 on 1984 x 1920 7.2 -> 5.4, N = 9 on
// 3840 x 5760 9.0 -> 7.6; three operand sets).  For 17..32 groups INT4 takes 8
// waves (N = 27 on 7552 x 2304 9.2 -> 8.5 against 4), but 4 past 24 groups with
// three weight fragments, whose eight waves' partial sums fill the LDS of a CU
// (N = 16 on 11008 x 4096 8.7 against 9.0 us); W4A16 4 (T = 19 on 3712 x 3584 the
// same; four waves leave room for more workgroups), or 2 of 11 groups up to 22
// from 8 tokens on in one round of the CUs (T = 12 on 1664 x 2560 5.15 against
// 5.45, 20 on 3840 x 2304 6.8 against 7.3); 33..44 groups stay on 4 (INT4 N = 12 on
// 11840 x 4864 12.4 against 13.5).
// (BIG_G = false: the caller never passes more than 64 groups, and the
// 11-group, 8-slice variant is not instantiated)
template <int WF, int XF, bool XS, int OUT, int RAWB = 0, bool BIG_G = true>
clove_status_t stream_by_k(const Args& a, hipStream_t stream) {
    const int G = a.G;
    if (G <= 12) return launch_stream<WF, XF, 3, 4, XS, OUT, RAWB>(a, stream);
    if (G <= 16) return launch_stream<WF, XF, 4, 4, XS, OUT, RAWB>(a, stream);
    if constexpr (XS) {
        if (G <= 24) return launch_stream<WF, XF, 3, 8, XS, OUT, RAWB>(a, stream);
        if constexpr (WF == 3) {
            if (G <= 32) return launch_stream<WF, XF, 8, 4, XS, OUT, RAWB>(a, stream);
        } else {
            if (G <= 32) return launch_stream<WF, XF, 4, 8, XS, OUT, RAWB>(a, stream);
        }
    } else {
        if constexpr (WF == 1) {
            if (G > 16 && G <= 22 && a.C >= 8) return launch_stream<WF, XF, 11, 2, XS, OUT, RAWB>(a, stream);
        }
        if (G <= 24) return launch_stream<WF, XF, 6, 4, XS, OUT, RAWB>(a, stream);
        if (G <= 32) return launch_stream<WF, XF, 8, 4, XS, OUT, RAWB>(a, stream);
    }
    if (G <= 44) return launch_stream<WF, XF, 11, 4, XS, OUT, RAWB>(a, stream);
    if constexpr (!(XS && XF == 2)) {  // (kRawB2MaxGroups)
        if (G <= 48) return launch_stream<WF, XF, 6, 8, XS, OUT, RAWB>(a, stream);
        if (!BIG_G || G <= 64) return launch_stream<WF, XF, 8, 8, XS, OUT, RAWB>(a, stream);
        if constexpr (BIG_G) return launch_stream<WF, XF, 11, 8, XS, OUT, RAWB>(a, stream);
    }
    return CLOVE_ERR_INVALID_ARG;
}

constexpr int kStreamMaxGroups = 88;  // K <= 11264

// Two weight fragments (32 rows) per workgroup once one fragment each would
// take a second round of the CUs (X is then read half as often; W4A16 T = 10
// on 5184 x 5248 11.5 -> 9.6 us, 14 on 13184 x 1280 8.9 -> 7.3).
// Two X fragments with two weight fragments and 11-group slices (K > 8192)
// need more registers than a lane has: those take one weight fragment.
bool stream_two_rows(const Args& a, int cus) { return cdiv(a.R, 16) > cus && (a.C <= 16 || a.G <= 64); }

clove_status_t run_stream(const Args& a, int cus, hipStream_t stream) {
    const bool wf2 = stream_two_rows(a, cus);
    if (a.C <= 16) return wf2 ? stream_by_k<2, 1, false, 1>(a, stream) : stream_by_k<1, 1, false, 1>(a, stream);
    if (wf2) return stream_by_k<2, 2, false, 1, 0, false>(a, stream);
    return stream_by_k<1, 2, false, 1>(a, stream);
}

// Every workgroup of the streaming kernel reads all of X (C rows x K fp16),
// so its cost grows with C x K per CU, while the split-K MFMA kernel reads
// each X tile once per 128 weight rows and is flat in C.  Measured (W4A16, 90
// shapes, T = 2..32, O 1024..11008, K 1024..11008; us per call, three operand sets
// in turn, which the Infinity Cache holds, stream against 128 x 32 tiles): up to 16 rows the stream is ahead below ~200 KB of
// X per CU, counting one copy per round of workgroups on a CU (T = 13 on 2048
// x 7424, 188 KB, 10.5 against 11.1; 2176 x 8704, 221 KB, 13.6 against 11.9);
// with two X fragments below ~128 KB and in one round (T = 24 on 2944 x 1664
// 5.7 against 7.4; T = 32 on 4864 x 2304, 144 KB, 10.4 against 8.1; T = 20 on
// 9216 x 1152, 90 KB in two rounds, 9.2 against 7.3).
int stream_rounds(const Args& a, int cus) { return cdiv(cdiv(a.R, stream_two_rows(a, cus) ? 32 : 16), cus); }
int64_t stream_bytes(const Args& a, int cus) { return (int64_t)a.C * a.K * 2 * stream_rounds(a, cus); }

bool stream_ahead(const Args& a, int cus) {
    const int64_t bytes = stream_bytes(a, cus);
    return a.C <= 16 ? bytes < 200 * 1024 : stream_rounds(a, cus) == 1 && bytes < 128 * 1024;
}

}  // namespace

bool try_i4w_w4a16(const W4A16Args& w, int cus, hipStream_t stream, clove_status_t* status) {
    // three or four tokens: the streaming kernel rather than the GEMV (three operand
    // sets in turn, T = 4: 4096x11008 12.1 against 22.0 us, 2176x2176 4.3 against 6.7, 1024 x
    // 1664 3.7 against 4.0; at T = 2 neither is ahead throughout)
    if (w.T <= 2 || w.K <= 0 || w.K % 128 != 0 || !aligned16(w.X) || !aligned16(w.W)) return false;
    if (!fits31((int64_t)w.T * w.K * 2) || !fits31((int64_t)w.O * (w.K / 2))) return false;
    Args a{};
    a.W = w.W;
    a.wscale = w.scale;
    a.wzero = w.zero;
    a.X = w.X;
    a.out = w.Y;
    a.R = w.O;
    a.C = w.T;
    a.K = w.K;
    a.G = w.K / 128;
    a.alpha = w.alpha;
    a.beta = w.beta;
    const bool streams = w.T <= 32 && a.G <= kStreamMaxGroups;
    if (streams && stream_ahead(a, cus)) {
        *status = run_stream(a, cus, stream);
        return true;
    }
    if (w.T <= 4) return false;  // (the GEMV, outside the stream's domain)
    // without scratch for the K split, the stream while it reads up to 256 KB of X
    // per CU (at most 1.4 times the split tiles' time there)
    const bool other = streams && stream_bytes(a, cus) < 256 * 1024;
    *status = by_shape<false, 1>(a, cus, 0, stream, [](Args&, char*) { return CLOVE_OK; }, other);
    if (other && scratch_short(*status)) *status = run_stream(a, cus, stream);
    return true;
}

bool try_i4w_w4a16_swiglu(const W4A16Args& w, int cus, hipStream_t stream, clove_status_t* status) {
    if (w.T <= 2 || w.K <= 0 || w.K % 128 != 0 || !aligned16(w.X) || !aligned16(w.W)) return false;
    if (!fits31((int64_t)w.T * w.K * 2) || !fits31((int64_t)2 * w.O * (w.K / 2))) return false;
    Args a{};
    a.W = w.W;
    a.wscale = w.scale;
    a.wzero = w.zero;
    a.X = w.X;
    a.out = w.Y;
    a.R = w.O;  // outputs; the weight has 2 O rows (gate, then up)
    a.C = w.T;
    a.K = w.K;
    a.G = w.K / 128;
    a.alpha = 1.0f;
    a.beta = 0.0f;
    // (up to four tokens the caller has its GEMV)
    *status = by_shape<false, 2>(a, cus, 0, stream, [](Args&, char*) { return CLOVE_OK; }, w.T <= 4);
    return true;
}

// (raw B with two column fragments: K <= 5632, 88 KB of B in LDS)
constexpr int kRawB2MaxGroups = 44;

bool try_i4w_int4(const Int4Args& q, int cus, hipStream_t stream, clove_status_t* status) {
    if (q.mode != CLOVE_INT4_GROUPWISE || q.N <= 8 || q.K <= 0 || q.K % 128 != 0 || !aligned16(q.A))
        return false;
    const int Npad = (q.N + 63) / 64 * 64;
    const int G = q.K / 128;
    if (!fits31((int64_t)Npad * q.K * 2) || !fits31((int64_t)q.M * (q.K / 2))) return false;
    const size_t xt_bytes = round256((size_t)Npad * q.K * 2);
    const size_t xs_bytes = round256((size_t)G * Npad * 4);
    Args a{};
    a.W = q.A;
    a.wscale = q.A_scale;
    a.wzero = q.A_zero;
    a.out = q.C;
    a.R = q.M;
    a.C = q.N;
    a.K = q.K;
    a.G = G;
    a.ldxs = Npad;
    a.alpha = 1.0f;
    a.beta = 0.0f;
    const int ldb = (q.N + 1) / 2;
    auto prep = [&](Args& args, char* extra) -> clove_status_t {
        uint16_t* xt = reinterpret_cast<uint16_t*>(extra);
        float* xs = reinterpret_cast<float*>(extra + xt_bytes);
        CLOVE_LAUNCH(i4w_prep_b, dim3((unsigned)G, (unsigned)cdiv(Npad, 128)), dim3(256), 0, stream, q.B,
                           ldb, q.B_scale, q.B_zero, q.N, q.K, G, Npad, xt, xs);
        args.X = xt;
        args.xs = xs;
        return check_launch();
    };
    *status = by_shape<true, 0>(a, cus, xt_bytes + xs_bytes, stream, prep);
    return true;
}

// Weight rows per workgroup of the raw-B stream, 16 WF (WF = 1..3): the fewest
// rows on the busiest CU, counting whole rounds of workgroups; on a tie the
// larger workgroups when each has four or more K-slice waves (G > 16), else
// the smaller.  Cold graph replays, us per call for WF = 1 / 2 / 3 (N = 16):
// 11008 x 4096 9.57 / 11.23 / 9.09, 11008 x 8192 19.73 / 20.62 / 15.90,
// 8192 x 4096 7.58 / 7.30 / 8.66, 16384 x 4096 12.06 / 11.17 / 14.40,
// 4096 x 4096 5.52 / 6.87 / 8.29, 14336 x 2048 7.48 / 9.15 / 11.13, 11008 x
// 2048 7.17 / 8.98 / 7.81: the rule picks the fastest of the three in each.
// (most: two with two column fragments, whose accumulators take the registers;
// WF = 1 / 2 at N = 23: 8384 x 2944 11.2 / 13.8, 10816 x 3456 N = 25 15.1 / 18.4)
int rawb_wf(int R, int G, int cus, int most) {
    int best = 1;
    int64_t best_rows = -1;
    for (int wf = 1; wf <= most; ++wf) {
        const int64_t rows = (int64_t)cdiv(cdiv(R, 16 * wf), cus) * wf;
        if (best_rows < 0 || rows < best_rows || (rows == best_rows && G > 16)) {
            best = wf;
            best_rows = rows;
        }
    }
    return best;
}

bool try_i4w_int4_rawb(const Int4Args& q, int cus, hipStream_t stream, clove_status_t* status) {
    // up to 32 columns: B rows of at most 16 bytes, read in place (no transpose pass)
    const int G = q.K / 128;
    if (q.mode != CLOVE_INT4_GROUPWISE || q.N < 5 || q.N > 32 || q.K <= 0 || q.K % 128 != 0 || !aligned16(q.A) ||
        !fits31((int64_t)q.M * (q.K / 2)))
        return false;
    // (B and its constants stay in LDS whole; two column fragments past 32 groups
    // only in one round of 32-row workgroups: 8256 x 20 x 4352 24.2 against 19.0 us on
    // the 128 x 32 tiles, 9856 x 22 x 4224 25.7 against 19.3; 7232 x 18 x 4608 13.7 against
    // 18.1)
    if (G > (q.N <= 16 ? kStreamMaxGroups : kRawB2MaxGroups)) return false;
    if (q.N > 16 && G > 32 && cdiv(q.M, 32) > cus) return false;
    Args a{};
    a.W = q.A;
    a.wscale = q.A_scale;
    a.wzero = q.A_zero;
    a.out = q.C;
    a.R = q.M;
    a.C = q.N;
    a.K = q.K;
    a.G = G;
    a.B = q.B;
    a.bscale = q.B_scale;
    a.bzero = q.B_zero;
    a.N = q.N;
    a.ldb = (q.N + 1) / 2;
    a.alpha = 1.0f;
    a.beta = 0.0f;
    const int wf = rawb_wf(a.R, G, cus, q.N > 16 ? 2 : 3);
    if (q.N > 16) {
        *status = wf == 2 ? stream_by_k<2, 2, true, 0, 2, false>(a, stream) : stream_by_k<1, 2, true, 0, 2, false>(a, stream);
        return true;
    }
    if (a.ldb == 8 && aligned16(q.B))
        *status = wf == 3   ? stream_by_k<3, 1, true, 0, 1>(a, stream)
                  : wf == 2 ? stream_by_k<2, 1, true, 0, 1>(a, stream)
                            : stream_by_k<1, 1, true, 0, 1>(a, stream);
    else
        *status = wf == 3   ? stream_by_k<3, 1, true, 0, 2>(a, stream)
                  : wf == 2 ? stream_by_k<2, 1, true, 0, 2>(a, stream)
                            : stream_by_k<1, 1, true, 0, 2>(a, stream);
    return true;
}

}  // namespace clove
