// Host side of the skinny GEMM (skinny_gemm.hpp): tile configuration by M,
// split-K plan, scratch.
#include "dispatch.hpp"
#include "skinny_gemm.hpp"

namespace clove {
namespace {

using namespace sk;

// (I8, BM, BN, WM, WN, stages)
// (three stages: two workgroups fit a CU and the first stage waits behind a
// smaller burst, which measured at least as fast as five on every shape with
// M <= 32 and up to 128 K tiles: 12 x 1344 x 2816 13.4 -> 9.3 us, 7 x 8057 x
// 1015 13.0 -> 11.5)
using F16M32 = Cfg<false, 32, 128, 1, 4, 3>;
using F16M32S5 = Cfg<false, 32, 128, 1, 4, 5>;  // past 128 K tiles (27 x 11840 x 10240 46.8 -> 44.6)
using F16M128 = Cfg<false, 128, 64, 4, 1, 4>;
// mid-size shapes (M > 256) whose 256x256 tile grid would leave CUs idle:
// 128x128 tiles (waves of 64x64)
// (hot launches: 2048^3 25 us with 128x128 against 45 us on the generic
// register-staged kernel; 512x4096x4096 29 us with 128x128 in two K splits
// against 33 us with 128x64)
using F16T128 = Cfg<false, 128, 128, 2, 2, 3>;
// few tiles: 64x64, 64 KB of LDS, so that two workgroups share a CU (505 x 2304
// x 1088 14.6 -> 10.5 us against six stages; see pick_f16_tile).  Four stages at
// any K: with two, for K <= 512, 109 x 5376 x 512 took 8.6 us against 5.8
using F16T64 = Cfg<false, 64, 64, 2, 2, 4>;
// 72 KB of LDS, two workgroups per CU (see pick_f16_tile)
using F16W128 = Cfg<false, 64, 128, 2, 2, 3>;
// small products (short K, at most one 32x32 tile per CU): 32x32 tiles whose
// four waves take one k-step of every K tile each, two stages ahead -- 4x the
// workgroups of 64x64 tiles at a quarter of the operand bytes each (hot graph
// replays, us per call, against the 64x64 / 32x128 tiles: 512^3 4.98 / 5.61
// -> 4.27, 512 x 512 x 1024 6.90 / 7.83 -> 5.51, 64 x 4096 x 1024 6.91 / 7.83
// -> 5.49, 3 x 8192 x 1024 6.72 / 7.71 -> 5.33, 100 x 200 x 320 4.04 / 4.53
// -> 3.67; one or three stages ahead no faster; at 512 such tiles and more it
// only ties or loses: 512 x 1024 x 512 5.27 -> 5.21, 1024 x 1024 x 512 5.81
// -> 7.13)
using F16K32 = Cfg<false, 32, 32, 1, 1, 3, 1, 4>;
// up to 32 rows, small products: 32x64 tiles, two k slices, 64 KB of LDS
using F16N64 = Cfg<false, 32, 64, 1, 2, 4, 1, 2>;
using I8M32 = Cfg<true, 32, 128, 1, 4, 3>;
using I8T64 = Cfg<true, 64, 64, 2, 2, 4>;
using I8W128 = Cfg<true, 64, 128, 2, 2, 3>;  // 72 KB LDS: two workgroups per CU
using I8M128 = Cfg<true, 128, 64, 4, 1, 4>;
using I8T128 = Cfg<true, 128, 128, 2, 2, 3>;

// K tiles per split: split K until about one workgroup per CU, not with four
// k slices.  128-row tiles keep two K tiles per split and are not split for
// short K (<= 16 K tiles), where the publish / count / reload tail costs more
// than the shorter stream saves; the smaller tiles, whose tail is shorter,
// keep four (two a split measured slower on most) and split INT8 past 9 K tiles
// (9 x 5633 x 2048 17.1 -> 12.0 us, 10 x 1228 x 1536 12.1 -> 8.9; up to 9 250 x 1792 x
// 1024 7.3 -> 6.4 unsplit, 28 x 12160 x 1024 7.6 -> 6.8; 32-row tiles past 13 where
// they cover a quarter of the CUs, 9 x 12544 x 1408 8.1 -> 7.7), FP16 past 13 K tiles
// with 64-row tiles (101 x 960 x 576 6.1 in two splits, 5.5 unsplit; 221 x 6976 x
// 832 7.6, 6.8; at 15 and 16 K tiles they tie; not unaligned operands, 32 x 166 x
// 64 x 484 9.9 in two splits, 12.0 unsplit) and past 15 with 32x128 ones (7 x
// 8057 x 1015 13.0 -> 11.5; 18 x 10496 x 896 7.9 -> 8.9 in three splits).
template <class CF>
int tiles_per_split(int M, int N, int K, int batch, int cus, bool ua = false) {
    const int tiles = cdiv(M, CF::BM) * cdiv(N, CF::BN) * batch;
    const int nk = cdiv(K, CF::BK);
    int ns = tiles >= cus ? 1 : cus / tiles;
    ns = max(1, min(ns, nk / (CF::BM == 128 ? 2 : 4)));
    if ((CF::BM == 128 && nk <= 16) || CF::KW > 2) ns = 1;
    const int unsplit = !CF::I8 ? (CF::BM == 32 ? 15 : 13) : CF::BM == 32 && 4 * tiles > cus ? 13 : 9;
    if (nk <= unsplit && !(ua && (CF::I8 || CF::BM != 32))) ns = 1;
    return cdiv(nk, ns);
}

template <class CF, int OUT, bool ZP = false, Feed FEED = kWhole>
clove_status_t run(Args a, int batch, int cus, hipStream_t stream, int kt_per = 0) {
    a.tiles_m = cdiv(a.M, CF::BM);
    a.tiles_n = cdiv(a.N, CF::BN);
    a.batch = batch;
    const int tiles = a.tiles_m * a.tiles_n * batch;
    const int nk = cdiv(a.K, CF::BK);
    if (kt_per == 0) kt_per = tiles_per_split<CF>(a.M, a.N, a.K, batch, cus, FEED == kUnaligned);
    a.kps = kt_per * CF::BK;
    a.nsplit = cdiv(nk, kt_per);
    if (a.nsplit > 1) {
        Scratch s;
        const size_t bytes =
            (size_t)tiles * a.nsplit * CF::NT * CF::NB * CF::FM * CF::FN * (16 / CF::KW) * sizeof(float);
        const bool unsplit = runs_unsplit(FEED != kWhole, batch, a.M, a.N, a.K, CF::BK, cus);
        const clove_status_t st = acquire_scratch(stream, bytes, (size_t)tiles, &s, unsplit);
        if (unsplit && scratch_short(st)) {
            a.kps = nk * CF::BK;
            a.nsplit = 1;
        } else if (st != CLOVE_OK) {
            return st;
        }
        a.part = s.partials;
        a.counters = s.counters;
    }
    auto k = skinny_gemm<CF, OUT, ZP, FEED>;
    constexpr int lds = FEED == kUnaligned ? CF::LDS_UA : CF::LDS;
    if (ensure_lds(reinterpret_cast<const void*>(k), lds) != CLOVE_OK)
        return CLOVE_ERR_LAUNCH;
    CLOVE_LAUNCH(k, dim3((unsigned)(tiles * a.nsplit)), dim3(CF::NT), lds, stream, a);
    return check_launch();
}

bool fits31(int64_t bytes) { return bytes < ((int64_t)1 << 31); }

// The FP16 tile shapes, chosen by shape alone (so that the fused SwiGLU below
// picks the same tiles, and with them the same split plan, as the two GEMMs
// it replaces).
enum class F16Tile { kM32, kN64, kM128, kT128, kW128, kT64, kK32 };

F16Tile pick_f16_tile(int batch, int M, int N, int K, int cus) {
    const int nk = cdiv(K, F16T64::BK);
    const bool short_k = nk <= 16;
    const bool long_k = K >= 4096;
    // (from 17 K tiles on, tiles that split K are ahead: 26 x 896 x 1344 9.4 us with
    // 32x32, 6.4 with 32x64; 50 x 576 x 1472 10.0 against 6.6 with 64x64)
    if (nk <= 16 && (int64_t)cdiv(M, F16K32::BM) * cdiv(N, F16K32::BN) * batch <= cus) return F16Tile::kK32;
    // 64x64 tiles (up to 32 rows, where half of such a tile is padding, 32x64) while
    // the product is small, whatever its M: their time is about tiles x K tiles (us
    // per call over operands that rotate past the Infinity Cache, 400 shapes,
    // against the tiles below: 153 x 1280 x 6080 16.8 -> 13.0, 190 x 3712 x 1792 13.7
    // -> 11.8, 249 x 3200 x 2048 14.1 -> 12.7, 20 x 12096 x 1600 11.4 -> 10.1).  Not
    //  * past 28 tiles x K tiles a CU (182 x 4096 x 3008, 35 a CU, 19.4 against 17.1
    //    with 128x64; 128 x 4096 x 4096, 32, 18.3 against 17.3, although with three
    //    operand sets, which that cache holds, 13.4 against 15.1), 33 where there are
    //    splits or a second round to balance it (141 x 9024 x 1216 14.5 against 22.0;
    //    269 x 768 x 8256, 30, 14.9 against 26.1 with 128x128; 81 x 2944 x 6528, 37, 18.8
    //    against 16.7);
    //  * in a second round of the CUs (182 x 5888 x 1728, 276 tiles, 19.0 against
    //    15.0) past 6 K tiles (314 x 5120 x 320 5.3 against 6.0), unless the 128x64
    //    tiles take one too (32 x 159 x 320 x 512 8.7 against 13.2);
    //  * past 32 K tiles where more than half the CUs have a tile, which leaves no
    //    room for a split (123 x 4224 x 3520 19.5 against 15.9, 7 x 9984 x 2752 14.5
    //    against 13.8), 40 where 128-row tiles would pad another 64 rows (166 x 2944 x
    //    2560 14.6 against 15.8); the fused SwiGLU takes the same tiles and loses
    //    earlier (70 x 5120 x 2304 23.4 against 19.9, 151 x 3072 x 3072 27.5 against 23.6);
    //  * up to 32 rows of unaligned operands past 28 K tiles and 64 tiles (4 x 5723 x
    //    4904 24.2 against 19.2).
    const int64_t t64 = (int64_t)cdiv(M, F16T64::BM) * cdiv(N, F16T64::BN) * batch;
    const int64_t t128x64 = (int64_t)cdiv(M, F16M128::BM) * cdiv(N, F16M128::BN) * batch;
    const bool pads = M > 64 && cdiv(M, 64) % 2 == 1;
    const int rounds = M > 32 && (nk <= 6 || t128x64 > cus) ? 2 : 1;
    const bool small = t64 <= rounds * cus && t64 * nk <= (2 * t64 < cus || t64 > cus ? 33 : 28) * cus &&
                       (2 * t64 <= cus || nk <= (pads ? 40 : 32));
    if (M <= 32)
        return 4 * t64 <= cus || (small && (nk <= 28 || (K % 8 == 0 && N % 8 == 0))) ? F16Tile::kN64 : F16Tile::kM32;
    if (M <= 64 || small) return F16Tile::kT64;
    // 128x128 tiles, split K when they are few: for M > 256 once they cover
    // half the CUs or K is long, for 128 < M <= 256 on long K and N >= 4096
    // (cold weights, against 64x64 tiles for M > 256 and 128x64 up to 256:
    // 11008x4096 at M = 192 44.3 against 64.2 us, 4096x11008 at M = 384 64.1
    // against 108.6 us, 2048x8192 at M = 512 35.2 against 47.4 us)
    if (M > 256) {
        const int64_t t128 = (int64_t)cdiv(M, 128) * cdiv(N, 128) * batch;
        // 64x128 between them, two workgroups a CU: where the 128x128 grid is
        // too small but this one fills 3/4 of the CUs (334 x 4288 x 1664 20.4 ->
        // 16.7 us against 64x64, 333 x 5001 x 2050 31.9 -> 25.8), and for short
        // K up to 8 K tiles (16 x 962 x 448 x 128 13.4 -> 12.0 against 128x128) or where
        // the 128x128 tiles take a second round (1729 x 2752 x 704 23.4 -> 19.8; in one
        // round 359 x 8384 x 960 stays, 15.5 against 20.8, and with longer K 559 x 4352 x
        // 2688, 29.3 against 41.3)
        const int64_t w64 = (int64_t)cdiv(M, F16W128::BM) * cdiv(N, F16W128::BN) * batch;
        if (t128 >= cus / 2 ? short_k && (nk <= 8 || t128 > cus) : !long_k && 4 * w64 >= 3 * cus) return F16Tile::kW128;
        return (t128 >= cus / 2 || long_k) ? F16Tile::kT128 : F16Tile::kT64;
    }
    if (M > 128 && long_k && N >= 4096) return F16Tile::kT128;
    // and for 64 < M <= 128 on wide weights (N >= 10240, K >= 4096), in two K
    // splits: half the A-panel bytes per workgroup of the 128x64 tiles (cold,
    // 128 x 11008 x 4096 35.1 -> 30.2 us, 96 x 11008 x 4096 31.2 -> 28.5,
    // 80 x 11008 x 4096 30.8 -> 27.7, 128 x 14336 x 4096 39.0 -> 34.1; not at
    // N = 8192, K = 2048 or N = 4096, K = 11008, where 128x64 stays ahead)
    if (M > 64 && M <= 128 && long_k && N >= 10240) return F16Tile::kT128;
    // short K with few 128-row tiles: 32-row tiles make 4x the workgroups
    // without a split; with many tiles (batches of heads), 64x128, two workgroups a
    // CU (64 x 199 x 960 x 96 29.2 -> 21 us, 16 x 158 x 1312 x 512 19.5 -> 16.1; the
    // same times where the stores are the bound)
    if (short_k && t64 > 2 * cus) return F16Tile::kW128;
    return short_k && 2 * t128x64 < cus ? F16Tile::kM32 : F16Tile::kM128;
}

bool f16_domain(int batch, const void* A, const void* B, const void* C, int M, int N, int K) {
    if (M <= 0 || K <= 0 || K % 8 != 0 || N < 8 || N % 8 != 0) return false;
    if (M <= 4 && !skinny_before_gemv(batch, M, N, K)) return false;
    if (!aligned16(A) || !aligned16(B) || !aligned16(C)) return false;
    // (the DMA offsets of the padded rows m < M + 128 must stay 32-bit)
    return fits31((int64_t)(M + 128) * K * 2) && fits31((int64_t)(K + 64) * N * 2) && fits31((int64_t)M * N * 2);
}

// The unaligned variant (UA): any strides and element-aligned pointers.  Both
// operands hold at least one 16-byte chunk, and a row of B does (a chunk of
// any K tile but the last then stays inside B).
bool ua_domain(int M, int N, int K, int es) {
    return M >= 1 && K >= 1 && N * es >= 16 && (int64_t)M * K * es >= 16 && fits31((int64_t)(M + 128) * K * es) &&
           fits31((int64_t)(K + 128) * N * es);
}

// two-B-operand (gate, up) counterparts of the tiles above; fewer stages
// where both B tiles would not fit the LDS
using SwM32 = Cfg<false, 32, 128, 1, 4, 4, 2>;
using SwN64 = Cfg<false, 32, 64, 1, 2, 3, 2, 2>;
using SwM128 = Cfg<false, 128, 64, 4, 1, 4, 2>;
using SwT128 = Cfg<false, 128, 128, 2, 2, 3, 2>;
using SwT64 = Cfg<false, 64, 64, 2, 2, 4, 2>;
using SwK32 = Cfg<false, 32, 32, 1, 1, 3, 2, 4>;

}  // namespace

bool try_skinny_fp16(const uint16_t* A, const uint16_t* B, uint16_t* C, int batch, int M, int N, int K,
                     float alpha, float beta, int cus, hipStream_t stream, clove_status_t* status) {
    const bool al = f16_domain(batch, A, B, C, M, N, K);
    if (!al && !ua_domain(M, N, K, 2)) return false;
    Args a{};
    a.A = A;
    a.B = B;
    a.C = C;
    a.alpha = alpha;
    a.beta = beta;
    a.M = M;
    a.N = N;
    a.K = K;
    a.sA = (int64_t)M * K;
    a.sB = (int64_t)K * N;
    a.sC = (int64_t)M * N;
    auto go = [&](auto cfg) {
        using CF = decltype(cfg);
        if (!al) return run<CF, kF16AlphaBeta, false, kUnaligned>(a, batch, cus, stream);
        return K % CF::BK == 0 ? run<CF, kF16AlphaBeta>(a, batch, cus, stream)
                               : run<CF, kF16AlphaBeta, false, kRagged>(a, batch, cus, stream);
    };
    switch (pick_f16_tile(batch, M, N, K, cus)) {
        case F16Tile::kM32: *status = K > 128 * F16M32::BK ? go(F16M32S5{}) : go(F16M32{}); break;
        case F16Tile::kN64: *status = go(F16N64{}); break;
        case F16Tile::kM128: *status = go(F16M128{}); break;
        case F16Tile::kT128: *status = go(F16T128{}); break;
        case F16Tile::kW128: *status = go(F16W128{}); break;
        case F16Tile::kT64: *status = go(F16T64{}); break;
        case F16Tile::kK32: *status = go(F16K32{}); break;
    }
    return true;
}

bool try_skinny_swiglu(const uint16_t* X, const uint16_t* W_gate, const uint16_t* W_up, uint16_t* out, int T,
                       int hidden, int inter, int cus, hipStream_t stream, clove_status_t* status) {
    if (!f16_domain(1, X, W_gate, out, T, inter, hidden) || !aligned16(W_up) || hidden % 64 != 0) return false;
    Args a{};
    a.A = X;
    a.B = W_gate;
    a.B2 = W_up;
    a.C = out;
    a.alpha = 1.0f;
    a.M = T;
    a.N = inter;
    a.K = hidden;
    a.sA = (int64_t)T * hidden;
    a.sB = (int64_t)hidden * inter;
    a.sC = (int64_t)T * inter;
    switch (pick_f16_tile(1, T, inter, hidden, cus)) {
        case F16Tile::kM32: *status = run<SwM32, kF16SwiGLU>(a, 1, cus, stream); break;
        case F16Tile::kN64: *status = run<SwN64, kF16SwiGLU>(a, 1, cus, stream); break;
        case F16Tile::kM128: *status = run<SwM128, kF16SwiGLU>(a, 1, cus, stream); break;
        case F16Tile::kT128: *status = run<SwT128, kF16SwiGLU>(a, 1, cus, stream); break;
        case F16Tile::kW128: {
            // (never split there; two B tiles leave one workgroup a CU, so the
            // larger tile where its grid is large)
            const int nk = cdiv(hidden, F16W128::BK);
            *status = (int64_t)cdiv(T, 128) * cdiv(inter, 128) >= cus / 2
                          ? run<SwT128, kF16SwiGLU>(a, 1, cus, stream, nk)
                          : run<SwT64, kF16SwiGLU>(a, 1, cus, stream, nk);
            break;
        }
        case F16Tile::kT64: {
            // (96 KB of LDS, one workgroup a CU: past one round of them 128x64 tiles
            // under the same split, 219 x 4224 x 1280 25.5 -> 17.7 us)
            const int kt_per = tiles_per_split<F16T64>(T, inter, hidden, 1, cus);
            *status = T > 64 && T <= 256 && cdiv(T, 64) * cdiv(inter, 64) > cus
                          ? run<SwM128, kF16SwiGLU>(a, 1, cus, stream, kt_per)
                          : run<SwT64, kF16SwiGLU>(a, 1, cus, stream, kt_per);
            break;
        }
        case F16Tile::kK32: *status = run<SwK32, kF16SwiGLU>(a, 1, cus, stream); break;
    }
    return true;
}

bool try_skinny_int8(const Int8Args& q, int cus, hipStream_t stream, clove_status_t* status) {
    const bool al = q.K > 0 && q.K % 16 == 0 && q.N >= 16 && q.N % 16 == 0 && aligned16(q.A) && aligned16(q.B) &&
                    aligned16(q.C) && fits31((int64_t)(q.M + 128) * q.K) && fits31((int64_t)(q.K + 128) * q.N) &&
                    fits31((int64_t)q.M * q.N * 4);
    if (!al && !ua_domain(q.M, q.N, q.K, 1)) return false;
    Args a{};
    a.A = q.A;
    a.B = q.B;
    a.C = q.C;
    a.sa = q.sa;
    a.sb = q.sb;
    a.scale = q.scale;
    a.za = q.za;
    a.zb = q.zb;
    a.acc_add = q.acc_add;
    a.M = q.M;
    a.N = q.N;
    a.K = q.K;
    const bool zp = q.za != 0 || q.zb != 0;
    auto pick = [&](auto out_tag) -> clove_status_t {
        constexpr int OUT = decltype(out_tag)::value;
        auto go = [&](auto cfg) {
            using CF = decltype(cfg);
            // (the unaligned variant always carries the zero points)
            if (!al) return run<CF, OUT, true, kUnaligned>(a, 1, cus, stream);
            return zp ? run<CF, OUT, true>(a, 1, cus, stream) : run<CF, OUT>(a, 1, cus, stream);
        };
        // (us per call, 350 shapes over operands that rotate past the Infinity Cache
        // unless three sets are named, which it holds; "was": 32x128 in five stages
        // up to M = 64, or 128 on weights up to 32 Mi, else 128x64)
        const int64_t t64 = (int64_t)cdiv(q.M, I8T64::BM) * cdiv(q.N, I8T64::BN);
        const int64_t w64 = (int64_t)cdiv(q.M, I8W128::BM) * cdiv(q.N, I8W128::BN);
        const int64_t t128x64 = (int64_t)cdiv(q.M, I8M128::BM) * cdiv(q.N, I8M128::BN);
        const int nk = cdiv(q.K, I8T64::BK);
        if (q.M <= 32) return go(I8M32{});
        // 64 rows: 64x128 tiles once 64x64 ones fill a quarter of the CUs over a
        // longer K, 18 tiles x K tiles a CU (39 x 13376 x 4736, 30 a CU, 28.8 -> 19.2, 62
        // x 4620 x 8512, 19, 28.7 -> 21.8, three sets; 56 x 7616 x 9984, 36, 27.0 with 64x64,
        // 22.7; 42 x 4480 x 4736, 10, 11.8 with 64x64, 13.5), else 64x64 (34 x 6848 x 896
        // 6.5 -> 5.3, 39 x 960 x 5376 12.4 -> 10.5, three sets)
        if (q.M <= 64) return 4 * t64 > cus && t64 * nk > 18 * cus ? go(I8W128{}) : go(I8T64{});
        // small products, at any M, in one round of the CUs (two where unaligned, 276 x
        // 5703 x 498 12.7 against 16.1): 64x64 (187 x 512 x 9728
        // 19.8 -> 12.9, 509 x 512 x 5376 16.9 -> 11.6, three sets; from 16 tiles x K
        // tiles a CU, 20 from 129 rows, 70 x 4224 x 4754 19.9 -> 23.7, 683 x 2432 x
        // 3200 14.8 -> 18.2, 128 x 4096 x 4096 14.1 -> 14.4; in a second round 245 x 5696 x 1152 9.2 -> 12.0, 132 x 6336
        // x 1664 11.5 -> 14.5)
        if (t64 <= (al ? 1 : 2) * cus && t64 * nk < (q.M <= 128 ? 16 : 20) * cus) return go(I8T64{});
        if (q.M <= 128) {
            // 32-row tiles in one round on weights up to 32 Mi, 128x128 on wide
            // weights, as for FP16 (128 x 11008 x 4096 23.7 -> 20.5; 128 x 4096 x 11008
            // stays on 128x64); unaligned past one round 64x128 (82 x 10958 x 2634 36.1
            // -> 26.5), aligned 128x64 (75 x 12864 x 2816 14.9, with 64x128 18.8)
            const bool large_w = (int64_t)q.N * q.K > ((int64_t)32 << 20);
            if (!large_w && (int64_t)cdiv(q.M, I8M32::BM) * cdiv(q.N, I8M32::BN) <= cus) return go(I8M32{});
            if (large_w && q.N >= 10240 && q.K >= 4096) return go(I8T128{});
            return !al && !large_w ? go(I8W128{}) : go(I8M128{});
        }
        // 64x128, two workgroups a CU, where that fills the chip (aligned: 577 x 4096 x
        // 13952 120.8 -> 75.5, 986 x 2816 x 4224 43.2 -> 28.4, 1474 x 4480 x 8704 157.5 ->
        // 103.6, three sets, 512 x 4096 x 4096 22.9 -> 22.0; with 135 tiles 1666 x 576 x
        // 13440 39.3 -> 67.7; unaligned operands, whose K tiles go through registers, only
        // tie), unless it starts a second round that 128x64 does not (339 x 5440 x 2304
        // 15.6 -> 20.7).  Up to 256 rows each B panel is read by as many 64-row tiles from
        // HBM, and 128x64 stays (199 x 11328 x 4480 43.1 -> 48.6) unless it takes a second
        // round and either pads another 64 rows (134 x 9280 x 10368 98.9 -> 63.8, three
        // sets, 141 x 11200 x 1664 20.5 -> 13.4) or K is short (194 x 11008 x 1664 25.0 ->
        // 17.1).  Up to M = 2048, and with ragged K beyond, this kernel is ahead of the
        // register-staged MFMA GEMM (K % 128 != 0: 4096 x 4096 x 4112 163 -> 117, 2100 x
        // 4096 x 1040 165 -> 27); with whole K tiles at M = 4096 it is not.
        if (al && (q.M <= 256 ? (q.M <= 192 || nk <= 16) && t128x64 > cus
                               : 4 * w64 >= 3 * cus && (w64 <= cus || t128x64 > cus)))
            return go(I8W128{});
        return go(I8M128{});
    };
    switch (q.out) {
        case Int8Out::kHalfPerTensor: *status = pick(std::integral_constant<int, kI8Tensor>{}); break;
        case Int8Out::kHalfRowCol: *status = pick(std::integral_constant<int, kI8RowCol>{}); break;
        case Int8Out::kAcc32: *status = pick(std::integral_constant<int, kI8Acc32>{}); break;
        default: return false;
    }
    return true;
}

}  // namespace clove
