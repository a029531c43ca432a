// Host side of the group-wise INT4 x INT4 int8-MFMA GEMM (i4i4_gemm.hpp):
// eligibility, the Bt pre-pass, tile / split-K plan and scratch.
#include "dispatch.hpp"
#include "i4i4_gemm.hpp"

namespace clove {
namespace {

using namespace i4i4;

bool fits31(int64_t bytes) { return bytes < ((int64_t)1 << 31); }
size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

// One workgroup per CU (the rings take most of the LDS): 64-row tiles, split
// over groups until the grid reaches the CUs, never past them (a second round
// of workgroups would double the time), at least two groups per split.
struct Plan {
    int tiles_m, nsplit, gps;
};

Plan plan_for(int M, int tiles_n, int G, int cus) {
    Plan pl{};
    pl.tiles_m = cdiv(M, BR);
    const int tiles = pl.tiles_m * tiles_n;
    int ns = tiles >= cus ? 1 : cus / tiles;
    ns = max(1, min(ns, G / 2));
    // (an even number of groups per split: every stage starts on an even group,
    // whose (g, g + 1) pair of zA / sA is one aligned dword)
    pl.gps = 2 * cdiv(cdiv(G, ns), 2);
    pl.nsplit = cdiv(G, pl.gps);
    return pl;
}

}  // namespace

namespace {

// The shared body of the GEMM and the partials hook: plan, scratch, the Bt
// pre-pass, the launch.  P != null selects the partials mode (scales unused).
clove_status_t run(const Int4Args& q, int32_t* P, int cus, hipStream_t stream, bool optional = false) {
    const int G = cdiv(q.K, 128);
    const int Npad = cdiv(q.N, BC) * BC;
    Args a{};
    a.A = q.A;
    // (the partials mode never reads the scales; its weight DMA still needs a
    // valid [M, G] fp16 array to read from)
    a.sA = P ? q.A_zero : q.A_scale;
    a.zA = q.A_zero;
    a.C = q.C;
    a.P = P;
    a.M = q.M;
    a.N = q.N;
    a.K = q.K;
    a.G = G;
    a.Npad = Npad;
    a.tiles_n = Npad / BC;
    a.B = q.B;
    a.sB = q.B_scale;
    a.zB = q.B_zero;
    a.ldb = (q.N + 1) / 2;
    const bool anyk = q.K % 256 != 0;
    const int G2 = G + (G & 1);
    const Plan pl = plan_for(q.M, a.tiles_n, G2, cus);
    a.tiles_m = pl.tiles_m;
    a.nsplit = pl.nsplit;
    a.gps = pl.gps;
    const int tiles = a.tiles_m * a.tiles_n;
    const size_t slab = (size_t)BR * BC * 4;  // one fp32 partial tile
    const size_t part_bytes = !P && a.nsplit > 1 ? (size_t)tiles * a.nsplit * slab : 0;
    const size_t bt_bytes = round256((size_t)Npad * G2 * 128);
    const size_t sb_bytes = round256((size_t)G2 * Npad * 4);
    Scratch s;
    clove_status_t st = acquire_scratch(stream, part_bytes + bt_bytes + sb_bytes, (size_t)tiles, &s, optional);
    if (st != CLOVE_OK) return st;
    char* base = reinterpret_cast<char*>(s.partials);
    a.part = s.partials;
    a.counters = s.counters;
    int8_t* bt = reinterpret_cast<int8_t*>(base + part_bytes);
    float* sbf = reinterpret_cast<float*>(base + part_bytes + bt_bytes);
    a.Bt = bt;
    a.sBf = sbf;
    CLOVE_LAUNCH(anyk ? i4_prep_bt<true> : i4_prep_bt<false>, dim3((unsigned)G2, (unsigned)(Npad / PREP_COLS)), dim3(128), 0, stream, q.B, a.ldb,
                 P ? nullptr : q.B_scale, q.B_zero, q.N, q.K, Npad, bt, sbf);
    auto k = P ? i4i4_gemm<true> : anyk ? i4i4_gemm<false, true> : i4i4_gemm<false>;
    if (ensure_lds(reinterpret_cast<const void*>(k), LDS) != CLOVE_OK)
        return CLOVE_ERR_LAUNCH;
    CLOVE_LAUNCH(k, dim3((unsigned)(tiles * a.nsplit)), dim3(NT), LDS, stream, a);
    return check_launch();
}

// K a multiple of 256 (whole two-group stages; every (g, g + 1) fp16 pair of
// zA / sA is one aligned dword), a 16-byte aligned A, and offsets that fit
// the 32-bit buffer ranges
bool eligible(const Int4Args& q) {
    if (q.K <= 0 || q.K % 256 != 0 || !aligned16(q.A)) return false;
    const int G = q.K / 128;
    const int Npad = cdiv(q.N, BC) * BC;
    return fits31((int64_t)(q.M + BR) * (q.K / 2)) && fits31((int64_t)Npad * q.K) &&
           fits31((int64_t)q.M * G * 2) && fits31((int64_t)G * Npad * 4);
}

}  // namespace

// any other K, any alignment (at least one 16-byte piece of A)
bool eligible_anyk(const Int4Args& q) {
    if (q.K <= 0 || (int64_t)q.M * (q.K / 2) < 16) return false;
    const int64_t G2 = 2 * cdiv(q.K, 256), Npad = cdiv(q.N, BC) * BC;
    return fits31((int64_t)(q.M + BR) * (q.K / 2) + 256) && fits31(Npad * G2 * 128) && fits31((int64_t)q.M * G2 * 2);
}

// Group-wise mode with N >= 64 columns and K % 256 == 0 (fewer columns go to
// the GEMV / streaming kernels, K % 256 == 128 to the INT4-weight kernel, which
// needs no padding group: 8704 x 132 x 4224 37.8 us there, 62.7 here), and any
// N > 8 with K % 128 != 0, whose alternative is the generic kernel's byte
// gathers (us per call: 9856 x 233 x 10076 2058 -> 132, 5634 x 126 x 9196 629
// -> 41, 8768 x 18 x 4240 207 -> 32, 1728 x 76 x 1534 30 -> 18.5).
bool try_i4i4(const Int4Args& q, int cus, hipStream_t stream, clove_status_t* status) {
    if (q.mode != CLOVE_INT4_GROUPWISE) return false;
    if (q.N >= 64 && eligible(q)) {
        *status = run(q, nullptr, cus, stream);
        return true;
    }
    if (q.K % 128 == 0 || !eligible_anyk(q)) return false;
    // without scratch for the Bt pass, the generic kernel, whose plan needs none
    // where its 64 x 64 tiles cover the CUs or K is short
    *status = run(q, nullptr, cus, stream, (int64_t)cdiv(q.M, 64) * cdiv(q.N, 64) >= cus || q.K < 512);
    return !scratch_short(*status);
}

clove_status_t launch_i4i4_partials(const Int4Args& q, int32_t* P, int cus, hipStream_t stream) {
    if (!eligible(q)) return CLOVE_ERR_INVALID_ARG;
    return run(q, P, cus, stream);
}

}  // namespace clove
