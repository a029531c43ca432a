// Tile constants of the skinny kernel, and where the loads of its unaligned form
// fall.  Plain C++ without device code: tests/test_skinny_unaligned_plan.py builds
// it for the host and replays every load.
#pragma once

namespace clove {
namespace sk {

// KW > 1: KW waves share each wave tile and take disjoint slices of every K
// tile's four k-steps, summed through LDS after the K loop (slice order, so
// deterministic): KW times the workgroups of the same wave tiles for small
// products (split K only with KW = 2)
template <bool I8_, int BM_, int BN_, int WM_, int WN_, int S_, int NB_ = 1, int KW_ = 1>
struct Cfg {
    static constexpr bool I8 = I8_;
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_, NB = NB_, KW = KW_;
    static constexpr int ES = I8 ? 1 : 2;  // bytes per element
    static constexpr int NW = WM * WN * KW, NT = 64 * NW;
    static constexpr int NKS = 4 / KW;     // k-steps per K tile per wave
    static constexpr int BK = 128 / ES;    // K per stage: 128 bytes of every A row
    static constexpr int BNB = BN * ES;    // bytes of one B k-row in the tile
    static constexpr int FM = BM / (32 * WM), FN = BN / (32 * WN);
    static constexpr int A_BYTES = BM * 128, B_BYTES = BK * BNB;
    static constexpr int SB = A_BYTES + NB * B_BYTES;
    static constexpr int DA = A_BYTES / 1024 / NW, DB = B_BYTES / 1024 / NW;  // DB per B operand
    static constexpr int D = DA + NB * DB;  // DMA instructions per thread per stage
    static_assert(NW == 4, "four waves");
    static_assert(NB == 1 || (NB == 2 && !I8), "two B operands: FP16 only");
    static_assert(FM >= 1 && FN >= 1 && BM == 32 * FM * WM && BN == 32 * FN * WN, "wave tiles");
    static_assert(BNB == 64 || BNB == 128 || BNB == 256 || BNB == 512, "B row bytes");
    static_assert(A_BYTES % (1024 * NW) == 0 && B_BYTES % (1024 * NW) == 0, "DMA split");
    static_assert(S >= 2 && S <= 9 && (S - 2) * D <= 63, "stages");
    static_assert(KW == 1 || ((KW == 2 || KW == 4) && !I8), "k slices");
    // the k-slice sums: every wave's NB FN FM 32x32 blocks, 4 KB each
    static constexpr int RED = KW > 1 ? NW * NB * FN * FM * 4096 : 0;
    static constexpr int LDS = S * SB + RED;
    static_assert(LDS <= 160 * 1024, "LDS");
    // UA: K tiles held in registers (16 D bytes per thread each), two LDS stages
    static constexpr int P = D <= 2 ? 6 : D <= 5 ? 4 : D <= 6 ? 3 : 2;
    static constexpr int LDS_UA = 2 * SB + RED;
};

// chunk swizzle of B k-row r (see skinny_gemm.hpp): the rows one
// transposing read touches (4 rows x 2 chunks for fp16, 8 rows x 1 chunk for
// int8) land in 8 different bank groups
// (rows of 128 or 256 bytes start on bank 0, rows of 64 bytes alternate halves)
template <int BNB, bool I8>
constexpr int swz_b(int r) {
    if constexpr (BNB >= 128) return I8 ? (r & 7) : 2 * (r & 3);
    else return I8 ? ((r >> 1) & 3) : 2 * ((r >> 1) & 1);
}

// ---- the unaligned form's 16-byte loads (byte offsets from the operand) ----
// Load `slot` (wave * DA + i of A, wave * DB + i of B) of a lane fills the same 16
// bytes of LDS as that DMA instruction's lane.

// A: byte within its row's 128 bytes of a K tile
constexpr int ua_col_a(int lane) { return 16 * ((lane & 7) ^ (lane >> 3)); }

// A: chunk of K tile 0 (row 0 for rows past M)
template <class CF>
constexpr unsigned ua_chunk_a(int m0, int slot, int lane, int M, int K) {
    const int row = m0 + 8 * slot + (lane >> 3);
    return (unsigned)(row < M ? row : 0) * K * CF::ES + ua_col_a(lane);
}

// B: chunk of K tile 0 (column 0 for chunks past N)
template <class CF>
constexpr unsigned ua_chunk_b(int n0, int slot, int lane, int N) {
    constexpr int CPR = CF::BNB / 16, RPI = 1024 / CF::BNB;  // chunks per B row, rows per instruction
    const int row = RPI * slot + lane / CPR;
    const int nb = n0 * CF::ES + 16 * ((lane % CPR) ^ swz_b<CF::BNB, CF::I8>(row));
    return (unsigned)row * N * CF::ES + (nb < N * CF::ES ? nb : 0);
}

// a load that may pass the operand's end comes from at most 16 bytes before it
// and is shifted into place
constexpr unsigned ua_inside(unsigned off, unsigned end) { return off < end - 16 ? off : end - 16; }

// A: bytes of a chunk of the K tile at k0 that lie before K (may pass 16 or be < 0)
template <class CF>
constexpr int ua_keep_a(int k0, int lane, int K) { return (K - k0) * CF::ES - ua_col_a(lane); }

// K tiles of a split whose chunks all lie inside the operands as they are: not
// the operands' last (a B chunk that passes its row's end reads into the next row)
template <class CF>
constexpr int ua_whole_tiles(int kbeg, int nkt, int K) { return kbeg + nkt * CF::BK < K ? nkt : nkt - 1; }

// the steady loop goes from K tile t to t + P while it loads whole tiles only
template <class CF>
constexpr bool ua_steady(int t, int whole) { return t + 2 * CF::P <= whole; }

}  // namespace sk
}  // namespace clove
