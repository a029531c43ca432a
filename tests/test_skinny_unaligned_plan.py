"""Host replay of the unaligned skinny GEMM's operand loads (skinny_gemm.hpp, UA).

Every 16-byte load of every workgroup, wave, lane and K tile: inside its
operand, and holding the operand's bytes (zero past K; anything for rows past M
and columns past N, which only reach outputs that are never stored).
"""
import numpy as np
import pytest

LANE = np.arange(64)


def swz_b(bnb, i8, r):
    if bnb >= 128:
        return (r & 7) if i8 else 2 * (r & 3)
    return ((r >> 1) & 3) if i8 else 2 * ((r >> 1) & 1)


def careful(buf, off, keep):
    """load_any16 at min(off, end - 16), shift_bytes, keep_bytes"""
    at = np.minimum(off, buf.size - 16)
    assert at.min() >= 0 and at.max() + 16 <= buf.size
    s = off - at
    j = np.arange(16)
    src = at[:, None] + s[:, None] + j
    v = np.where(s[:, None] + j < 16, buf[np.minimum(src, buf.size - 1)], 0)
    return np.where(j < keep[:, None], v, 0)


def fast(buf, off):
    assert off.min() >= 0 and off.max() + 16 <= buf.size
    return buf[off[:, None] + np.arange(16)]


# (int8, BM, BN, P): the tiles of skinny_gemm.hip and their K tiles in registers
TILES = [(False, 32, 128, 4), (False, 128, 64, 3), (False, 128, 128, 2), (False, 64, 64, 4), (False, 32, 32, 6),
         (False, 64, 128, 3), (False, 32, 64, 4), (True, 32, 128, 4), (True, 128, 64, 3), (True, 128, 128, 2), (True, 64, 64, 4),
         (True, 64, 128, 3)]


@pytest.mark.parametrize("i8,BM,BN,P", TILES)
@pytest.mark.parametrize("M,N,K,ns", [(1, 17, 17, 1), (1, 16, 16, 1), (3, 130, 300, 1), (33, 33, 129, 1), (130, 200, 64, 1),
                                      (5, 16, 1157, 2), (40, 131, 1283, 3), (129, 65, 1024, 1), (2, 24, 2050, 4)])
def test_chunks(i8, BM, BN, P, M, N, K, ns):
    es = 1 if i8 else 2
    g = np.random.default_rng(M * 1000003 + N * 1009 + K)
    A = g.integers(1, 256, M * K * es, dtype=np.uint8)  # no zero bytes: a stray byte shows
    B = g.integers(1, 256, K * N * es, dtype=np.uint8)
    A2 = A.reshape(M, K * es)
    B2 = B.reshape(K, N * es)
    BK, BNB = 128 // es, BN * es
    DA, DB = BM * 128 // 4096, BK * BNB // 4096
    CPR, RPI = BNB // 16, 1024 // BNB
    nk = -(-K // BK)
    kps = -(-nk // ns) * BK
    for m0 in range(0, M, BM):
        for n0 in range(0, N, BN):
            for kbeg in range(0, K, kps):
                nkt = -(-(min(K, kbeg + kps) - kbeg) // BK)
                whole = nkt if kbeg + nkt * BK < K else nkt - 1
                t_fast = set()  # K tiles the steady loop loads
                t = 0
                while t + 2 * P <= whole:
                    t_fast.update(range(t + P, t + 2 * P))
                    t += P
                for t in range(nkt):
                    k0 = kbeg + t * BK
                    for w in range(4):
                        for i in range(DA):
                            lrow = 8 * (w * DA + i) + (LANE >> 3)
                            row = m0 + lrow
                            c = 16 * ((LANE & 7) ^ (LANE >> 3))
                            off = np.where(row < M, row, 0) * K * es + c + k0 * es
                            got = fast(A, off) if t in t_fast else careful(A, off, (K - k0) * es - c)
                            for ln in range(64):
                                want = np.zeros(16, np.uint8)
                                seg = A2[row[ln] if row[ln] < M else 0, k0 * es + c[ln]:k0 * es + c[ln] + 16]
                                want[:seg.size] = seg
                                assert np.array_equal(got[ln], want)
                        for i in range(DB):
                            row = RPI * (w * DB + i) + LANE // CPR
                            nb = n0 * es + 16 * ((LANE % CPR) ^ swz_b(BNB, i8, row))
                            cb = np.where(nb < N * es, nb, 0)
                            off = row * N * es + cb + k0 * N * es
                            got = fast(B, off) if t in t_fast else careful(B, off, np.full(64, 16))
                            for ln in range(64):
                                k = k0 + row[ln]
                                if k >= K:
                                    assert not got[ln].any()
                                else:
                                    seg = B2[k, cb[ln]:cb[ln] + 16]
                                    assert np.array_equal(got[ln][:seg.size], seg)
