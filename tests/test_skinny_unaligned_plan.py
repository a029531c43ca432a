"""Host replay of the unaligned skinny GEMM's operand loads (skinny_gemm.hpp, UA).

Every 16-byte load of every workgroup, wave, lane and K tile: inside its
operand, and holding the operand's bytes (zero past K; anything for rows past M
and columns past N, which only reach outputs that are never stored). The offsets,
the clamp at the operand's end, the bytes kept and the K tiles of the steady loop
come from the kernel's own skinny_plan.hpp, built for the host.
"""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "clove_compute_amd", "csrc")

LANE = np.arange(64)


# the kernel's tiles, from skinny_gemm.hip (one B operand: those that run unaligned)
with open(os.path.join(CSRC, "skinny_gemm.hip")) as f:
    TILES = dict(re.findall(r"^using ((?:F16|I8)\w+) = (Cfg<[^;]*>);", f.read(), re.M))

CODE = """
#include "skinny_plan.hpp"
using namespace clove::sk;
struct Plan { int i8, bm, bn, bk, da, db, p; };
template <class CF> void plan(Plan* o) { *o = {CF::I8, CF::BM, CF::BN, CF::BK, CF::DA, CF::DB, CF::P}; }
// one load of the 64 lanes: offset in K tile 0 and, for K tile k0, the place it is
// loaded from and (A) the bytes kept
template <class CF>
void chunk(int a, int x0, int slot, int M, int N, int K, int k0, unsigned end, unsigned* off, unsigned* at, int* keep) {
    for (int l = 0; l < 64; ++l) {
        off[l] = (a ? ua_chunk_a<CF>(x0, slot, l, M, K) : ua_chunk_b<CF>(x0, slot, l, N)) +
                 (unsigned)k0 * (a ? 1 : N) * CF::ES;
        at[l] = ua_inside(off[l], end);
        keep[l] = a ? ua_keep_a<CF>(k0, l, K) : 16;
    }
}
extern "C" {
%s
}
"""
EACH = """
void plan_%(n)s(Plan* o) { plan<%(c)s>(o); }
int whole_%(n)s(int kbeg, int nkt, int K) { return ua_whole_tiles<%(c)s>(kbeg, nkt, K); }
int steady_%(n)s(int t, int whole) { return ua_steady<%(c)s>(t, whole); }
void chunk_%(n)s(int a, int x0, int slot, int M, int N, int K, int k0, unsigned end, unsigned* off, unsigned* at, int* keep) {
    chunk<%(c)s>(a, x0, slot, M, N, K, k0, end, off, at, keep);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, so = str(d / "plan.cpp"), str(d / "plan.so")
    with open(src, "w") as f:
        f.write(CODE % "".join(EACH % dict(n=n, c=c) for n, c in TILES.items()))
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, src, "-o", so], check=True)
    return ctypes.CDLL(so)


def swz_b(bnb, i8, r):
    """the LDS layout of B that the fragment reads expect"""
    if bnb >= 128:
        return (r & 7) if i8 else 2 * (r & 3)
    return ((r >> 1) & 3) if i8 else 2 * ((r >> 1) & 1)


def careful(buf, off, at, keep):
    """load_any16 at `at`, shift_bytes by off - at, keep_bytes"""
    assert at.min() >= 0 and at.max() + 16 <= buf.size and (off >= at).all()
    s = off - at
    j = np.arange(16)
    src = at[:, None] + s[:, None] + j
    v = np.where(s[:, None] + j < 16, buf[np.minimum(src, buf.size - 1)], 0)
    return np.where(j < keep[:, None], v, 0)


def fast(buf, off):
    assert off.min() >= 0 and off.max() + 16 <= buf.size
    return buf[off[:, None] + np.arange(16)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,ns", [(1, 17, 17, 1), (1, 16, 16, 1), (3, 130, 300, 1), (33, 33, 129, 1), (130, 200, 64, 1),
                                      (5, 16, 1157, 2), (40, 131, 1283, 3), (129, 65, 1024, 1), (2, 24, 2050, 4)])
def test_chunks(plan, tile, M, N, K, ns):
    c = (ctypes.c_int * 7)()
    getattr(plan, "plan_" + tile)(c)
    i8, BM, BN, BK, DA, DB, P = c
    whole_tiles, steady = getattr(plan, "whole_" + tile), getattr(plan, "steady_" + tile)

    def chunk(a, x0, slot, k0, end):
        off, at, keep = np.empty(64, np.uint32), np.empty(64, np.uint32), np.empty(64, np.int32)
        getattr(plan, "chunk_" + tile)(a, x0, slot, M, N, K, k0, ctypes.c_uint(end),
                                       *(v.ctypes.data_as(ctypes.c_void_p) for v in (off, at, keep)))
        return off.astype(np.int64), at.astype(np.int64), keep

    es = 1 if i8 else 2
    g = np.random.default_rng(M * 1000003 + N * 1009 + K)
    A = g.integers(1, 256, M * K * es, dtype=np.uint8)  # no zero bytes: a stray byte shows
    B = g.integers(1, 256, K * N * es, dtype=np.uint8)
    A2 = A.reshape(M, K * es)
    B2 = B.reshape(K, N * es)
    assert BK * es == 128
    # (LDS holds 128 bytes of an A row, its 16-byte chunk c at c ^ (row & 7), and BNB
    # bytes of a B row, chunk c at c ^ swz_b(row))
    BNB = BN * es
    CPR, RPI = BNB // 16, 1024 // BNB
    nk = -(-K // BK)
    kps = -(-nk // ns) * BK
    for m0 in range(0, M, BM):
        for n0 in range(0, N, BN):
            for kbeg in range(0, K, kps):
                nkt = -(-(min(K, kbeg + kps) - kbeg) // BK)
                whole = whole_tiles(kbeg, nkt, K)
                t_fast = set()  # K tiles the steady loop loads
                t = 0
                while steady(t, whole):
                    t_fast.update(range(t + P, t + 2 * P))
                    t += P
                for t in range(nkt):
                    k0 = kbeg + t * BK
                    for slot in range(4 * DA):
                        row = m0 + 8 * slot + (LANE >> 3)
                        off, at, keep = chunk(1, m0, slot, k0, A.size)
                        got = fast(A, off) if t in t_fast else careful(A, off, at, keep)
                        c = 16 * ((LANE & 7) ^ (LANE >> 3))
                        for ln in range(64):
                            want = np.zeros(16, np.uint8)
                            seg = A2[row[ln] if row[ln] < M else 0, k0 * es + c[ln]:k0 * es + c[ln] + 16]
                            want[:seg.size] = seg
                            assert np.array_equal(got[ln], want)
                    for slot in range(4 * DB):
                        row = RPI * slot + LANE // CPR
                        off, at, keep = chunk(0, n0, slot, k0, B.size)
                        got = fast(B, off) if t in t_fast else careful(B, off, at, keep)
                        nb = n0 * es + 16 * ((LANE % CPR) ^ swz_b(BNB, i8, row))
                        cb = np.where(nb < N * es, nb, 0)
                        for ln in range(64):
                            k = k0 + row[ln]
                            if k >= K:
                                assert not got[ln].any()
                            else:
                                seg = B2[k, cb[ln]:cb[ln] + 16]
                                assert np.array_equal(got[ln][:seg.size], seg)
