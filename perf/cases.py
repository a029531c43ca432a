"""Workloads of the GEMM library, measured through its Python entry points.

Each kind below is one use of the library: FP16 products (decode, prefill,
odd shapes, attention heads, the FP16 MLP), W8A8, W4A4 and the W4A16 linear
layers of a Llama-style transformer.  `listed` names the standing cases,
`draw` gives more of the same ranges, `prepare` / `run` build and execute one.
Inputs come from a seeded generator on the GPU.
"""
from __future__ import annotations

import math

import torch

import clove_compute_amd as cg

GROUP = cg.INT4_GROUP_SIZE
MOST_FLOPS = 2.0 * 4096 ** 3  # no drawn case does more than the largest listed one


def listed():
    return [
        # one token through one FP16 projection: the smallest call, where
        # latency and launches count
        dict(name="fp16_decode", kind="fp16", M=1, N=4096, K=4096, beta=0.0),
        # a 128-token prompt chunk through a 7B-class down projection, added to
        # the residual stream
        dict(name="fp16_chunk", kind="fp16", M=128, N=4096, K=11008, beta=1.0),
        # the benchmark's headline: a large square product (long prefill)
        dict(name="fp16_square", kind="fp16", M=4096, N=4096, K=4096, beta=0.0),
        # odd sizes in every dimension: nothing aligned, nothing a multiple of a tile
        dict(name="fp16_ragged", kind="fp16", M=333, N=5001, K=2050, beta=0.0),
        # attention scores and values of 32 heads over a 512-token prompt
        dict(name="fp16_heads", kind="heads", batch=32, T=512, S=512, D=64),
        # the FP16 MLP's gate / up projections and SwiGLU, a 512-token prefill
        dict(name="fp16_mlp", kind="mlp", T=512, H=2048, I=8192, fused=True),
        # one token through one W8A8 projection, symmetric quantisation
        dict(name="int8_decode", kind="int8", M=1, N=4096, K=4096, za=0, zb=0, rowcol=False),
        # a 512-token prefill through a W8A8 projection with asymmetric
        # activations (a zero point on the activations, none on the weights)
        dict(name="int8_prefill", kind="int8", M=512, N=4096, K=4096, za=-9, zb=0, rowcol=False),
        # one token through a W4A4 projection of a 7B-class MLP
        dict(name="int4_decode", kind="int4", M=4096, N=1, K=11008),
        # a 128-token chunk through a W4A4 projection of a 7B-class MLP
        dict(name="int4_prefill", kind="int4", M=11008, N=128, K=4096),
        # one token through the linear layers of a 16-layer 1B-class model on
        # INT4 weights, recorded once into a graph and replayed per token
        dict(name="w4a16_decode", kind="w4a16", T=1, H=2048, QKV=3072, I=8192, layers=16, fused=True, graph=True),
        # a 512-token prefill through one such layer
        dict(name="w4a16_prefill", kind="w4a16", T=512, H=2048, QKV=3072, I=8192, layers=1, fused=True, graph=False),
    ]


def _logint(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    while True:
        kind = rng.choice(["fp16", "fp16", "heads", "mlp", "int8", "int8", "int4", "int4", "w4a16", "w4a16"])
        if kind == "fp16":
            # weights of 1B..13B-class projections or any sizes at all, one
            # token to a long prompt, with and without a residual
            odd = rng.random() < 0.35
            lo, hi, step = (33, 8192, 1) if odd else (512, 14336, 64)
            c = dict(kind=kind, M=_logint(rng, 1, 4096), N=_logint(rng, lo, hi, step), K=_logint(rng, lo, hi, step),
                     beta=rng.choice([0.0, 0.0, 1.0]))
            if c["N"] * c["K"] < 1 << 18:
                continue
        elif kind == "heads":
            c = dict(kind=kind, batch=rng.choice([8, 16, 32, 40, 64]), T=_logint(rng, 1, 1024),
                     S=_logint(rng, 16, 2048, rng.choice([1, 8, 64])), D=rng.choice([64, 80, 96, 128]))
            if c["batch"] * c["T"] * c["S"] > 32 * 1024 * 1024:
                continue
        elif kind == "mlp":
            c = dict(kind=kind, T=_logint(rng, 1, 1024), H=_logint(rng, 1024, 5120, 128),
                     I=_logint(rng, 2816, 13824, 128), fused=rng.random() < 0.75)
        elif kind == "int8":
            za, zb = rng.choice([(0, 0), (-9, 0), (17, 0), (-3, 5)])
            c = dict(kind=kind, M=_logint(rng, 1, 2048), N=_logint(rng, 512, 14336, rng.choice([1, 64, 64])),
                     K=_logint(rng, 512, 14336, rng.choice([2, 64, 128])), za=za, zb=zb, rowcol=rng.random() < 0.4)
        elif kind == "int4":
            c = dict(kind=kind, M=_logint(rng, 1024, 14336, rng.choice([1, 64, 64])), N=_logint(rng, 1, 1024),
                     K=_logint(rng, 1024, 14336, rng.choice([2, 128, 128, 256])))
        else:
            decode = rng.random() < 0.5
            c = dict(kind=kind, T=_logint(rng, 1, 32) if decode else _logint(rng, 33, 1024), H=_logint(rng, 1024, 4096, 128),
                     QKV=0, I=_logint(rng, 2816, 11008, 128), layers=rng.randint(2, 8) if decode else 1,
                     fused=rng.random() < 0.75, graph=decode)
            c["QKV"] = c["H"] + 128 * rng.choice([4, 8, c["H"] // 64])
        if work(c)["flops"] <= MOST_FLOPS:
            return c


# ---- inputs -----------------------------------------------------------------

class _Gen:
    """Seeded device tensors with the distributions the paths meet."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return (torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32) * std).half()

    def probs(self, *shape):
        return torch.softmax(torch.randn(*shape, generator=self.g, device="cuda"), -1).half()

    def int8(self, *shape, mean=0.0):
        v = torch.randn(*shape, generator=self.g, device="cuda") * 32.0 + mean
        return v.round_().clamp_(-128, 127).to(torch.int8)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)

    def scales(self, *shape, lo=0.002, hi=0.006):
        return (torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo).half()

    def zeros(self, *shape):
        """Integer zero points of 4-bit groups, around the middle of the range."""
        return torch.randint(5, 11, shape, generator=self.g, device="cuda").half()


def _empty(*shape):
    return torch.empty(*shape, dtype=torch.float16, device="cuda")


def _groups(K):
    return -(-K // GROUP)


def _inputs(c, seed):
    """The operands of a case, from its seed alone."""
    g, k = _Gen(seed), c["kind"]
    if k == "fp16":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(A=g.normal(M, K), B=g.normal(K, N, std=0.02), R=g.normal(M, N) if c["beta"] else None)
    if k == "heads":
        b, T, S, D = c["batch"], c["T"], c["S"], c["D"]
        return dict(Q=g.normal(b, T, D), Kt=g.normal(b, D, S), P=g.probs(b, T, S), V=g.normal(b, S, D))
    if k == "mlp":
        T, H, I = c["T"], c["H"], c["I"]
        return dict(X=g.normal(T, H), Wg=g.normal(H, I, std=0.02), Wu=g.normal(H, I, std=0.02))
    if k == "int8":
        M, N, K = c["M"], c["N"], c["K"]
        st = dict(A=g.int8(M, K, mean=c["za"]), B=g.int8(K, N, mean=c["zb"]))
        if c["rowcol"]:
            st.update(sa=g.scales(M, lo=0.01, hi=0.03), sb=g.scales(N, lo=0.0005, hi=0.001))
        return st
    if k == "int4":
        M, N, K, G = c["M"], c["N"], c["K"], _groups(c["K"])
        return dict(A=g.bytes(M, K // 2), sA=g.scales(M, G), zA=g.zeros(M, G), B=g.bytes(K, (N + 1) // 2),
                    sB=g.scales(G, N, lo=0.1, hi=0.3), zB=g.zeros(G, N))
    T, H, I = c["T"], c["H"], c["I"]

    def weight(O, K):
        return g.bytes(O, K // 2), g.scales(O, _groups(K)), g.zeros(O, _groups(K))

    return dict(R=g.normal(T, H),
                layers=[dict(xa=g.normal(T, H), attn=g.normal(T, H), xm=g.normal(T, H), qkv=weight(c["QKV"], H),
                             o=weight(H, H), gu=weight(2 * I, H), down=weight(H, I)) for _ in range(c["layers"])])


def _w4a16_pass(st):
    """The linear layers as a runtime sequences them: QKV, output projection
    into the residual stream, gate / up with SwiGLU, down projection into it."""
    c, h = st["case"], st["hidden"]
    T, H, I = c["T"], c["H"], c["I"]
    h.copy_(st["R"])
    for L in st["layers"]:
        cg.gemm_w4a16(L["xa"], *L["qkv"], L["yq"], T, c["QKV"], H)
        cg.gemm_w4a16(L["attn"], *L["o"], h, T, H, H, 1.0, 1.0)
        if c["fused"]:
            cg.w4a16_swiglu(L["xm"], *L["gu"], L["act"], T, I, H)
        else:
            q, s, z = L["gu"]
            cg.gemm_w4a16(L["xm"], q[:I], s[:I], z[:I], L["gate"], T, I, H)
            cg.gemm_w4a16(L["xm"], q[I:], s[I:], z[I:], L["up"], T, I, H)
            cg.swiglu(L["gate"], L["up"], L["act"], T * I)
        cg.gemm_w4a16(L["act"], *L["down"], h, T, H, I, 1.0, 1.0)


def prepare(case, seed):
    c = dict(case)
    st = _inputs(c, seed)
    st["case"] = c
    k = c["kind"]
    if k == "fp16":
        st["C"] = _empty(c["M"], c["N"])
    elif k == "heads":
        st["scores"], st["out"] = _empty(c["batch"], c["T"], c["S"]), _empty(c["batch"], c["T"], c["D"])
    elif k == "mlp":
        st["act"] = _empty(c["T"], c["I"])
        if not c["fused"]:
            st["gate"], st["up"] = _empty(c["T"], c["I"]), _empty(c["T"], c["I"])
    elif k in ("int8", "int4"):
        st["C"] = _empty(c["M"], c["N"])
    else:
        st["hidden"] = _empty(c["T"], c["H"])
        for L in st["layers"]:
            L["yq"], L["act"] = _empty(c["T"], c["QKV"]), _empty(c["T"], c["I"])
            if not c["fused"]:
                L["gate"], L["up"] = _empty(c["T"], c["I"]), _empty(c["T"], c["I"])
        if c["graph"]:
            _record(st)
    return st


def _record(st):
    """Records the pass into a graph over a caller-owned workspace, as a
    serving loop that must not allocate does."""
    with cg.workspace_query() as q:
        _w4a16_pass(st)
    st["ws"] = torch.zeros(q.bytes, dtype=torch.uint8, device="cuda") if q.bytes else None
    if q.bytes:
        cg.workspace_bind(st["ws"])
    try:
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            _w4a16_pass(st)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=s):
            _w4a16_pass(st)
    finally:
        if q.bytes:
            cg.workspace_bind()


# ---- one pass ---------------------------------------------------------------

def run(state):
    c = state["case"]
    k = c["kind"]
    if k == "fp16":
        if c["beta"]:
            state["C"].copy_(state["R"])  # the residual stream that the product is added to
        cg.gemm_fp16(state["A"], state["B"], state["C"], c["M"], c["N"], c["K"], 1.0, c["beta"])
        return state["C"]
    if k == "heads":
        b, T, S, D = c["batch"], c["T"], c["S"], c["D"]
        cg.gemm_fp16_batched(state["Q"], state["Kt"], state["scores"], b, T, S, D, 1.0 / math.sqrt(D))
        cg.gemm_fp16_batched(state["P"], state["V"], state["out"], b, T, D, S)
        return [state["scores"], state["out"]]
    if k == "mlp":
        T, H, I = c["T"], c["H"], c["I"]
        if c["fused"]:
            cg.swiglu_fused(state["X"], state["Wg"], state["Wu"], state["act"], T, H, I)
        else:
            cg.gemm_fp16(state["X"], state["Wg"], state["gate"], T, I, H)
            cg.gemm_fp16(state["X"], state["Wu"], state["up"], T, I, H)
            cg.swiglu(state["gate"], state["up"], state["act"], T * I)
        return state["act"]
    if k == "int8":
        if c["rowcol"]:
            cg.gemm_int8_rowcol(state["A"], state["B"], state["sa"], state["sb"], state["C"], c["M"], c["N"], c["K"],
                                c["za"], c["zb"])
        else:
            cg.gemm_int8(state["A"], state["B"], state["C"], c["M"], c["N"], c["K"], 0.02, c["za"], 0.0008, c["zb"])
        return state["C"]
    if k == "int4":
        cg.gemm_int4(state["A"], state["sA"], state["zA"], state["B"], state["sB"], state["zB"], state["C"],
                     c["M"], c["N"], c["K"])
        return state["C"]
    if c["graph"]:
        state["graph"].replay()
    else:
        _w4a16_pass(state)
    return [state["hidden"]] + [x for L in state["layers"] for x in (L["yq"], L["act"])]


def _w4_bytes(O, K):
    return O * K / 2 + 4 * O * _groups(K)


def work(case):
    """Bytes with every operand read once and every output written once."""
    c, k = case, case["kind"]
    if k == "fp16":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 2.0 * (M * K + K * N + (2 if c["beta"] else 1) * M * N), "flops": 2.0 * M * N * K}
    if k == "heads":
        b, T, S, D = c["batch"], c["T"], c["S"], c["D"]
        return {"bytes": 4.0 * b * (T * D + D * S + T * S), "flops": 4.0 * b * T * S * D}
    if k == "mlp":
        T, H, I = c["T"], c["H"], c["I"]
        return {"bytes": 2.0 * (T * H + 2 * H * I + T * I), "flops": 4.0 * T * H * I}
    if k == "int8":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 1.0 * (M * K + K * N + 2 * M * N + (2 * (M + N) if c["rowcol"] else 0)), "flops": 2.0 * M * N * K}
    if k == "int4":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": _w4_bytes(M, K) + K * ((N + 1) // 2) + 4.0 * _groups(K) * N + 2.0 * M * N, "flops": 2.0 * M * N * K}
    T, H, I, Q = c["T"], c["H"], c["I"], c["QKV"]
    weights = _w4_bytes(Q, H) + _w4_bytes(H, H) + _w4_bytes(2 * I, H) + _w4_bytes(H, I)
    acts = 2.0 * T * (3 * H + Q + I + (I + 4 * H))
    return {"bytes": c["layers"] * (weights + acts), "flops": c["layers"] * 2.0 * T * (H * (Q + H + 2 * I) + H * I)}


def tolerance(case):
    """Four times what one rounding of the result to fp16 leaves against 64
    bits (2.1e-4), and four units in the last place at most; the residual
    stream of the W4A16 layers is rounded after every addition to it (8.4e-4
    over 16 layers).  INT8 results are one rounding chain over an exact
    integer, the same for every implementation."""
    if case["kind"] == "int8":
        return "exact"
    return {"rel": 3.4e-3, "max": 1.6e-2} if case["kind"] == "w4a16" else {"rel": 8.4e-4, "max": 4e-3}


# ---- 64-bit results -----------------------------------------------------------

def _unpack(q):
    """[R, C/2] bytes -> [R, C] values, the even column in the high nibble."""
    return torch.stack((q >> 4, q & 15), -1).reshape(q.shape[0], -1)


def _per_k(v, K, dim):
    return v.double().repeat_interleave(GROUP, dim).narrow(dim, 0, K)


def _dequant(w):
    q, s, z = w
    K = 2 * q.shape[1]
    return (_unpack(q).double() - _per_k(z, K, 1)) * _per_k(s, K, 1)


def _swiglu64(gate, up):
    # both projections are fp16 results of their own before the activation
    gate, up = gate.half().double(), up.half().double()
    return gate / (1.0 + torch.exp(-gate)) * up


def exact(case, seed):
    c, k = case, case["kind"]
    st = _inputs(c, seed)
    if k == "fp16":
        r = st["A"].double() @ st["B"].double()
        return r + st["R"].double() if c["beta"] else r
    if k == "heads":
        scores = torch.stack([q.double() @ kt.double() for q, kt in zip(st["Q"], st["Kt"])]) / math.sqrt(c["D"])
        return [scores, torch.stack([p.double() @ v.double() for p, v in zip(st["P"], st["V"])])]
    if k == "mlp":
        x = st["X"].double()
        return _swiglu64(x @ st["Wg"].double(), x @ st["Wu"].double())
    if k == "int8":
        acc = (st["A"].double() - c["za"]) @ (st["B"].double() - c["zb"])
        return acc * (st["sa"].double()[:, None] * st["sb"].double()) if c["rowcol"] else acc * (0.02 * 0.0008)
    if k == "int4":
        N, K = c["N"], c["K"]
        b = (_unpack(st["B"])[:, :N].double() - _per_k(st["zB"], K, 0)) * _per_k(st["sB"], K, 0)
        return _dequant((st["A"], st["sA"], st["zA"])) @ b
    h, rest = st["R"].double(), []
    for L in st["layers"]:
        rest.append(L["xa"].double() @ _dequant(L["qkv"]).T)
        h = h + L["attn"].double() @ _dequant(L["o"]).T
        gate, up = (L["xm"].double() @ _dequant(L["gu"]).T).split(c["I"], 1)
        act = _swiglu64(gate, up)
        rest.append(act)
        h = h + act @ _dequant(L["down"]).T
    return [h] + rest
