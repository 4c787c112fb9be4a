"""The calls by which a decoder spends its time in this package, with inputs, work and tolerances.

Each case is one entry point (a quantizing prep, one matrix product at a batch
size, the load of one matrix) or one whole call (two layers of a batched
decode step as a captured graph, a whole decoded token). Sizes are those of
the 27B shapes that the benchmark uses (width 5120, FFN 17408, QKV 7168,
vocabulary 248320) and what lies around them.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "bonsai-ternary-fast_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

EPS = 1e-6
BLOCK = 1024  # the transform's block at the 27B shapes
STAGING = 64 << 20  # one pinned slot of the loader


def listed():
    return [
        # Input prep of one decoded token: RMSNorm, signs, FWHT 1024, Q8. The smallest call.
        {"name": "prep_token", "kind": "prep", "M": 1, "n": 5120, "norm": True, "perm": False},
        # The same call over a prompt's rows, at the widest input (the FFN's hidden vector).
        {"name": "prep_prompt", "kind": "prep", "M": 512, "n": 17408, "norm": False, "perm": False},
        # One decoded token through a square projection: latency.
        {"name": "gemv_o", "kind": "gemm", "M": 1, "K": 5120, "N": 5120, "segs": 1, "mode": "store"},
        # The output projection of one token: the largest single matrix.
        {"name": "gemv_head", "kind": "gemm", "M": 1, "K": 5120, "N": 248320, "segs": 1, "mode": "store"},
        # Gate and up of one token on PTQ1_0 rows as the file holds them.
        {"name": "gateup_packed", "kind": "packed", "M": 1, "K": 5120, "N": 17408, "segs": 2, "mode": "swiglu"},
        # Gate and up of 16 requests, with the Q8 that down reads next.
        {"name": "gateup_m16", "kind": "fused", "M": 16, "K": 5120, "N": 17408, "segs": 2, "mode": "swiglu"},
        # Q, K and V of 32 requests in one call.
        {"name": "qkv_m32", "kind": "gemm", "M": 32, "K": 5120, "N": 5120, "segs": 3, "mode": "store"},
        # A prompt of 512 tokens through gate and up: the largest product.
        {"name": "prefill_gateup", "kind": "gemm", "M": 512, "K": 5120, "N": 17408, "segs": 2, "mode": "swiglu"},
        # A prompt of an odd length through down: the longest sums.
        {"name": "prefill_down", "kind": "gemm", "M": 203, "K": 17408, "N": 5120, "segs": 1, "mode": "store"},
        # Two layers of a decode step of 8 requests, captured once and replayed, as a serving loop does.
        {"name": "layers_m8", "kind": "layers", "M": 8, "E": 5120, "QKV": 7168, "F": 17408, "layers": 2},
        # One whole token of the 27B shapes in one launch: embedding, 64 layers, head, pick.
        {"name": "token_27b", "kind": "token", "E": 5120, "QKV": 7168, "F": 17408, "V": 248320, "layers": 64},
        # One FFN matrix from host memory to its resident layout.
        {"name": "load_down", "kind": "load", "K": 17408, "N": 5120},
    ]


def _spread(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["prep", "gemv", "packed", "fused", "batch", "batch", "prefill", "prefill", "layers", "token",
                       "load"])
    if kind == "prep":
        return {"kind": "prep", "M": _spread(rng, 1, 512, 1), "n": _spread(rng, 512, 17408, 128),
                "norm": rng.random() < 0.5, "perm": rng.random() < 0.25}
    if kind == "load":
        return {"kind": "load", "K": _spread(rng, 1024, 17408, 128), "N": _spread(rng, 512, 17408, 1)}
    if kind == "layers":
        return {"kind": "layers", "M": _spread(rng, 3, 32, 1), "E": rng.choice([1024, 2048, 3072, 5120]),
                "QKV": 256 * rng.randint(6, 28), "F": 256 * rng.randint(12, 68), "layers": rng.randint(1, 2)}
    if kind == "token":
        return {"kind": "token", "E": rng.choice([2048, 4096, 5120]), "QKV": 512 * rng.randint(6, 14),
                "F": 1024 * rng.randint(8, 17), "V": 32 * rng.randint(1000, 7760), "layers": rng.randint(2, 48)}
    mode, segs = rng.choice([("store", 1), ("store", 3), ("swiglu", 2)])
    M = {"gemv": rng.randint(1, 2), "packed": rng.randint(1, 2), "fused": _spread(rng, 3, 32, 1),
         "batch": _spread(rng, 3, 32, 1), "prefill": _spread(rng, 33, 512, 1)}[kind]
    if kind == "fused" and mode == "store":
        segs = 1
    K = _spread(rng, 1024, 10240 if kind == "fused" else 17408, 128)
    N = _spread(rng, 512, 17408, 32) if kind == "fused" else _spread(rng, 512, 17408 // segs, 1)
    if kind == "prefill" and K > 8192:
        N = min(N, 8192)
    return {"kind": kind if kind in ("packed", "fused") else "gemm", "M": M, "K": K, "N": N, "segs": segs,
            "mode": mode}


# ---- inputs (plain torch, from the seed alone) ----
class Source:
    """Seeded inputs on the GPU, the same for prepare() and exact()."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        # P(-1, 0, +1) = (0.3, 0.4, 0.3): four codes (trit + 1) to a byte of the resident layout
        c = np.random.default_rng(11).choice(3, p=[0.3, 0.4, 0.3], size=(65536, 4))
        self.t2 = torch.from_numpy((c << np.array([0, 2, 4, 6])).sum(1).astype(np.uint8)).cuda()
        # five codes to a byte of a PTQ1_0 block: ceil(value * 256 / 243)
        c = np.random.default_rng(12).choice(3, p=[0.3, 0.4, 0.3], size=(65536, 5))
        v = c @ np.array([81, 27, 9, 3, 1])
        self.b3 = torch.from_numpy(((v * 256 + 242) // 243).astype(np.uint8)).cuda()

    def _bytes(self, lut, shape):
        at = torch.randint(0, 65536, (math.prod(shape),), generator=self.g, device="cuda", dtype=torch.int32)
        return lut.index_select(0, at).view(shape)

    def _scales(self, shape):
        s = torch.rand(shape, generator=self.g, device="cuda") * 0.04 + 0.01
        return s.to(torch.float16)

    def matrix(self, N, K):
        """(codes [N][K/4], scales [N][K/128] fp16) of the resident layout."""
        return self._bytes(self.t2, (N, K // 4)), self._scales((N, K // 128))

    def packed(self, N, K):
        """PTQ1_0 rows [N][K/128][28]."""
        b = torch.empty((N, K // 128, 28), dtype=torch.uint8, device="cuda")
        b[..., :26] = self._bytes(self.b3, (N, K // 128, 26))
        b[..., 26:] = self._scales((N, K // 128)).view(torch.uint8).view(N, K // 128, 2)
        return b

    def rows(self, M, n, rms=1.0):
        """Activations: normal values, each row with a size of its own."""
        x = torch.randn((M, n), generator=self.g, device="cuda")
        return x * torch.exp(0.5 * torch.randn((M, 1), generator=self.g, device="cuda")) * rms

    def norm(self, n):
        return 1.0 + 0.1 * torch.randn(n, generator=self.g, device="cuda")

    def signs(self, n):
        return torch.where(torch.rand(n, generator=self.g, device="cuda") < 0.5, -1.0, 1.0)

    def q8(self, M, K):
        """Quantized rows (q int8, d, s) as the prep leaves them."""
        x = self.rows(M, K).view(M, K // 32, 32)
        amax = x.abs().amax(-1)
        q = torch.round(x * (127.0 / amax)[..., None])
        d = (amax / 127.0).to(torch.float16).float()
        return q.to(torch.int8).view(M, K), d, q.sum(-1).to(torch.int32)

    def tokens(self, M, V):
        return torch.randint(0, V, (M,), generator=self.g, device="cuda", dtype=torch.int32)


def _zero(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _q8_out(hip, M, K):
    return hip.Q8Act(_zero(M, K, dtype=torch.int8), _zero(M, K // 32), _zero(M, K // 32, dtype=torch.int32))


def _block(n):
    """The transform's block for a width: the largest power of two up to 1024 that divides it."""
    return min(BLOCK, n & -n)


def _perm(c):
    return (32, c["n"] // 64, 2) if c["perm"] else (0, 0, 0)


def _hip():
    import btf_hip
    btf_hip.kernels_init(0)
    return btf_hip


def _layer_parts(src, c):
    """Weights, norms, signs and inputs of a stack of layers, in the order in which both users draw them."""
    E, F, Q = c["E"], c["F"], c["QKV"]
    layers = []
    for _ in range(c["layers"]):
        layers.append({"qkv": src.matrix(Q, E), "o": src.matrix(E, E), "gate": src.matrix(F, E),
                       "up": src.matrix(F, E), "down": src.matrix(E, F), "na": src.norm(E), "nf": src.norm(E),
                       "sq": src.signs(E), "so": src.signs(E), "sg": src.signs(E), "sd": src.signs(F)})
    V = c.get("V", 4096)
    M = c.get("M", 1)
    return {"layers": layers, "table": src.matrix(V, E), "emb_signs": src.signs(E), "tok": src.tokens(M, V),
            "att": src.rows(M, E, 2.0)}


def prepare(case, seed):
    hip = _hip()
    src = Source(seed)
    c, kind, G = case, case["kind"], hip.GemvMode
    st = {"kind": kind, "hip": hip, "c": c}
    if kind == "prep":
        n, M = c["n"], c["M"]
        hd, nk, rep = _perm(c)
        st.update(x=src.rows(M, n, 3.0), w=src.norm(n) if c["norm"] else None,
                  hx=hip.Hx(_block(n), hd, nk, rep, src.signs(n)), a=_q8_out(hip, M, n))
    elif kind in ("gemm", "packed", "fused"):
        M, K, N = c["M"], c["K"], c["N"]
        st["act"] = hip.Q8Act(*src.q8(M, K))
        st["y"] = [_zero(M, N) for _ in range(1 if c["mode"] == "swiglu" else c["segs"])]
        st["mode"] = {"store": G.kStore, "swiglu": G.kSwiglu}[c["mode"]]
        st["segs"] = []
        for i in range(c["segs"]):
            codes, scales = (src.packed(N, K), None) if kind == "packed" else src.matrix(N, K)
            y = st["y"][i] if i < len(st["y"]) else None
            st["segs"].append(hip.GemvSeg(codes, scales, N, y, N if y is not None else 0))
        if kind == "fused":
            st["out"] = _q8_out(hip, M, N)
    elif kind == "layers":
        _prepare_layers(hip, st, src, c)
    elif kind == "token":
        _prepare_token(hip, st, src, c)
    else:
        K, N = c["K"], c["N"]
        st["rows"] = src.packed(N, K).cpu().numpy()
        st["codes"], st["scales"] = _zero(N, K // 4, dtype=torch.uint8), _zero(N, K // 128, dtype=torch.int16)
        st["loader"] = hip.Loader(STAGING)
    return st


def _prepare_layers(hip, st, src, c):
    """The launches of a batched decode step, captured as a serving loop captures them."""
    M, E, F, Q, G = c["M"], c["E"], c["F"], c["QKV"], hip.GemvMode
    p = _layer_parts(src, c)
    x, qkv, h = _zero(M, E), _zero(M, Q), _zero(M, F)
    a, ah = _q8_out(hip, M, E), _q8_out(hip, M, F)
    be, bf = _block(E), _block(F)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = hip.Graph(stream)
    with graph:
        hip.launch_embed(*p["table"], p["tok"], M, E, hip.Hx(be, signs=p["emb_signs"]), x, stream)
        for L in p["layers"]:
            hip.launch_prep(x, E, M, E, L["na"], EPS, hip.Hx(be, signs=L["sq"]), None, 0, a, stream)
            hip.launch_gemv([hip.GemvSeg(*L["qkv"], Q, qkv, Q)], E, M, a, G.kStore, stream)
            hip.launch_prep(p["att"], E, M, E, None, 0.0, hip.Hx(be, signs=L["so"]), None, 0, a, stream)
            hip.launch_gemv([hip.GemvSeg(*L["o"], E, x, E)], E, M, a, G.kAdd, stream)
            hip.launch_prep(x, E, M, E, L["nf"], EPS, hip.Hx(be, signs=L["sg"]), None, 0, a, stream)
            hip.launch_gemv([hip.GemvSeg(*L["gate"], F, h, F), hip.GemvSeg(*L["up"], F, None, 0)], E, M, a, G.kSwiglu,
                            stream)
            hip.launch_prep(h, F, M, F, None, 0.0, hip.Hx(bf, signs=L["sd"]), None, 0, ah, stream)
            hip.launch_gemv([hip.GemvSeg(*L["down"], E, x, E)], F, M, ah, G.kAdd, stream)
    st.update(graph=graph, keep=(p, a, ah, stream), x=x, qkv=qkv, h=h)


def _prepare_token(hip, st, src, c):
    E, F, Q, V, G = c["E"], c["F"], c["QKV"], c["V"], hip.GemvMode
    p = _layer_parts(src, c)
    head, norm, signs = src.matrix(V, E), src.norm(E), src.signs(E)
    hx = lambda s: hip.Hx(block=BLOCK, signs=s)  # noqa: E731
    res, qkv, h, logits = _zero(E), _zero(Q), _zero(F), _zero(V)
    pick, pos = _zero(1, dtype=torch.int32), _zero(1, dtype=torch.int32)
    ops = [hip.StepEmbed(0, *p["table"], p["tok"], hx(p["emb_signs"]))]
    for L in p["layers"]:
        ops += [hip.StepGemv(G.kStore, E, Q, *L["qkv"], 0, 1, normw=L["na"], eps=EPS, hx=hx(L["sq"])),
                hip.StepGemv(G.kAdd, E, E, *L["o"], 2, 0, hx=hx(L["so"])),
                hip.StepGemv(G.kSwiglu, E, F, *L["gate"], 0, 3, *L["up"], normw=L["nf"], eps=EPS, hx=hx(L["sg"])),
                hip.StepGemv(G.kAdd, F, E, *L["down"], 3, 0, hx=hx(L["sd"]))]
    ops += [hip.StepGemv(G.kStore, E, V, *head, 0, 4, normw=norm, eps=EPS, hx=hx(signs)),
            hip.StepArgmax(4, pick, pos)]
    vecs = [hip.StepVec(E, res), hip.StepVec(Q, qkv), hip.StepVec(E, p["att"][0]), hip.StepVec(F, h),
            hip.StepVec(V, logits)]
    st.update(prog=hip.StepProgram(vecs, ops), res=res, logits=logits, pick=pick, keep=(p, head, pos))


def run(st):
    hip, c, kind = st["hip"], st["c"], st["kind"]
    s = torch.cuda.current_stream().cuda_stream
    if kind == "prep":
        a = st["a"]
        hip.launch_prep(st["x"], c["n"], c["M"], c["n"], st["w"], EPS, st["hx"], None, 0, a, s)
        return a.q, a.d, a.s
    if kind == "gemm":
        hip.launch_gemv(st["segs"], c["K"], c["M"], st["act"], st["mode"], s)
        return st["y"]
    if kind == "packed":
        hip.launch_gemv_ptq1_0(st["segs"], c["K"], c["M"], st["act"], st["mode"], s)
        return st["y"]
    if kind == "fused":
        o = st["out"]
        hip.launch_gemv_ex(st["segs"], c["K"], c["M"], st["act"], mode=st["mode"], out=o, stream=s)
        return st["y"][0], o.q, o.d, o.s
    if kind == "layers":
        st["graph"].stream = s
        st["graph"].launch()
        return st["x"], st["qkv"], st["h"]
    if kind == "token":
        st["prog"].launch(s)
        return {"logits": st["logits"], "residual": st["res"], "token": st["pick"]}
    st["loader"].upload_ptq1_0(st["rows"], c["N"], c["K"], st["codes"], st["scales"], s)
    st["loader"].finish()
    return st["codes"], st["scales"]


# ---- what a pass cannot do without ----
def _weights(N, K):
    return N * K // 4 + N * K // 64


def _q8_bytes(M, K):
    return M * (K + K // 4)


def work(case):
    c, kind = case, case["kind"]
    M = c.get("M", 1)
    if kind == "prep":
        n = c["n"]
        return {"bytes": 4 * M * n + _q8_bytes(M, n) + 4 * n * (2 if c["norm"] else 1),
                "flops": M * n * (int(math.log2(_block(n))) + 6)}
    if kind == "load":
        return {"bytes": c["N"] * c["K"] // 128 * 28 + _weights(c["N"], c["K"]), "flops": 0}
    if kind in ("gemm", "packed", "fused"):
        K, N, S = c["K"], c["N"], c["segs"]
        outs = 1 if c["mode"] == "swiglu" else S
        w = S * (N * K // 128 * 28 if kind == "packed" else _weights(N, K))
        return {"bytes": w + _q8_bytes(M, K) + 4 * M * N * outs + (_q8_bytes(M, N) if kind == "fused" else 0),
                "flops": 2 * M * K * N * S}
    E, F, Q = c["E"], c["F"], c["QKV"]
    w = _weights(Q + E + 2 * F, E) + _weights(E, F)
    # the residual, the attention's output and h enter and leave each product once
    rows = 4 * M * (Q + 2 * E + E + 2 * E + 2 * F) + 4 * (2 * E + 3 * E + F)
    got = {"bytes": c["layers"] * (w + rows) + M * (E // 4 + E // 64),
           "flops": 2 * M * c["layers"] * (E * (Q + E + 2 * F) + E * F)}
    if kind == "token":
        V = c["V"]
        got = {"bytes": got["bytes"] + _weights(V, E) + 4 * V, "flops": got["flops"] + 2 * E * V}
    return got


def tolerance(case):
    kind = case["kind"]
    if kind == "load":
        return "exact"
    if kind in ("gemm", "packed"):
        return {"rel": 1e-6, "max": 4e-5}  # 32-bit sums of up to 17408 products: 2e-7 off 64 bits at the most
    if kind in ("prep", "fused"):
        # a value at a tie of the quantizer, or an fp16 step of one block's scale, falls the other way
        return {"rel": 1e-4, "max": 2e-3, "differ": 2e-3}
    # Such ties, seen by every later layer: 0.003 off 64 bits after 2 layers, 0.03 after 64.
    return {"rel": 0.03, "max": 0.9} if kind == "token" else {"rel": 1e-2, "max": 0.3}


# ---- 64 bits, in plain torch ----
def _trits(codes):
    """codes [N][K/4] of the resident layout -> trits [N][K] (column e of a
    128-block: byte 8 (e / 32) + 4 ((e / 16) % 2) + e % 4, bits 2 ((e / 4) % 4))."""
    N, kb = codes.shape
    b = codes.view(N, kb // 32, 4, 2, 1, 4)
    sh = torch.arange(0, 8, 2, device=codes.device, dtype=torch.uint8).view(1, 1, 1, 1, 4, 1)
    return (((b >> sh) & 3).to(torch.int8) - 1).reshape(N, kb * 4)


def _packed_trits(rows):
    """PTQ1_0 rows [N][B][28] -> (trits [N][128 B], scales [N][B])."""
    N, B, _ = rows.shape
    v = rows[..., :26].to(torch.int32)
    digit = torch.stack([(((v * 3 ** n) & 255) * 3) >> 8 for n in range(5)], 2)  # [N][B][5][26]
    t = torch.cat([digit[:, :, :, :16].reshape(N, B, 80), digit[:, :, :, 16:24].reshape(N, B, 40),
                   digit[:, :, :4, 24:].reshape(N, B, 8)], 2)
    return (t.to(torch.int8) - 1).reshape(N, B * 128), rows[..., 26:].contiguous().view(torch.float16).view(N, B)


def _product(x, trits_of, N):
    """x [M][K] float64 times the rows' transpose, a slice of rows at a time."""
    out = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
    step = max(1, (1 << 27) // x.shape[1])
    for a in range(0, N, step):
        t, s = trits_of(a, min(N, a + step))
        w = (t.view(t.shape[0], -1, 128).double() * s.double()[..., None]).view(t.shape[0], -1)
        out[:, a:a + step] = x @ w.t().contiguous()
    return out


def _matmul(x, mat):
    codes, scales = mat
    return _product(x, lambda a, b: (_trits(codes[a:b]), scales[a:b]), codes.shape[0])


def _dequant(q, d):
    M, K = q.shape
    return (q.view(M, K // 32, 32).double() * d.double()[..., None]).view(M, K)


def _silu(g, u):
    return g / (1 + torch.exp(-g)) * u


def _fwht(x, block):
    shape, n = x.shape, 1
    x = x.reshape(-1, block)
    while n < block:
        v = x.view(x.shape[0], -1, 2, n)
        x = torch.stack([v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]], 2).reshape(-1, block)
        n *= 2
    return (x / math.sqrt(block)).view(shape)


def _quantize(x):
    """float64 rows -> (q, d) of their Q8."""
    b = x.view(x.shape[0], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    q = torch.round(torch.where(amax > 0, b * (127.0 / amax), torch.zeros_like(b))).view(x.shape)
    return q, (amax / 127.0)[..., 0].to(torch.float16).double()


def _prep(x, normw, block, signs, perm=(0, 0, 0)):
    x = x.double()
    if normw is not None:
        x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * normw.double()
    hd, nk, rep = perm
    if rep > 1:
        x = x.view(-1, rep, nk, hd).transpose(1, 2).reshape(x.shape)
    return _quantize(_fwht(x * signs.double(), block))


def _lookup(table, tok, signs, block):
    codes, scales = table
    at = tok.long()
    t, s = _trits(codes[at]), scales[at].double()
    x = (t.view(len(at), -1, 128).double() * s[..., None]).view(len(at), -1)
    return _fwht(x, block) * signs.double()


def _stack(p, be, bf):
    """The layers of _layer_parts: (residual, last qkv, last h)."""
    x = _lookup(p["table"], p["tok"], p["emb_signs"], be)
    qkv = h = None
    for L in p["layers"]:
        qkv = _matmul(_dequant(*_prep(x, L["na"], be, L["sq"])), L["qkv"])
        x = x + _matmul(_dequant(*_prep(p["att"], None, be, L["so"])), L["o"])
        a = _dequant(*_prep(x, L["nf"], be, L["sg"]))
        h = _silu(_matmul(a, L["gate"]), _matmul(a, L["up"]))
        x = x + _matmul(_dequant(*_prep(h, None, bf, L["sd"])), L["down"])
    return x, qkv, h


def exact(case, seed):
    c, kind = case, case["kind"]
    src = Source(seed)
    if kind == "load":
        return None  # bytes
    if kind == "prep":
        n, M = c["n"], c["M"]
        x, w = src.rows(M, n, 3.0), src.norm(n) if c["norm"] else None
        return None, _prep(x, w, _block(n), src.signs(n), _perm(c))[1], None
    if kind in ("gemm", "packed", "fused"):
        M, K, N = c["M"], c["K"], c["N"]
        q, d, _ = src.q8(M, K)
        x, y = _dequant(q, d), []
        for _ in range(c["segs"]):
            if kind == "packed":
                rows = src.packed(N, K)
                y.append(_product(x, lambda a, b: _packed_trits(rows[a:b]), N))
            else:
                y.append(_matmul(x, src.matrix(N, K)))
        if c["mode"] == "swiglu":
            y = [_silu(*y)]
        return (y[0], None, _quantize(y[0])[1], None) if kind == "fused" else y
    p = _layer_parts(src, c)
    if kind == "layers":
        return _stack(p, _block(c["E"]), _block(c["F"]))
    head, norm, signs = src.matrix(c["V"], c["E"]), src.norm(c["E"]), src.signs(c["E"])
    x, _, _ = _stack(p, BLOCK, BLOCK)
    logits = _matmul(_dequant(*_prep(x, norm, BLOCK, signs)), head)[0]
    return {"logits": logits, "residual": x[0], "token": None}
