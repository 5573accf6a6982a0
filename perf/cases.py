"""The work that a program on top of this library has it do, as timed cases.

Four kinds, each through the library's public entry points:

* ``gemm``: Y[N][M] = X[N][K] W^T (``okf_gemm``; N = 1 is ``okf_gemv``): one
  projection of a decode step (N = 1), of a speculative verify (N = 2..5) or
  of a prompt (any N past that, short and ragged ones included).
* ``ffn``: the FFN block of one decode step (``okf_ffn``: gate, up, SiLU, down).
* ``head``: the end of one decode step: RMSNorm of the last hidden state, the
  vocabulary projection and the argmax over it.
* ``embed``: the start of a prompt: embedding rows gathered by token id, then
  the residual add and RMSNorm over them.

Weights are GGUF blocks of random codes with scales in the range that the
repository's own synthetic weights use; activations are N(0, 1) in fp32.
"""
import json
import os

import torch

import chatokf_amd as ok

# formats of the models this library is used with (K-quant mixes, the 4-bit
# levels, the 2-bit grid format, the ternary one, 8-bit): the range of draw()
FORMATS = ("q2_0", "q4_k", "iq4_xs", "iq2_xxs", "q8_0", "iq4_nl", "q5_k", "q6_k", "q4_0")
# the fp16 scale fields of a block: (byte offset, low, high) each
SCALES = {
    "q8_0": ((0, 1e-3, 1e-2),),
    "q2_0": ((0, 0.01, 0.05),),
    "q4_0": ((0, 1e-3, 1e-2),),
    "iq4_nl": ((0, 1e-3, 1e-2),),
    "q4_k": ((0, 1e-3, 1e-2), (2, 1e-3, 1e-2)),
    "q5_k": ((0, 1e-3, 1e-2), (2, 1e-3, 1e-2)),
    "q6_k": ((208, 1e-4, 1e-3),),
    "iq4_xs": ((0, 1e-4, 1e-3),),
    "iq2_xxs": ((0, 1e-3, 1e-2),),
}
MAX_FLOPS = 2.0 * 17408 * 5120 * 512  # what a drawn case may cost
EPS = 1e-6


def listed():
    return [
        # an attention projection of a small model, one token: the smallest call
        {"name": "q8_0_matvec_2048", "kind": "gemm", "fmt": "q8_0", "M": 2048, "K": 2048, "N": 1},
        # the FFN of one decode step, 1.7B ternary model
        {"name": "q2_0_ffn_6144x2048", "kind": "ffn", "fmt": "q2_0", "H": 6144, "D": 2048},
        # the FFN of one decode step, 27B models in two of their formats
        {"name": "q4_k_ffn_17408x5120", "kind": "ffn", "fmt": "q4_k", "H": 17408, "D": 5120},
        {"name": "iq4_xs_ffn_17408x5120", "kind": "ffn", "fmt": "iq4_xs", "H": 17408, "D": 5120},
        # the verify pass of four drafted tokens, 27B model
        {"name": "iq2_xxs_verify4_17408x5120", "kind": "gemm", "fmt": "iq2_xxs", "M": 17408, "K": 5120, "N": 4},
        # the end of a decode step: norm, vocabulary projection, argmax (the most bytes)
        {"name": "q6_k_head_248320x5120", "kind": "head", "fmt": "q6_k", "M": 248320, "K": 5120},
        # a chat turn's few tokens on a 2B model
        {"name": "iq4_nl_prompt19_6144x2048", "kind": "gemm", "fmt": "iq4_nl", "M": 6144, "K": 2048, "N": 19},
        # a chat turn's sentences on a 27B model
        {"name": "q4_k_prompt101_17408x5120", "kind": "gemm", "fmt": "q4_k", "M": 17408, "K": 5120, "N": 101},
        # whole prompt chunks: the 27B FFN's up projection (the most flops) and
        # a ragged last chunk of its down projection, the ternary model's up projection
        {"name": "q4_k_pp512_17408x5120", "kind": "gemm", "fmt": "q4_k", "M": 17408, "K": 5120, "N": 512},
        {"name": "iq4_xs_pp333_5120x17408", "kind": "gemm", "fmt": "iq4_xs", "M": 5120, "K": 17408, "N": 333},
        {"name": "q2_0_pp512_6144x2048", "kind": "gemm", "fmt": "q2_0", "M": 6144, "K": 2048, "N": 512},
        # the start of a prompt chunk: embedding rows, residual add and norm
        {"name": "q4_k_embed_norm_512x5120", "kind": "embed", "fmt": "q4_k", "M": 248320, "K": 5120, "N": 512},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("gemm1", "gemm1", "verify", "prompt", "prompt", "prompt", "ffn", "ffn", "head", "embed"))
    fmt = rng.choice(FORMATS)
    D = max(4, _log(rng, 4, 20)) * 256          # a hidden width: 1024 .. 5120
    H = max(D // 256 + 1, int(round(D / 256 * rng.uniform(2.0, 3.5)))) * 256  # an FFN width
    if kind == "ffn":
        return {"kind": "ffn", "fmt": fmt, "H": H, "D": D}
    if kind == "head":
        return {"kind": "head", "fmt": fmt, "M": _log(rng, 16000, 248320), "K": D}
    if kind == "embed":
        return {"kind": "embed", "fmt": fmt, "M": _log(rng, 16000, 248320), "K": D, "N": _log(rng, 1, 512)}
    M, K = rng.choice(((H, D), (D, H), (D, D)))
    if rng.random() < 0.25:                     # a ragged number of rows
        M = max(1, M - rng.randrange(1, 200))
    N = 1 if kind == "gemm1" else rng.randint(2, 5) if kind == "verify" else _log(rng, 6, 1024)
    N = max(1, min(N, int(MAX_FLOPS / (2.0 * M * K))))
    return {"kind": "gemm", "fmt": fmt, "M": M, "K": K, "N": N}


_ENC = None


def _enc():
    """One context for the process, as a program keeps it."""
    global _ENC
    if _ENC is None:
        _ENC = ok.Enc(0)
    return _ENC


def _blocks(fmt, M, K, gen):
    """M rows of K random weights as GGUF blocks on the GPU: uint8 [M * K / block][block bytes]."""
    t = ok.BY_NAME[fmt]
    nb = M * (K // ok.block_elems(t))
    bb = ok.row_bytes(t, ok.block_elems(t))
    b = torch.empty((nb, bb), dtype=torch.uint8, device="cuda")
    b.view(-1).random_(0, 256, generator=gen)
    if fmt == "q2_0":   # ternary: the code 3 is not in use
        pairs = torch.randint(0, 81, (nb, bb - 2), device="cuda", generator=gen, dtype=torch.int32)
        b[:, 2:] = (pairs % 3 | (pairs // 3 % 3) << 2 | (pairs // 9 % 3) << 4 | (pairs // 27) << 6).to(torch.uint8)
    for off, lo, hi in SCALES[fmt]:
        d = (lo + (hi - lo) * torch.rand(nb, device="cuda", generator=gen)).half()
        b[:, off:off + 2] = d.view(torch.uint8).reshape(nb, 2)
    return b


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    k, fmt = case["kind"], case["fmt"]
    if k == "ffn":
        H, D = case["H"], case["D"]
        return {"gate": _blocks(fmt, H, D, gen), "up": _blocks(fmt, H, D, gen), "down": _blocks(fmt, D, H, gen),
                "x": torch.randn(D, device="cuda", generator=gen)}
    M, K = case["M"], case["K"]
    t = {"w": _blocks(fmt, M, K, gen)}
    if k == "gemm":
        t["x"] = torch.randn(case["N"], K, device="cuda", generator=gen)
    elif k == "head":
        t["x"] = torch.randn(1, K, device="cuda", generator=gen)
        t["norm"] = torch.rand(K, device="cuda", generator=gen) + 0.5
    else:
        t["ids"] = torch.randint(0, M, (case["N"],), device="cuda", generator=gen, dtype=torch.int32)
        t["r"] = torch.randn(case["N"], K, device="cuda", generator=gen)
        t["norm"] = torch.rand(K, device="cuda", generator=gen) + 0.5
    return t


def prepare(case, seed):
    enc, t, fmt = _enc(), _inputs(case, seed), ok.BY_NAME[case["fmt"]]
    s = {"case": case, "enc": enc, "t": t}
    new = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if case["kind"] == "ffn":
        H, D = case["H"], case["D"]
        s["w"] = [ok.QuantTensor(t["gate"], D, H, fmt).c(), ok.QuantTensor(t["up"], D, H, fmt).c(),
                  ok.QuantTensor(t["down"], H, D, fmt).c()]
        s["g"], s["u"], s["y"] = new(H), new(H), new(D)
        s["p"] = [v.data_ptr() for v in (t["x"], s["g"], s["u"], s["y"])]
        return s
    M, K = case["M"], case["K"]
    s["q"] = ok.QuantTensor(t["w"], K, M, fmt)
    s["w"] = s["q"].c()
    if case["kind"] == "gemm":
        s["y"] = new(case["N"], M)
        s["p"] = (t["x"].data_ptr(), s["y"].data_ptr())
    elif case["kind"] == "head":
        s["h"], s["y"] = new(1, K), new(1, M)
        s["tok"] = torch.empty(1, dtype=torch.int32, device="cuda")
    else:
        s["x"], s["y"] = new(case["N"], K), new(case["N"], K)
    return s


def run(s):
    case, enc, t = s["case"], s["enc"], s["t"]
    k = case["kind"]
    if k == "gemm":
        x, y = s["p"]
        if case["N"] == 1:
            enc.raw_gemv(s["w"], x, y)
        else:
            enc.raw_gemm(s["w"], x, case["N"], y)
        return s["y"]
    if k == "ffn":
        enc.raw_ffn(*s["w"], *s["p"])
        return {"g": s["g"], "u": s["u"], "y": s["y"]}
    if k == "head":
        enc.add_rmsnorm(t["x"], None, t["norm"], s["h"], case["K"], 1, EPS)
        enc.raw_gemv(s["w"], s["h"].data_ptr(), s["y"].data_ptr())
        enc.argmax_rows(s["y"], case["M"], 1, s["tok"])
        return {"logits": s["y"], "token": s["tok"]}
    enc.embed_batch(s["q"], t["ids"], case["N"], s["x"])
    enc.add_rmsnorm(s["x"], t["r"], t["norm"], s["y"], case["K"], case["N"], EPS)
    return {"x": s["x"], "y": s["y"]}


def _bytes(fmt, M, K):
    return M * ok.row_bytes(ok.BY_NAME[fmt], K)


def work(case):
    """Weights and inputs read once, outputs written once; one multiply and one add a weight and column."""
    k, fmt = case["kind"], case["fmt"]
    if k == "ffn":
        H, D = case["H"], case["D"]
        return {"bytes": 2 * _bytes(fmt, H, D) + _bytes(fmt, D, H) + 4 * (D + 2 * H + D), "flops": 6.0 * H * D}
    M, K = case["M"], case["K"]
    if k == "gemm":
        N = case["N"]
        return {"bytes": _bytes(fmt, M, K) + 4 * N * (K + M), "flops": 2.0 * M * K * N}
    if k == "head":
        return {"bytes": _bytes(fmt, M, K) + 4 * (2 * K + M + 1), "flops": 2.0 * M * K}
    N = case["N"]
    return {"bytes": _bytes(fmt, N, K) + 4 * (N + 3 * N * K + K), "flops": 5.0 * N * K}


def tolerance(case):
    if case["kind"] == "gemm" and case["N"] > 5:
        # weights and activations rounded to fp16 once, fp32 sums
        return {"rel": 1.5e-3, "max": 1.5e-2}
    if case["kind"] == "head":
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.01}
    # fp32 activations, fp32 sums
    return {"rel": 4e-6, "max": 4e-5}


# ---------------------------------------------------------------- 64 bits
def _tables():
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "golden",
                        "iq2xxs_tables.json")
    with open(path) as f:
        j = json.load(f)
    grid = torch.tensor([[(int(str(e), 0) >> (8 * i)) & 255 for i in range(8)] for e in j["iq2xxs_grid"]],
                        dtype=torch.float64, device="cuda")
    sign = torch.tensor([[-1.0 if (int(str(v), 0) >> i) & 1 else 1.0 for i in range(8)] for v in j["ksigns"]],
                        dtype=torch.float64, device="cuda")
    return grid, sign


_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _f16(b, off):
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _scale_min(s):
    """The eight 6-bit scales and mins of a Q4_K / Q5_K header's 12 bytes."""
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6) << 4], 1)
    return sc.double(), mn.double()


def _dequant(fmt, b):
    """Blocks [n][bytes] as float64 weights [n][weights]."""
    n = b.shape[0]
    i = lambda lo, hi: b[:, lo:hi].int()  # noqa: E731
    levels = torch.tensor(_LEVELS, dtype=torch.float64, device=b.device)
    if fmt == "q8_0":
        return _f16(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()
    if fmt == "q2_0":
        q = torch.stack([i(2, 34) >> v & 3 for v in (0, 2, 4, 6)], 2).reshape(n, 128)
        return _f16(b, 0) * (q - 1).double()
    if fmt in ("q4_0", "iq4_nl"):
        q = torch.cat([i(2, 18) & 15, i(2, 18) >> 4], 1)
        return _f16(b, 0) * (levels[q.long()] if fmt == "iq4_nl" else (q - 8).double())
    if fmt in ("q4_k", "q5_k"):
        sc, mn = _scale_min(i(4, 16))
        at = 16 if fmt == "q4_k" else 48
        qs = i(at, at + 128).reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if fmt == "q5_k":
            q = q + 16 * torch.stack([i(16, 48) >> v & 1 for v in range(8)], 1)
        w = (_f16(b, 0) * sc)[:, :, None] * q.double() - (_f16(b, 2) * mn)[:, :, None]
        return w.reshape(n, 256)
    if fmt == "q6_k":
        ql, qh = i(0, 128).reshape(n, 2, 2, 32), i(128, 192).reshape(n, 2, 32)
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        high = torch.stack([qh >> v & 3 for v in (0, 2, 4, 6)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        q = (low + 16 * high - 32).double().reshape(n, 2, 4, 2, 16)
        return (_f16(b, 208)[:, :, None, None, None] * sc * q).reshape(n, 256)
    if fmt == "iq4_xs":
        sh = i(2, 3) | i(3, 4) << 8
        ls = torch.stack([(b[:, 4 + v // 2].int() >> 4 * (v % 2) & 15) | (sh[:, 0] >> 2 * v & 3) << 4
                          for v in range(8)], 1)
        qs = i(8, 136).reshape(n, 8, 16)
        q = levels[torch.cat([qs & 15, qs >> 4], 2).long()]
        return ((_f16(b, 0) * (ls - 32).double())[:, :, None] * q).reshape(n, 256)
    grid, sign = _tables()  # iq2_xxs
    qs = b[:, 2:].reshape(n, 8, 8).long()
    a1 = qs[:, :, 4] | qs[:, :, 5] << 8 | qs[:, :, 6] << 16 | qs[:, :, 7] << 24
    db = _f16(b, 0) * (0.5 + (a1 >> 28).double()) * 0.25
    s = torch.stack([a1 >> 7 * v & 127 for v in range(4)], 2)
    return (db[:, :, None, None] * grid[qs[:, :, :4]] * sign[s]).reshape(n, 256)


def _product(fmt, blocks, M, K, X):
    """X [N][K] times the M x K weights, in float64, some rows at a time."""
    per = blocks.shape[0] // M
    out = torch.empty((X.shape[0], M), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // K)
    for r in range(0, M, step):
        m = min(step, M - r)
        W = _dequant(fmt, blocks[r * per:(r + m) * per]).reshape(m, K)
        out[:, r:r + m] = torch.mm(X, W.t().contiguous())
    return out


def _norm(x, w):
    return x * w.double() / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)


def exact(case, seed):
    t, fmt, k = _inputs(case, seed), case["fmt"], case["kind"]
    if k == "ffn":
        H, D = case["H"], case["D"]
        x = t["x"].double()[None]
        g, u = _product(fmt, t["gate"], H, D, x), _product(fmt, t["up"], H, D, x)
        g = g / (1 + torch.exp(-g)) * u
        return {"g": g[0], "u": u[0], "y": _product(fmt, t["down"], D, H, g)[0]}
    M, K = case["M"], case["K"]
    if k == "gemm":
        return _product(fmt, t["w"], M, K, t["x"].double())
    if k == "head":
        return {"logits": _product(fmt, t["w"], M, K, _norm(t["x"].double(), t["norm"])), "token": None}
    per = t["w"].shape[0] // M
    rows = t["w"].reshape(M, per, -1)[t["ids"].long()].reshape(case["N"] * per, -1)
    x = _dequant(fmt, rows).reshape(case["N"], K) + t["r"].double()
    return {"x": x, "y": _norm(x, t["norm"])}
