"""The work a program has this package do, as cases that can be timed and compared.

A case is a dict of plain values; `kind` names the entry points it goes through:

  gemv     Weight.gemv: one matrix, 1 to 16 activation rows (a decode step)
  layers   gemv_multi_fused: decoder layers of one or two sequences, every product of a layer in order
  gemm     Weight.gemm: one matrix, a prompt's rows (prefill)
  mlp      mlp_step: the SwiGLU feed-forward of a layer
  moe      moe_router + RoutedMoe (routing on the device) or moe_ffn (routing lists on the host)
  encode   quantize a tensor on the device
  decode   expand a payload to fp32 on the device

listed() has the sizes of one 8-billion-parameter decoder (hidden 4096, feed-forward 14336, k / v projections of 1024
rows, a vocabulary of 128256) and of a layer of eight such feed-forward experts; draw() gives cases of the same ranges.
Weights are N(0, 0.02), or Laplace(0, 0.015) for the low-bit superblock formats, quantized by the package's encoder;
activations are N(0, 1).
"""
import importlib
import math

import torch

tfq = importlib.import_module("transformers-fusion_amd")

TILED = ("B32S4", "B32S8", "Q_G_4", "Q_G_8", "Q_8", "Q_G_3", "Q_G_2", "SB256A3", "SB256A2")
PAIRED = ("B32S4", "B32S8", "Q_G_4", "Q_G_8")  # formats of the fused layer, the feed-forward and the experts
WIRE = ("Q_4", "Q_G_6")                        # formats that are multiplied from their wire layout
LOW_BIT = ("Q_G_2", "SB256A3", "SB256A2")
LINE_GRID = ("Q_8", "Q_G_8")                   # companded grid, multiplied as the line that fits it
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # the smallest product of a decode step: one k projection for one sequence; launch latency counts
        {"name": "k_proj", "kind": "gemv", "fmt": "B32S4", "N": 1024, "K": 4096, "B": 1, "dtype": "bf16"},
        # a 3-bit superblock matrix for eight sequences at once
        {"name": "gate_lowbit_batch8", "kind": "gemv", "fmt": "SB256A3", "N": 14336, "K": 4096, "B": 8, "dtype": "bf16"},
        # the projection onto the vocabulary, kept at six bits, for one sequence: the longest single weight stream
        {"name": "vocabulary_6bit", "kind": "gemv", "fmt": "Q_G_6", "N": 128256, "K": 4096, "B": 1, "dtype": "bf16"},
        # the tall projection of a layer for sixteen sequences
        {"name": "down_batch16", "kind": "gemv", "fmt": "Q_G_4", "N": 4096, "K": 14336, "B": 16, "dtype": "bf16"},
        # one token through decoder layers: norm + q/k/v, o + residual, norm + gate/up, down + residual
        {"name": "decoder_layers", "kind": "layers", "fmt": "B32S4", "layers": 4, "D": 4096, "KV": 1024, "F": 14336, "B": 1},
        # a prompt of 2048 tokens through the wide projection
        {"name": "prefill_2048", "kind": "gemm", "fmt": "B32S4", "N": 14336, "K": 4096, "M": 2048, "dtype": "bf16"},
        # a short ragged prompt whose activations stay fp32, as in the engine this package serves
        {"name": "prefill_ragged_f32", "kind": "gemm", "fmt": "Q_G_4", "N": 4096, "K": 14336, "M": 333, "dtype": "f32"},
        # a prompt through a matrix of the plain 4-bit lattice, which is kept in wire layout
        {"name": "prefill_lattice", "kind": "gemm", "fmt": "Q_4", "N": 14336, "K": 4096, "M": 512, "dtype": "bf16"},
        # the feed-forward of a layer for three sequences with fp32 activations
        {"name": "mlp_f32", "kind": "mlp", "fmt": "Q_G_8", "D": 4096, "F": 14336, "B": 3, "dtype": "f32"},
        # a layer of eight experts, two per token, for a batch of sixteen tokens, router included
        {"name": "experts_16", "kind": "moe", "fmt": "B32S4", "D": 4096, "F": 14336, "E": 8, "k": 2, "T": 16, "routed": True},
        # quantizing a checkpoint's matrix with the iterative affine encoder
        {"name": "encode_affine", "kind": "encode", "fmt": "Q_G_4", "n": 14336 * 4096},
        # expanding a stored tensor to fp32
        {"name": "decode_affine", "kind": "decode", "fmt": "Q_G_4", "n": 14336 * 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, hi=16384):
    """Rows of a matrix: half of them whole tiles of 64, half any number."""
    n = _log(rng, 256, hi)
    return max(64, n // 64 * 64) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "gemv", "layers", "gemm", "gemm", "gemm", "mlp", "moe", "encode", "decode"))
    if kind == "gemv":
        fmt = rng.choice(TILED + WIRE)
        return {"kind": kind, "fmt": fmt, "N": _rows(rng), "K": 256 * _log(rng, 4, 64), "B": _log(rng, 1, 16),
                "dtype": rng.choice(("bf16", "bf16", "bf16", "f32"))}
    if kind == "layers":
        D = 256 * _log(rng, 4, 16)
        return {"kind": kind, "fmt": rng.choice(PAIRED), "layers": rng.randint(1, 4), "D": D, "KV": max(128, D // rng.choice((1, 4, 8))),
                "F": 256 * _log(rng, D // 128, D // 73), "B": rng.choice((1, 1, 2))}
    if kind == "gemm":
        fmt = rng.choice(TILED + TILED + WIRE)
        dtype = rng.choice(("bf16", "bf16", "f32"))
        wide = fmt in TILED and fmt not in LOW_BIT and dtype == "bf16"
        K = 256 * _log(rng, 4, 56)
        return {"kind": kind, "fmt": fmt, "N": _rows(rng, min(16384, 14336 * 4096 // K)), "K": K, "M": _log(rng, 17, 2048 if wide else 512),
                "dtype": dtype}
    if kind == "mlp":
        D = 256 * _log(rng, 4, 16)
        return {"kind": kind, "fmt": rng.choice(PAIRED), "D": D, "F": 256 * _log(rng, D // 128, D // 73), "B": _log(rng, 1, 256),
                "dtype": rng.choice(("bf16", "f32"))}
    if kind == "moe":
        D = 256 * _log(rng, 4, 16)
        routed = rng.random() < 0.5
        return {"kind": kind, "fmt": rng.choice(PAIRED), "D": D, "F": 256 * _log(rng, D // 256, D // 73), "E": rng.choice((4, 8, 8, 16)),
                "k": rng.choice((1, 2, 2, 4)), "T": _log(rng, 1, 64 if routed else 128), "routed": routed}
    fmt = rng.choice(TILED + WIRE)
    n = _log(rng, 1 << 16, 14336 * 4096)
    return {"kind": kind, "fmt": fmt, "n": n // 32 * 32 if fmt in ("B32S4", "B32S8") else n}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _values(fmt, n, g):
    if fmt in ("SB256A3", "SB256A2"):
        u = torch.rand(n, device="cuda", generator=g) - 0.5
        return u.sign() * torch.log1p(u.abs().mul_(-2.0).clamp_(min=-0.9999999)) * -0.015
    return torch.randn(n, device="cuda", generator=g).mul_(0.02)


def _matrix(fmt, N, K, g):
    return tfq.Weight(fmt, N, K, tfq.encode(fmt, _values(fmt, N * K, g)))


def _acts(rows, K, dtype, g):
    return torch.randn(rows, K, device="cuda", generator=g).to(DTYPES[dtype])


def prepare(case, seed):
    tfq.init(0)
    g = _gen(seed)
    kind, fmt = case["kind"], case["fmt"]
    s = dict(case)
    if kind in ("gemv", "gemm"):
        s["w"] = _matrix(fmt, case["N"], case["K"], g)
        s["x"] = _acts(case["B"] if kind == "gemv" else case["M"], case["K"], case["dtype"], g)
    elif kind == "layers":
        D, KV, F, B = case["D"], case["KV"], case["F"], case["B"]
        s["stack"] = []
        for _ in range(case["layers"]):
            ly = {n: _matrix(fmt, r, k, g) for n, r, k in (("q", D, D), ("k", KV, D), ("v", KV, D), ("o", D, D), ("gate", F, D),
                                                           ("up", F, D), ("down", D, F))}
            for n in ("norm1", "norm2"):
                ly[n] = torch.randn(D, device="cuda", generator=g).mul_(0.1)
            s["stack"].append(ly)
        s["embedding"] = torch.randn(B, D, device="cuda", generator=g)
        s["h"] = torch.empty(B, D, device="cuda")
        s["qkv"] = [torch.empty(B, n, device="cuda") for n in (D, KV, KV)]
        s["mid"] = torch.empty(B, F, device="cuda", dtype=torch.bfloat16)
    elif kind == "mlp":
        D, F = case["D"], case["F"]
        s["gate"], s["up"], s["down"] = (_matrix(fmt, n, k, g) for n, k in ((F, D), (F, D), (D, F)))
        s["x"] = _acts(case["B"], D, case["dtype"], g)
    elif kind == "moe":
        D, F, E, T, k = case["D"], case["F"], case["E"], case["T"], case["k"]
        s["gate"], s["up"], s["down"] = ([_matrix(fmt, n, c, g) for _ in range(E)] for n, c in ((F, D), (F, D), (D, F)))
        s["x"] = _acts(T, D, "bf16", g)
        s["router"] = torch.randn(E, D, device="cuda", generator=g).mul_(D ** -0.5)
        if case["routed"]:
            s["ffn"] = tfq.RoutedMoe(s["gate"], s["up"], s["down"], T, k)
            s["y"] = torch.empty(T, D, device="cuda")
        else:
            _, _, idx, wts = tfq.moe_router(s["x"], s["router"], k)
            s["idx"], s["wts"] = idx.cpu().numpy().astype("int64"), wts.cpu().numpy()
    elif kind == "encode":
        s["values"] = _values(fmt, case["n"], g)
    elif kind == "decode":
        s["payload"] = tfq.encode(fmt, _values(fmt, case["n"], g))
    return s


def run(s):
    kind = s["kind"]
    if kind == "gemv":
        return s["w"].gemv(s["x"])
    if kind == "gemm":
        return s["w"].gemm(s["x"], out_dtype=s["x"].dtype)
    if kind == "layers":
        h, mid = s["h"], s["mid"]
        q, k, v = s["qkv"]
        h.copy_(s["embedding"])
        for ly in s["stack"]:
            tfq.gemv_multi_fused([ly["q"], ly["k"], ly["v"]], h, [q, k, v], rmsnorm=ly["norm1"])
            # attention itself is outside the package; the o projection takes q
            tfq.gemv_multi_fused([ly["o"]], q, [h], accumulate=True)
            tfq.gemv_multi_fused([ly["gate"], ly["up"]], h, [mid], rmsnorm=ly["norm2"], pair_swiglu=True)
            tfq.gemv_multi_fused([ly["down"]], mid, [h], accumulate=True)
        return h, q, k, v, mid
    if kind == "mlp":
        return tfq.mlp_step(s["gate"], s["up"], s["down"], s["x"])
    if kind == "moe":
        if s["routed"]:
            logits, probs, idx, wts = tfq.moe_router(s["x"], s["router"], s["k"])
            return s["ffn"](idx, wts, s["x"], s["y"]), logits, probs, idx, wts
        return tfq.moe_ffn(s["gate"], s["up"], s["down"], s["idx"], s["wts"], s["x"])
    if kind == "encode":
        return tfq.encode(s["fmt"], s["values"])
    return tfq.decode(s["fmt"], s["payload"], s["n"])


def _packed(fmt, n):
    return n // 256 * tfq.block_bytes(fmt) + (tfq.block_bytes(fmt, n % 256) if n % 256 else 0)


def work(case):
    kind, fmt = case["kind"], case["fmt"]
    size = {"bf16": 2, "f32": 4}.get(case.get("dtype"), 4)
    if kind in ("gemv", "gemm"):
        N, K, rows = case["N"], case["K"], case["B"] if kind == "gemv" else case["M"]
        return {"bytes": _packed(fmt, N * K) + rows * K * size + rows * N * (4 if kind == "gemv" else size), "flops": 2.0 * rows * N * K}
    if kind == "layers":
        D, KV, F, B, L = case["D"], case["KV"], case["F"], case["B"], case["layers"]
        weights = 2 * D * D + 2 * D * KV + 3 * D * F
        return {"bytes": L * (_packed(fmt, weights) + 8 * D) + B * 4 * (2 * D + D + 2 * KV) + B * 2 * F, "flops": 2.0 * B * L * weights}
    if kind == "mlp":
        D, F, B = case["D"], case["F"], case["B"]
        return {"bytes": _packed(fmt, 3 * D * F) + B * D * (size + 4), "flops": 6.0 * B * D * F}
    if kind == "moe":
        D, F, E, T, k = case["D"], case["F"], case["E"], case["T"], case["k"]
        active = E * (1.0 - (1.0 - k / E) ** T)  # experts that at least one token goes to, on average
        return {"bytes": active * _packed(fmt, 3 * D * F) + T * D * 6 + (E * D * 4 if case["routed"] else 0), "flops": 6.0 * T * k * D * F}
    return {"bytes": _packed(fmt, case["n"]) + 4 * case["n"], "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("encode", "decode"):
        return "exact"
    if kind in ("gemv", "gemm", "mlp") and case["dtype"] == "f32":
        # fp32 activations and fp32 sums; the line is within 7.5e-5 of the companded grid
        return {"rel": 3e-4 if case["fmt"] in LINE_GRID else 5e-5}
    if kind == "layers":  # bf16 feed-forward activations, carried through the layers
        return {"rel": 1e-2}
    if kind == "moe":  # a routing decision may fall the other way where two logits agree to fp32 rounding
        return {"rel": 1e-2, "differ": 1e-3}
    return {"rel": 5e-3}  # bf16 activations
