"""The work that a model's forward pass has the quantized-matmul operators do.

A case is one piece of a transformer layer, called through forge_amd.ops as a
program that holds its weights on the device calls it:

  layer    fused_qkv, the output projection, ffn_up_fused, ffn_down_residual
  ffn      ffn_up_fused, then ffn_down_residual (gate and up in one format,
           down in another, as a mixed K-quant file has it)
  matmul   one projection: matmul_transB (GGUF bytes) or gemv_packed
  dequant  dequantize_weight, the fp32 copy of a weight

Sizes: a small model's layer (hidden 2048, FFN 5632), 7B and 8B layers (3584 /
18944 and 4096 / 14336) and the 152064-row head.  M is the number of tokens in
the call: 1 decodes, 2 .. 32 verifies a draft or serves a small batch, more is
a prompt.  `layout` is "gguf" for the file's bytes as they are or "packed" for
the aligned layout (batch 1 only).
"""
from __future__ import annotations

import math

import torch

from forge_amd import formats as F
from forge_amd import ops

LARGEST = dict(M=1999, hidden=3584, ffn=18944)


def listed():
    return [
        # one token through a small model's layer: launches and latency
        dict(name="decode layer, small model", op="layer", layout="gguf", fmt="q4_0", down="q4_0",
             M=1, hidden=2048, kv=256, ffn=5632),
        # one token through a 7B FFN of a mixed Q4_K / Q6_K file
        dict(name="decode ffn, 7b", op="ffn", layout="gguf", fmt="q4_k", down="q6_k",
             M=1, hidden=3584, ffn=18944),
        # one token through an 8B Q8_0 layer repacked at load time
        dict(name="decode layer, 8b aligned", op="layer", layout="packed", fmt="q8_0", down="q8_0",
             M=1, hidden=4096, kv=1024, ffn=14336),
        # the vocabulary projection of every decoded token
        dict(name="decode head, aligned", op="matmul", layout="packed", fmt="q6_k",
             M=1, N=152064, K=3584, bias=False),
        # verifying three drafted tokens and the one after them
        dict(name="verify 4, ffn 7b", op="ffn", layout="gguf", fmt="q4_0", down="q4_0",
             M=4, hidden=3584, ffn=18944),
        # eight requests decoding together
        dict(name="batch 8, layer 8b", op="layer", layout="gguf", fmt="q4_k", down="q6_k",
             M=8, hidden=4096, kv=1024, ffn=14336),
        # the vocabulary projection of sixteen requests
        dict(name="batch 16, head", op="matmul", layout="gguf", fmt="q6_k",
             M=16, N=152064, K=3584, bias=False),
        # the largest decode batch of the batched path
        dict(name="batch 32, ffn 8b", op="ffn", layout="gguf", fmt="q4_k", down="q6_k",
             M=32, hidden=4096, ffn=14336),
        # a short chat turn, its token count as it comes
        dict(name="prompt 77, ffn 8b", op="ffn", layout="gguf", fmt="q5_k", down="q5_k",
             M=77, hidden=4096, ffn=14336),
        # one prompt chunk through a whole layer
        dict(name="prompt 512, layer 8b", op="layer", layout="gguf", fmt="q8_0", down="q8_0",
             M=512, hidden=4096, kv=1024, ffn=14336),
        # a long prompt in one call, a ragged token count
        dict(name="prompt 1999, ffn 7b", op="ffn", layout="gguf", fmt="q4_k", down="q6_k", **LARGEST),
        # an fp32 copy of a weight, for a layer that has no quantized kernel
        dict(name="dequantize, ffn 8b", op="dequant", layout="gguf", fmt="q4_k", N=14336, K=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a format by how common it is in model files, a token
    count from 1 to 1999, sizes from a small model's to the head's."""
    op = rng.choice(["layer", "ffn", "ffn", "matmul", "matmul", "matmul", "dequant"])
    fmt = rng.choice(["q4_k"] * 4 + ["q8_0"] * 3 + ["q4_0"] * 3 + ["q6_k"] * 2 +
                     ["q5_k"] * 2 + ["q4_1", "q5_0", "q5_1", "q3_k", "iq4_nl"])
    down = "q6_k" if fmt in ("q4_k", "q5_k") and rng.random() < 0.6 else fmt
    # decode, a small batch and a prompt are about as common
    M = rng.choice([1, rng.randint(2, 32), _log_int(rng, 33, 1999)])
    packed = M == 1 and F.fmt(fmt).dtype in F.PACKED and F.fmt(down).dtype in F.PACKED and \
        rng.random() < 0.5
    layout = "packed" if packed else "gguf"
    small_blocks = F.fmt(fmt).block_elems == 32 and F.fmt(down).block_elems == 32 and not packed

    def width(lo, hi):  # an input width: whole blocks of 256, or of 32 where the format has them
        unit = 32 if small_blocks and rng.random() < 0.25 else 256
        return max(unit, _log_int(rng, lo, hi) // unit * unit)

    def rows(lo, hi):  # an output width: usually round, sometimes odd
        n = _log_int(rng, lo, hi)
        return n | 1 if rng.random() < 0.3 else max(32, n // 32 * 32)

    if op == "dequant":
        return dict(op=op, layout="gguf", fmt=fmt, N=rows(256, 32000), K=width(1024, 8192))
    if op == "matmul":
        head = M <= 16 and rng.random() < 0.3
        N = rows(32000, 152064) if head else rows(256, 18944)
        K = width(1024, 4096) if head else width(1024, 18944)
        return dict(op=op, layout=layout, fmt=fmt, M=M, N=N, K=K, bias=rng.random() < 0.4)
    hidden, ffn = width(1024, 4096), width(2048, 14336)
    if op == "ffn":
        return dict(op=op, layout=layout, fmt=fmt, down=down, M=M, hidden=hidden, ffn=ffn)
    return dict(op=op, layout=layout, fmt=fmt, down=down, M=M, hidden=hidden,
                kv=max(64, hidden // rng.choice([1, 4, 8]) // 32 * 32), ffn=ffn)


# ---------------------------------------------------------------- matrices
def _matrices(case):
    """name -> (format, N, K) of the case's weights, in the order of its calls."""
    if case["op"] in ("matmul", "dequant"):
        return {"w": (case["fmt"], case["N"], case["K"])}
    h, f = case["hidden"], case["ffn"]
    out = {}
    if case["op"] == "layer":
        out = {"q": (case["fmt"], h, h), "k": (case["fmt"], case["kv"], h),
               "v": (case["fmt"], case["kv"], h), "o": (case["fmt"], h, h)}
    out.update(gate=(case["fmt"], f, h), up=(case["fmt"], f, h), down=(case["down"], h, f))
    return out


# Root mean square of a format's integer codes (times its integer sub-scales)
# as _blocks draws them: the scale that gives weights of variance 1 / K.
_CODE_RMS = {"q4_0": 4.6, "q4_1": 4.6, "q8_0": 73.0, "q5_0": 9.2, "q5_1": 9.2, "iq4_nl": 69.0,
             "q4_k": 4.6 * 42, "q5_k": 9.2 * 42, "q6_k": 18.5 * 84, "q3_k": 2.3 * 19}


def _blocks(fmt, N, K, g, dev):
    """Random GGUF blocks [N * K / block][bytes]: uniform codes, fp16 scales
    of the size that trained projections have (weights of about zero mean and
    variance 1 / K)."""
    f = F.fmt(fmt)
    n = N * (K // f.block_elems)
    b = torch.randint(0, 256, (n, f.block_bytes), dtype=torch.uint8, device=dev, generator=g)

    def put(at, v):
        b[:, at:at + 2] = v.to(torch.float16).view(torch.uint8).view(n, 2)

    def six(lo, hi):  # 6-bit sub-scales of a super-block's eight sub-blocks
        return torch.randint(lo, hi, (n, 8), dtype=torch.int32, device=dev, generator=g)

    d = (0.6 + 0.8 * torch.rand(n, device=dev, generator=g)) / (math.sqrt(K) * _CODE_RMS[fmt])
    if fmt in ("q4_0", "q5_0", "iq4_nl"):
        put(0, d)
    elif fmt == "q8_0":
        put(0, d)
        b[:, 2:] = torch.where(b[:, 2:] == 128, torch.zeros_like(b[:, 2:]), b[:, 2:])
    elif fmt in ("q4_1", "q5_1"):
        put(0, d)
        put(2, d * (-7.5 if fmt == "q4_1" else -15.5))
    elif fmt in ("q4_k", "q5_k"):
        put(0, d)
        put(2, d * (7.5 if fmt == "q4_k" else 15.5))
        sc = six(20, 64)
        m = (sc + six(-3, 4)).clamp(0, 63)
        s = torch.empty((n, 12), dtype=torch.int32, device=dev)
        s[:, 0:4] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        s[:, 4:8] = m[:, :4] | ((m[:, 4:] >> 4) << 6)
        s[:, 8:12] = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
        b[:, 4:16] = s.to(torch.uint8)
    elif fmt == "q6_k":
        put(208, d)
        sc = torch.randint(32, 129, (n, 16), dtype=torch.int32, device=dev, generator=g)
        sign = torch.randint(0, 2, (n, 16), dtype=torch.int32, device=dev, generator=g)
        b[:, 192:208] = torch.where(sign == 1, -sc, sc.clamp(max=127)).to(torch.int8).view(torch.uint8)
    elif fmt == "q3_k":
        put(108, d)
    return b


def _f16(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequant64(fmt, b, N, K):
    """The block formats' definitions in plain torch and 64 bits, [N, K]."""
    def nibbles(q):
        return torch.cat([q & 15, q >> 4], 1).to(torch.float64)

    def fifth(at):
        bits = torch.arange(8, dtype=torch.uint8, device=b.device)
        return ((b[:, at:at + 4, None] >> bits) & 1).reshape(-1, 32).to(torch.float64) * 16

    def six(s):  # (scales, minima) of the eight sub-blocks
        s = s.to(torch.int32)
        lo, hi, mix = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        return (torch.cat([lo & 63, (mix & 15) | ((lo >> 6) << 4)], 1).to(torch.float64),
                torch.cat([hi & 63, (mix >> 4) | ((hi >> 6) << 4)], 1).to(torch.float64))

    if fmt == "q4_0":
        w = _f16(b, 0) * (nibbles(b[:, 2:]) - 8)
    elif fmt == "q4_1":
        w = _f16(b, 0) * nibbles(b[:, 4:]) + _f16(b, 2)
    elif fmt == "q5_0":
        w = _f16(b, 0) * (nibbles(b[:, 6:]) + fifth(2) - 16)
    elif fmt == "q5_1":
        w = _f16(b, 0) * (nibbles(b[:, 8:]) + fifth(4)) + _f16(b, 2)
    elif fmt == "q8_0":
        w = _f16(b, 0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif fmt == "iq4_nl":
        table = torch.tensor(_IQ4, dtype=torch.float64, device=b.device)
        w = _f16(b, 0) * table[nibbles(b[:, 2:]).to(torch.int64)]
    elif fmt in ("q4_k", "q5_k"):
        sc, m = six(b[:, 4:16])
        qs = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).to(torch.float64)
        if fmt == "q5_k":
            bits = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(1, 8, 1)
            q = q + ((b[:, None, 16:48] >> bits) & 1).to(torch.float64) * 16
        w = (_f16(b, 0) * sc)[:, :, None] * q - (_f16(b, 2) * m)[:, :, None]
    elif fmt == "q6_k":
        ql = b[:, 0:128].reshape(-1, 2, 1, 2, 32)
        qh = b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2).reshape(-1, 2, 4, 32)
        shift = torch.arange(0, 8, 2, dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)).to(torch.float64) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        w = (_f16(b, 208) * sc)[:, :, None] * q.reshape(-1, 16, 16)
    elif fmt == "q3_k":
        s = b[:, 96:108].to(torch.int32)
        low = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        high = torch.cat([(s[:, 8:12] >> (2 * i)) & 3 for i in range(4)], 1)
        sc = (low | (high << 4)).to(torch.float64) - 32
        shift = torch.arange(0, 8, 2, dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
        q = ((b[:, 32:96].reshape(-1, 2, 1, 32) >> shift) & 3).to(torch.float64)
        bit = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(1, 2, 4, 1)
        q = q + 4 * ((b[:, :32].reshape(-1, 1, 1, 32) >> bit) & 1).to(torch.float64) - 4
        w = (_f16(b, 108) * sc)[:, :, None] * q.reshape(-1, 16, 16)
    return w.reshape(N, K)


def _inputs(case, seed):
    """Blocks of every weight, the activations (one normalized vector per
    token: unit variance, a few outlier channels) and the residual or bias."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    mats = _matrices(case)
    blocks = {k: _blocks(fmt, N, K, g, dev) for k, (fmt, N, K) in mats.items()}
    if case["op"] == "dequant":
        return mats, blocks, None, None, None
    M, K = case["M"], next(iter(mats.values()))[2]

    def tokens(width):
        x = torch.randn((M, width), device=dev, generator=g)
        at = torch.randint(0, width, (max(1, width // 256),), device=dev, generator=g)
        x[:, at] *= 8
        return x

    x = tokens(K)
    attn = tokens(case["hidden"]) if case["op"] == "layer" else None
    if case["op"] == "matmul":
        extra = torch.randn((case["N"],), device=dev, generator=g) if case["bias"] else None
    else:
        extra = torch.randn((M, case["hidden"]), device=dev, generator=g)
    return mats, blocks, x, attn, extra


def prepare(case, seed):
    mats, blocks, x, attn, extra = _inputs(case, seed)
    w = {k: ops.QWeight(blocks[k].reshape(-1), F.fmt(fmt).dtype, N, K)
         for k, (fmt, N, K) in mats.items()}
    if case["layout"] == "packed":
        w = {k: ops.pack_weights(v) for k, v in w.items()}
    return dict(op=case["op"], packed=case["layout"] == "packed", w=w, x=x, attn=attn, extra=extra)


def run(state):
    op, w, x, extra = state["op"], state["w"], state["x"], state["extra"]
    if op == "dequant":
        return ops.dequantize_weight(w["w"])
    if state["packed"]:
        if op == "matmul":
            return ops.gemv_packed(x, w["w"], extra)
        out = []
        if op == "layer":
            out = [ops.fused_qkv_packed(x, w["q"], w["k"], w["v"]),
                   ops.gemv_packed(state["attn"], w["o"])]
        h = ops.ffn_up_fused_packed(x, w["gate"], w["up"])
        return out + [h, ops.ffn_down_residual_packed(h, w["down"], extra)]
    if op == "matmul":
        return ops.matmul_transB(x, w["w"], extra)
    out = []
    if op == "layer":
        out = [ops.fused_qkv(x, w["q"], w["k"], w["v"]), ops.matmul_transB(state["attn"], w["o"])]
    h = ops.ffn_up_fused(x, w["gate"], w["up"])
    return out + [h, ops.ffn_down_residual(h, w["down"], extra)]


def exact(case, seed):
    mats, blocks, x, attn, extra = _inputs(case, seed)

    def weight(k):
        fmt, N, K = mats[k]
        return _dequant64(fmt, blocks[k], N, K)

    if case["op"] == "dequant":
        return weight("w")

    def times(v, k):
        return v.to(torch.float64) @ weight(k).T

    flat = case["layout"] == "packed"  # the packed entry points return vectors
    if case["op"] == "matmul":
        y = times(x, "w")
        y = y if extra is None else y + extra.to(torch.float64)
        return y.reshape(-1) if flat else y
    out = []
    if case["op"] == "layer":
        out = [torch.cat([times(x, k) for k in ("q", "k", "v")], 1), times(attn, "o")]
    g = times(x, "gate")
    h = g * torch.sigmoid(g) * times(x, "up")
    out += [h, times(h, "down") + extra.to(torch.float64)]
    return [y.reshape(-1) for y in out] if flat else out


def work(case):
    mats = _matrices(case)
    size = sum(F.fmt(fmt).matrix_bytes(N, K) for fmt, N, K in mats.values())
    if case["op"] == "dequant":
        return {"bytes": size + 4 * case["N"] * case["K"], "flops": case["N"] * case["K"]}
    M = case["M"]
    flops = sum(2 * M * N * K for _, N, K in mats.values())
    if case["op"] == "matmul":
        return {"bytes": size + 4 * M * (case["N"] + case["K"]) + 4 * case["N"] * case["bias"],
                "flops": flops}
    h, f = case["hidden"], case["ffn"]
    values = h + f + 2 * h  # x, the FFN's inner vector, the residual and the result
    if case["op"] == "layer":
        values += h + 2 * case["kv"] + 2 * h  # q, k, v; the output projection's x and y
    return {"bytes": size + 4 * M * values, "flops": flops}


def tolerance(case):
    """fp32 activations carried to 22 bits, 32-bit sums: measured against
    exact() at 4e-6 and below (batch 1 through gate * up); dequantized values
    are exact."""
    return "exact" if case["op"] == "dequant" else {"rel": 1.5e-5}
