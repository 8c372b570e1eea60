"""The products that a program on this framework runs, as timed cases.

A case names one product (``path``), the encoding of its weights, how they are kept
(``packed``: the tile-packed form of a weight bank; otherwise GGUF rows as the file holds
them) and its sizes.  Weights and activations follow the benchmark's distributions: codes
uniform, fp16 block scales |N(0, 1)| times the format's magnitude, activations N(0, 1).
"""
import math

import torch

from kadan_amd import ops

Q4_0, Q8_0, Q3_K, Q4_K, Q6_K, IQ4_NL, IQ4_XS, BF16 = 2, 8, 11, 12, 14, 20, 23, 30
# values and bytes of a block, byte offset of the fp16 scale, magnitude of the scale
FORMATS = {Q4_0: (32, 18, 0, 0.02), Q8_0: (32, 34, 0, 0.01), Q3_K: (256, 110, 108, 0.005),
           Q4_K: (256, 144, 0, 0.005), Q6_K: (256, 210, 208, 0.0005),
           IQ4_NL: (32, 18, 0, 0.0005), IQ4_XS: (256, 136, 0, 0.0002)}
IQ4_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


# ------------------------------------------------------------------------- the cases

def listed():
    return [
        # one decode token through a square attention projection: the smallest product
        gemv("gemv_q8_0_4096x4096", Q8_0, True, 4096, 4096, 1),
        # one decode token through an FFN gate or up matrix: the benchmark's headline
        gemv("gemv_q4_k_4096x14336", Q4_K, True, 4096, 14336, 1),
        # a few sequences decoding together through an FFN down matrix whose rows lie as
        # in the file (an encoding without a packed form)
        gemv("gemv_q3_k_rows_14336x4096_r4", Q3_K, False, 14336, 4096, 4),
        # a prefill chunk of 512 tokens through an FFN gate or up matrix of the bank
        gemm("gemm_q4_k_4096x14336_m512", Q4_K, True, 4096, 14336, 512),
        # the ragged last chunk of a prompt through an FFN down matrix of the bank
        gemm("gemm_q6_k_14336x4096_m77", Q6_K, True, 14336, 4096, 77),
        # the same chunk as above over rows as the file holds them
        gemm("gemm_iq4_xs_rows_4096x14336_m512", IQ4_XS, False, 4096, 14336, 512),
        # the benchmark's Q4_0 prefill product: fp16 activations quantised on the fly
        dict(name="gemm_q4_0_4096x14336_m512", path="gemm_q4_0", packed=True, k=4096, n=14336,
             m=512),
        # a decode token and a prefill chunk through a Qwen3-30B-A3B mixture layer
        moe_gguf("moe_gguf_t1", 1),
        moe_gguf("moe_gguf_t512", 512),
        # the benchmark's MXFP4 mixture layers: a decode token, a prefill of 256 tokens,
        # and 2048 tokens of which a quarter favours 8 hot experts of 128
        moe_mxfp4("moe_mxfp4_e32_t1", 32, 1, 0),
        moe_mxfp4("moe_mxfp4_e32_t256", 32, 256, 0),
        moe_mxfp4("moe_mxfp4_e128_t2048_hot", 128, 2048, 8),
    ]


def gemv(name, enc, packed, k, n, rows):
    return dict(name=name, path="gemv", enc=enc, packed=packed, k=k, n=n, m=rows)


def gemm(name, enc, packed, k, n, m):
    return dict(name=name, path="gemm", enc=enc, packed=packed, k=k, n=n, m=m)


def moe_gguf(name, m):
    return dict(name=name, path="moe_gguf", hidden=2048, experts=128, top_k=8, ff=768,
                shared_ff=768, down=Q6_K, shared=Q8_0, m=m)


def moe_mxfp4(name, experts, m, hot):
    return dict(name=name, path="moe_mxfp4", hidden=2880, experts=experts, top_k=4, inter=2880,
                hot=hot, m=m)


def draw(rng):
    def spread(low, high):  # log-uniform whole number
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    def chunk(least, k, n):  # rows of a prefill chunk, none dearer than the listed cases
        return min(spread(least, 1024), 10 ** 11 // (k * n))

    path = rng.choice(["gemv", "gemv", "gemm", "gemm", "gemm_q4_0", "moe_gguf", "moe_gguf",
                       "moe_mxfp4", "moe_mxfp4"])
    if path in ("gemv", "gemm"):
        packed = rng.random() < 0.6
        enc = rng.choice([Q4_K, Q8_0, Q6_K] if packed else
                         [Q3_K, IQ4_XS, IQ4_NL, Q4_K, Q6_K, BF16])
        k, n = 256 * spread(4, 56), spread(512, 16384)
        m = rng.choice([1, 1, 1, 2, 3, 4, 5, 8]) if path == "gemv" else chunk(9, k, n)
        return dict(path=path, enc=enc, packed=packed, k=k, n=n, m=m)
    if path == "gemm_q4_0":
        k, n = 256 * spread(4, 56), spread(512, 16384)
        return dict(path=path, packed=rng.random() < 0.7, k=k, n=n, m=chunk(1, k, n))
    if path == "moe_gguf":
        experts = rng.choice([16, 32, 60, 64, 128])
        return dict(path=path, hidden=256 * spread(4, 16), experts=experts,
                    top_k=rng.choice([2, 4, 6, 8]), ff=256 * spread(2, 6),
                    shared_ff=256 * spread(2, 6), down=rng.choice([Q6_K, Q4_K]),
                    shared=rng.choice([Q8_0, Q4_K]), m=spread(1, 512))
    top_k = rng.choice([1, 2, 4, 8])
    return dict(path=path, hidden=64 * spread(16, 45), experts=rng.choice([8, 16, 32, 64, 128]),
                top_k=top_k, inter=64 * spread(16, 45), hot=rng.choice([0, 0, 2]),
                m=spread(1, min(2048, 8192 // top_k)))


# ------------------------------------------------------------------------- their inputs

def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def gguf_rows(g, enc, n, k):
    """uint8 [n, row_bytes] of one encoding."""
    if enc == BF16:
        return (normal(g, n, k) * 0.02).bfloat16().view(torch.uint8)
    values, size, at, scale = FORMATS[enc]
    b = torch.randint(0, 256, (n, k // values, size), generator=g, dtype=torch.uint8,
                      device="cuda")
    for offset in (at, 2) if enc == Q4_K else (at,):
        d = (normal(g, n, k // values).abs() * scale).half()
        b[..., offset:offset + 2] = d.unsqueeze(-1).view(torch.uint8)
    return b.reshape(n, -1)


def mxfp4_stack(g, experts, rows, cols):
    """GPT-OSS layout: nibbles uint8 [experts, rows, cols/2], exponents [experts, rows, cols/32]."""
    blocks = torch.randint(0, 256, (experts, rows, cols // 2), generator=g, dtype=torch.uint8,
                           device="cuda")
    scales = torch.randint(119, 128, (experts, rows, cols // 32), generator=g,
                           dtype=torch.uint8, device="cuda")
    return blocks, scales


def gguf_moe_spec(c, g):
    H, E, F, S = c["hidden"], c["experts"], c["ff"], c["shared_ff"]
    spec = dict(hidden=H, experts=E, top_k=c["top_k"], ff=F, shared_ff=S)
    spec["router"] = (0, (normal(g, E, H) / math.sqrt(H)).view(torch.uint8))
    for name, enc, n, k in (("gate_exps", Q4_K, F, H), ("up_exps", Q4_K, F, H),
                            ("down_exps", c["down"], H, F)):
        spec[name] = (enc, gguf_rows(g, enc, E * n, k).reshape(E, n, -1))
    for name, enc, n, k in (("gate_shexp", c["shared"], S, H), ("up_shexp", c["shared"], S, H),
                            ("down_shexp", Q4_K, H, S)):
        spec[name] = (enc, gguf_rows(g, enc, n, k))
    spec["shared_gate"] = normal(g, H) / math.sqrt(H)
    return spec


def moe_logits(c, g):
    logits = normal(g, c["m"], c["experts"])
    if c["hot"]:
        picked = torch.randperm(c["experts"], generator=g, device="cuda")[:c["hot"]]
        logits[0::4, picked] += 3.0
    return logits


def prepare(case, seed):
    c, g = case, generator(seed)
    if c["path"] == "moe_gguf":
        spec = gguf_moe_spec(c, g)
        return dict(case=c, spec=spec, packed=ops.moe_gguf_pack(spec),
                    x=normal(g, c["m"], c["hidden"]))
    if c["path"] == "moe_mxfp4":
        H, E, I = c["hidden"], c["experts"], c["inter"]
        stacks = [ops.moe_mxfp4_pack(*mxfp4_stack(g, E, n, k), E, n, k)
                  for n, k in ((I, H), (I, H), (H, I))]
        return dict(case=c, stacks=stacks, x=normal(g, c["m"], H).bfloat16(),
                    logits=moe_logits(c, g), y=torch.empty(c["m"], H, device="cuda"))
    enc = Q4_0 if c["path"] == "gemm_q4_0" else c["enc"]
    w = gguf_rows(g, enc, c["n"], c["k"])
    if c["packed"]:
        w = ops.gguf_pack(enc, w, c["k"])
    x = normal(g, c["m"], c["k"])
    y = torch.empty(c["m"], c["n"], device="cuda")
    if c["path"] == "gemm_q4_0":
        x, y = x.half(), y.half()
    return dict(case=c, w=w, x=x, y=y)


# ------------------------------------------------------------------------- one pass

def run(state):
    c = state["case"]
    if c["path"] == "gemv":
        product = ops.gemv_packed if c["packed"] else ops.gemv
        return product(c["enc"], state["w"], state["x"], c["n"], out=state["y"])
    if c["path"] == "gemm":
        product = ops.gemm_packed if c["packed"] else ops.gemm_rows
        return product(c["enc"], state["w"], state["x"], c["n"], out=state["y"])
    if c["path"] == "gemm_q4_0":
        product = ops.gemm_q4_0_packed if c["packed"] else ops.gemm_q4_0
        return product(state["w"], state["x"], c["n"], out=state["y"])
    if c["path"] == "moe_gguf":
        return ops.moe_gguf(state["spec"], state["x"], packed=state["packed"])
    y, idx, w, _, _ = ops.moe_mxfp4_packed(state["x"], state["logits"], c["top_k"], c["inter"],
                                           *state["stacks"], routing=True, out=state["y"])
    return y, idx, w


# ------------------------------------------------------------------------- what it needs

def row_bytes(enc, k):
    return 2 * k if enc == BF16 else k // FORMATS[enc][0] * FORMATS[enc][1]


def touched(c):
    """Experts that m tokens of top_k distinct random experts reach, on average."""
    return c["experts"] * (1.0 - (1.0 - c["top_k"] / c["experts"]) ** c["m"])


def work(case):
    c, m = case, case["m"]
    if c["path"] == "moe_gguf":
        H, E, F, S = c["hidden"], c["experts"], c["ff"], c["shared_ff"]
        expert = 2 * F * row_bytes(Q4_K, H) + H * row_bytes(c["down"], F)
        shared = 2 * S * row_bytes(c["shared"], H) + H * row_bytes(Q4_K, S)
        return {"bytes": int(touched(c) * expert) + shared + 4 * E * H + 4 * H + 8 * m * H
                + 8 * m * c["top_k"],
                "flops": 2 * m * H * (E + 3 * F * c["top_k"] + 3 * S)}
    if c["path"] == "moe_mxfp4":
        H, E, I = c["hidden"], c["experts"], c["inter"]
        expert = 3 * H * I * 17 // 32
        return {"bytes": int(touched(c) * expert) + m * (2 * H + 4 * H + 4 * E + 8 * c["top_k"]),
                "flops": 6 * m * c["top_k"] * H * I}
    enc, element = (Q4_0, 2) if c["path"] == "gemm_q4_0" else (c["enc"], 4)
    return {"bytes": c["n"] * row_bytes(enc, c["k"]) + element * m * (c["k"] + c["n"]),
            "flops": 2 * m * c["n"] * c["k"]}


def tolerance(case):
    """About four times the distance from 64 bits that each product shows: the decode
    products carry activations as 16-bit block fixed point (2e-5), the prefill products
    round both operands to fp16 (4e-4, and 6e-4 through two products and the gate), the
    MXFP4 layer's activations are exact bf16 and its hidden rows about 12 bits (3e-5)."""
    if case["path"] == "gemv":
        return {"rel": 1e-4, "max": 1e-3}
    if case["path"] in ("gemm", "gemm_q4_0"):
        return {"rel": 1.5e-3, "max": 1.5e-2}
    if case["path"] == "moe_mxfp4":
        return {"rel": 1e-4, "max": 5e-3, "differ": 1e-3}
    if case["m"] <= 8:
        return {"rel": 2e-4, "max": 5e-3, "differ": 1e-3}
    return {"rel": 2.5e-3, "max": 0.1, "differ": 1e-3}


# ------------------------------------------------------------------------- in 64 bits

def f16(b):
    """The fp16 scale of each block, float64 [..., 1]."""
    return b.contiguous().view(torch.float16).double()


def decoded(enc, rows, k):
    """uint8 [n, row_bytes] -> float64 [n, k]."""
    n = rows.shape[0]
    if enc == BF16:
        return rows.contiguous().view(torch.bfloat16).double()
    values, size, at, _ = FORMATS[enc]
    b = rows.reshape(n, k // values, size)
    d = f16(b[..., at:at + 2])
    if enc == Q8_0:
        return (d * b[..., 2:].view(torch.int8).double()).reshape(n, k)
    if enc in (Q4_0, IQ4_NL):
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1)
        return (d * (levels(q) if enc == IQ4_NL else q.double() - 8)).reshape(n, k)
    if enc == IQ4_XS:
        q = b[..., 8:].reshape(n, -1, 8, 16)
        q = torch.cat([q & 15, q >> 4], -1)
        low = torch.stack([b[..., 4:8] & 15, b[..., 4:8] >> 4], -1).reshape(n, -1, 8)
        high = b[..., 2:4].long()
        high = (high[..., :1] | high[..., 1:] << 8) >> 2 * torch.arange(8, device=b.device) & 3
        scale = d * (low.long() + (high << 4) - 32)
        return (scale.unsqueeze(-1) * levels(q)).reshape(n, k)
    if enc == Q4_K:
        s = b[..., 4:16]
        low, mid, top = s[..., :4], s[..., 4:8], s[..., 8:]
        scale = torch.cat([low & 63, (top & 15) | (low >> 6) << 4], -1)
        least = torch.cat([mid & 63, (top >> 4) | (mid >> 6) << 4], -1)
        q = b[..., 16:].reshape(n, -1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], -2).reshape(n, -1, 8, 32)
        w = (d * scale).unsqueeze(-1) * q - (f16(b[..., 2:4]) * least).unsqueeze(-1)
        return w.reshape(n, k)
    two = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device)
    if enc == Q6_K:
        low = b[..., :128].reshape(n, -1, 2, 1, 64)
        low = torch.cat([low & 15, low >> 4], -2).reshape(n, -1, 2, 4, 32)
        high = b[..., 128:192].reshape(n, -1, 2, 1, 32) >> two[:, None] & 3
        scale = b[..., 192:208].contiguous().view(torch.int8).double()
        q = (low | high << 4).double() - 32
    else:  # Q3_K
        low = b[..., 32:96].reshape(n, -1, 2, 1, 32) >> two[:, None] & 3
        bit = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(2, 4, 1)
        high = b[..., :32].reshape(n, -1, 1, 1, 32) >> bit & 1
        nibble = torch.cat([b[..., 96:104] & 15, b[..., 96:104] >> 4], -1)
        pair = (b[..., 104:108].unsqueeze(-2) >> two[:, None] & 3).reshape(n, -1, 16)
        scale = (nibble | pair << 4).double() - 32
        q = (low | high << 2).double() - 4
    return ((d * scale).unsqueeze(-1) * q.reshape(n, -1, 16, 16)).reshape(n, k)


def levels(q):
    return torch.tensor(IQ4_LEVELS, dtype=torch.float64, device=q.device)[q.long()]


def mxfp4_decoded(blocks, scales):
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64,
                         device=blocks.device)
    q = torch.stack([blocks & 15, blocks >> 4], -1).reshape(*scales.shape, 32)
    w = table[q.long()] * torch.exp2(scales.double() - 127).unsqueeze(-1)
    return w.reshape(scales.shape[0], -1)


def routed(logits, top_k):
    """Softmax over every expert, the top_k largest, renormalised."""
    p = torch.softmax(logits.double(), -1)
    best, idx = torch.topk(p, top_k, dim=-1)
    return idx, best / best.sum(-1, keepdim=True).clamp_min(2.0 ** -14)


def mixture(x, idx, weights, experts, expert, hidden):
    y = torch.zeros(x.shape[0], hidden, dtype=torch.float64, device=x.device)
    for e in range(experts):
        token, slot = torch.nonzero(idx == e, as_tuple=True)
        if token.numel():
            gate, up, down = expert(e)
            h = torch.nn.functional.silu(x[token] @ gate.T) * (x[token] @ up.T)
            y[token] += weights[token, slot].unsqueeze(-1) * (h @ down.T)
    return y


def exact(case, seed):
    c, g = case, generator(seed)
    if c["path"] == "moe_gguf":
        spec = gguf_moe_spec(c, g)
        H, F, S = c["hidden"], c["ff"], c["shared_ff"]
        x = normal(g, c["m"], H).double()
        idx, weights = routed(x @ spec["router"][1].view(torch.float32).double().T, c["top_k"])

        def expert(e):
            return [decoded(spec[name][0], spec[name][1][e], k)
                    for name, k in (("gate_exps", H), ("up_exps", H), ("down_exps", F))]
        y = mixture(x, idx, weights, c["experts"], expert, H)
        gate, up, down = (decoded(*spec[name], k) for name, k in
                          (("gate_shexp", H), ("up_shexp", H), ("down_shexp", S)))
        shared = (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T
        y += torch.sigmoid(x @ spec["shared_gate"].double()).unsqueeze(-1) * shared
        return y, idx.int(), weights
    if c["path"] == "moe_mxfp4":
        H, E, I = c["hidden"], c["experts"], c["inter"]
        stacks = [mxfp4_stack(g, E, n, k) for n, k in ((I, H), (I, H), (H, I))]
        x = normal(g, c["m"], H).bfloat16().double()
        idx, weights = routed(moe_logits(c, g), c["top_k"])

        def expert(e):
            return [mxfp4_decoded(blocks[e], scales[e]) for blocks, scales in stacks]
        return mixture(x, idx, weights, E, expert, H), idx.int(), weights
    enc = Q4_0 if c["path"] == "gemm_q4_0" else c["enc"]
    w = decoded(enc, gguf_rows(g, enc, c["n"], c["k"]), c["k"])
    x = normal(g, c["m"], c["k"])
    if c["path"] == "gemm_q4_0":  # the product's own definition: x in int8 blocks of 32
        x = x.half().float().reshape(c["m"], -1, 32)
        top = x.abs().amax(-1, keepdim=True)
        codes = torch.round(x * torch.where(top > 0, 127.0 / top, 0.0))
        x = (codes.double() * (top / 127.0).double()).reshape(c["m"], -1)
    return x.double() @ w.T
