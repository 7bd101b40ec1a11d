"""The work a program has this library do, as measurable cases: the parts of one Gemma-4 12B layer
(hidden 3840, FFN 15360) in decode, in the verification of drafted tokens and in prefill, the lm-head,
and a run of decode layers, all through the `nsffn` entry points.

A case is a dict:
  part    "ffn"    gate/up + GeGLU, then down: `Context.ffn_block` (batch 1: the decode block with its RMSNorm)
          "attn"   the Q, K, V and output projections of one layer: `Context.qkv` and `Context.matmul`
          "head"   the 262,144-row Q6_K lm-head: `Context.matmul`
          "stack"  consecutive decode FFN blocks: `Context.ffn_stack_decode`
  batch   tokens: 1 decode, 2-4 verification, above that a prefill chunk of up to 2,048
  swa     ffn, batch > 4: a local layer (FP16 mode) or a global one (FP32 mode)
  down    "q4" / "q6": the type of ffn_down (the Q4_K_M mix has both)
  v       attn: "q4" / "q6" / "tied", the V projection's form
  layout  attn: "row" (as the GGUF holds it) or "cdna4" (re-tiled at load); the FFN and the head are re-tiled
  layers  stack: how many layers
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "neutron-star_amd"))
import nsffn as N  # noqa: E402

D, F, VOCAB = 3840, 15360, 262144
Q_ROWS, KV_ROWS = 4096, 2048  # 16 query heads and 8 key/value heads of 256
EPS = 1e-6
TYPES = {"q4": N.Q4_K, "q6": N.Q6_K}
LAYOUTS = {"row": N.ROW_MAJOR, "cdna4": N.CDNA4}

_ctx = []


def context():
    """The one context a program keeps (it owns the workspaces)."""
    if not _ctx:
        _ctx.append(N.Context(0))
    return _ctx[0]


def listed():
    return [
        # one generated token: the four attention projections, the smallest calls of the path
        dict(name="attn_decode", part="attn", batch=1, v="q6", layout="row"),
        # the last chunk of a 2,205-token prompt prefilled 1,024 tokens at a time
        dict(name="attn_prefill_157", part="attn", batch=157, v="q6", layout="row"),
        # one generated token: the FFN block, with the RMSNorm ahead of it
        dict(name="ffn_decode", part="ffn", batch=1, swa=True, down="q6"),
        # verification of two drafted tokens and the one before them
        dict(name="ffn_verify_3", part="ffn", batch=3, swa=True, down="q6"),
        # a one-line turn of a conversation whose prefix is cached
        dict(name="ffn_prefill_19", part="ffn", batch=19, swa=True, down="q4"),
        # the reference's published prompts of 225 and 775 tokens, and the full 1,024-token chunk
        dict(name="ffn_prefill_225", part="ffn", batch=225, swa=True, down="q6"),
        dict(name="ffn_prefill_775_global", part="ffn", batch=775, swa=False, down="q4"),
        dict(name="ffn_prefill_1024", part="ffn", batch=1024, swa=True, down="q6"),
        # the largest chunk the engine accepts
        dict(name="ffn_prefill_2048", part="ffn", batch=2048, swa=True, down="q4"),
        # logits of one generated token, and of a verification step
        dict(name="head_decode", part="head", batch=1),
        dict(name="head_verify_3", part="head", batch=3),
        # a stage of consecutive decode FFN layers, the Q4_K_M mix of down types
        dict(name="stack_decode_12", part="stack", batch=1, layers=12),
    ]


def draw(rng):
    part = rng.choice(["ffn", "ffn", "ffn", "attn", "attn", "head", "stack"])
    if part == "head":
        return dict(part=part, batch=rng.randint(1, 4))
    if part == "stack":
        return dict(part=part, batch=1, layers=rng.randint(2, 12))
    # decode and verification one time in four, else a prefill chunk, spread over its logarithm
    if rng.random() < 0.25:
        batch = rng.randint(1, 4)
    else:
        batch = min(2048, int(round(math.exp(rng.uniform(math.log(5), math.log(2048))))))
    if part == "attn":
        return dict(part=part, batch=batch, v=rng.choice(["q4", "q6", "tied"]), layout=rng.choice(["row", "row", "cdna4"]))
    return dict(part=part, batch=batch, swa=rng.random() < 5 / 6, down=rng.choice(["q4", "q6"]))


# ---- inputs ---------------------------------------------------------------------------------

def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + salt) % (1 << 62))


def _blocks(qtype, rows, cols, seed, salt):
    """Row-major super-blocks [rows*cols/256][bytes] of zero-mean weights of standard deviation ~0.02:
    any quants, scales and mins, with block factors around 1e-4 (Q4_K) and 1.5e-5 (Q6_K)."""
    nblk, size = rows * (cols // 256), N.BLOCK_BYTES[qtype]
    g = _generator(seed, salt)
    raw = torch.empty((nblk * size + 7) // 8, dtype=torch.int64, device="cuda").random_(-(1 << 63), None, generator=g)
    blk = raw.view(torch.uint8)[: nblk * size].view(nblk, size)
    u = torch.rand(nblk, 1, device="cuda", generator=g) + 0.5
    if qtype == N.Q4_K:
        blk[:, 0:2] = (u * 1e-4).half().view(torch.uint8)
        blk[:, 2:4] = (u * 7.5e-4).half().view(torch.uint8)
    else:
        blk[:, 208:210] = (u * 1.5e-5).half().view(torch.uint8)
    return blk


def _weights(qtype, rows, cols, seed, salt, layout=N.CDNA4):
    src = _blocks(qtype, rows, cols, seed, salt).reshape(-1)
    if layout == N.ROW_MAJOR:
        return src
    dst = torch.empty_like(src)
    N.retile_device(src, dst, qtype, cols, rows, N.ROW_MAJOR, layout)
    return dst


def _normal(seed, salt, *shape):
    return torch.randn(*shape, device="cuda", generator=_generator(seed, salt))


def _f32(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _f16(*shape):
    return torch.empty(shape, dtype=torch.float16, device="cuda")


def _norm_weight(seed, salt):
    return _normal(seed, salt, D) * 0.1 + 1.0


def _tokens(case, seed, cols, salt):
    """The activations: fp32 for one token and for the head, else fp16."""
    x = _normal(seed, salt, case["batch"], cols)
    return x if case["batch"] == 1 or case["part"] == "head" else x.half()


def _down_type(layer):
    return "q6" if layer % 2 == 0 else "q4"


def prepare(case, seed):
    ctx, b = context(), case["batch"]
    s = dict(case, ctx=ctx)
    if case["part"] == "head":
        s.update(w=_weights(N.Q6_K, VOCAB, D, seed, 1), x=_tokens(case, seed, D, 2), y=_f32(b, VOCAB))
    elif case["part"] == "attn":
        lay, vt = LAYOUTS[case["layout"]], TYPES.get(case["v"], N.Q4_K)
        s.update(lay=lay, vt=vt, x=_tokens(case, seed, D, 2), a=_tokens(case, seed, Q_ROWS, 3),
                 wq=_weights(N.Q4_K, Q_ROWS, D, seed, 4, lay), wk=_weights(N.Q4_K, KV_ROWS, D, seed, 5, lay),
                 wv=None if case["v"] == "tied" else _weights(vt, KV_ROWS, D, seed, 6, lay),
                 wo=_weights(N.Q4_K, D, Q_ROWS, seed, 7, lay),
                 q=_f32(b, Q_ROWS), k=_f32(b, KV_ROWS), vo=_f32(b, KV_ROWS), o=_f32(b, D))
    elif case["part"] == "ffn":
        half = b > 1
        s.update(x=_tokens(case, seed, D, 2), wg=_weights(N.Q4_K, F, D, seed, 4), wu=_weights(N.Q4_K, F, D, seed, 5),
                 dt=TYPES[case["down"]], wd=_weights(TYPES[case["down"]], D, F, seed, 6), nw=_norm_weight(seed, 7),
                 h=_f16(b, F) if half else _f32(b, F), y=_f32(b, D))
    else:
        n = case["layers"]
        s.update(x=_tokens(case, seed, D, 2), h=_f32(1, F), y=_f32(1, D),
                 wg=[_weights(N.Q4_K, F, D, seed, 10 + 4 * i) for i in range(n)],
                 wu=[_weights(N.Q4_K, F, D, seed, 11 + 4 * i) for i in range(n)],
                 wd=[_weights(TYPES[_down_type(i)], D, F, seed, 12 + 4 * i) for i in range(n)],
                 nw=[_norm_weight(seed, 13 + 4 * i) for i in range(n)], dt=[TYPES[_down_type(i)] for i in range(n)])
    return s


def run(s):
    ctx, b = s["ctx"], s["batch"]
    if s["part"] == "head":
        ctx.matmul(s["w"], N.Q6_K, N.CDNA4, D, VOCAB, b, s["x"], s["y"])
        return s["y"]
    if s["part"] == "attn":
        lay, vt = s["lay"], s["vt"]
        if b == 1:
            ctx.matmul(s["wq"], N.Q4_K, lay, D, Q_ROWS, 1, s["x"], s["q"])
            ctx.matmul(s["wk"], N.Q4_K, lay, D, KV_ROWS, 1, s["x"], s["k"])
            if s["wv"] is not None:
                ctx.matmul(s["wv"], vt, lay, D, KV_ROWS, 1, s["x"], s["vo"])
        else:
            ctx.qkv(s["wq"], s["wk"], s["wv"], vt, lay, D, Q_ROWS, KV_ROWS, b, s["x"], s["q"], s["k"], s["vo"])
        ctx.matmul(s["wo"], N.Q4_K, lay, Q_ROWS, D, b, s["a"], s["o"], half_input=b > 1)
        out = [s["q"], s["k"], s["o"]]
        return out if b == 1 and s["wv"] is None else out + [s["vo"]]
    if s["part"] == "ffn":
        if b == 1:
            ctx.ffn_block_decode(s["wg"], s["wu"], s["wd"], s["dt"], N.CDNA4, D, F, s["x"], s["h"], s["y"],
                                 norm_weight=s["nw"], eps=EPS)
        else:
            ctx.ffn_block(s["wg"], s["wu"], s["wd"], s["dt"], N.CDNA4, D, F, b, s["x"], s["h"], s["y"], True, s["swa"])
        return [s["h"], s["y"]]
    ctx.ffn_stack_decode(s["wg"], s["wu"], s["wd"], s["dt"], N.CDNA4, D, F, s["x"], s["h"], s["y"],
                         norm_weights=s["nw"], eps=EPS)
    return [s["h"], s["y"]]


# ---- what one pass cannot do without --------------------------------------------------------

def work(case):
    b, half = case["batch"], 4 if case["batch"] == 1 or case["part"] == "head" else 2

    def gemm(qtype, rows, cols, out=4, read_x=True):
        weights = rows * (cols // 256) * N.BLOCK_BYTES[qtype]
        return weights + (b * cols * half if read_x else 0) + b * rows * out, 2 * b * rows * cols

    if case["part"] == "head":
        parts = [gemm(N.Q6_K, VOCAB, D)]
    elif case["part"] == "attn":
        parts = [gemm(N.Q4_K, Q_ROWS, D), gemm(N.Q4_K, KV_ROWS, D, read_x=False), gemm(N.Q4_K, D, Q_ROWS)]
        if case["v"] != "tied":
            parts.append(gemm(TYPES[case["v"]], KV_ROWS, D, read_x=False))
        elif b > 1:
            parts.append((b * KV_ROWS * 4, 0))
    else:
        layers = [case["down"]] if case["part"] == "ffn" else [_down_type(i) for i in range(case["layers"])]
        parts = [(b * F * half, 0), (b * D * half + b * D * 4, 0)]  # the last h, the first x, the last y
        for down in layers:
            for qtype, rows, cols in ((N.Q4_K, F, D), (N.Q4_K, F, D), (TYPES[down], D, F)):
                parts.append((rows * (cols // 256) * N.BLOCK_BYTES[qtype], 2 * b * rows * cols))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times the distance from `exact` (2-norms), measured over the listed and drawn cases."""
    b = case["batch"]
    if case["part"] == "stack":
        return {"rel": 2e-4}  # 3.8e-5 after 12 chained layers
    if case["part"] == "ffn" and b > 1:
        # h is handed on in fp16 (2.1e-4); the FP16 mode rounds the weights to fp16 as well (8.3e-4)
        return {"rel": 3.3e-3 if case["swa"] and b > 4 else 8e-4}
    if case["part"] == "attn" and b > 4 and case["v"] == "q6":
        return {"rel": 6e-4}  # Q6_K scale times quant as one fp16 in the prefill product: 1.4e-4
    return {"rel": 1e-5}  # sums in 32 bits: 3e-7


# ---- the same in 64 bits --------------------------------------------------------------------

def _dequant(qtype, blk):
    """float64 weights [nblk][256] of row-major super-blocks (the GGUF element formulas)."""
    half = lambda c: blk[:, c:c + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if qtype == N.Q4_K:
        sb = blk[:, 4:16].to(torch.int16)
        sc = torch.cat([sb[:, 0:4] & 63, (sb[:, 8:12] & 15) | ((sb[:, 0:4] >> 6) << 4)], 1)
        m = torch.cat([sb[:, 4:8] & 63, (sb[:, 8:12] >> 4) | ((sb[:, 4:8] >> 6) << 4)], 1)
        qs = blk[:, 16:144].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        return ((half(0) * sc).unsqueeze(2) * q - (half(2) * m).unsqueeze(2)).view(-1, 256)
    ql, qh = blk[:, 0:128].reshape(-1, 2, 64), blk[:, 128:192].reshape(-1, 2, 32)
    lo = torch.stack([ql[:, :, :32] & 15, ql[:, :, 32:] & 15, ql[:, :, :32] >> 4, ql[:, :, 32:] >> 4], 2)
    hi = torch.stack([(qh >> (2 * j)) & 3 for j in range(4)], 2)
    v = ((lo | (hi << 4)).double() - 32.0).view(-1, 16, 16)
    sc = blk[:, 192:208].contiguous().view(torch.int8).double()
    return (v * (sc * half(208)).unsqueeze(2)).view(-1, 256)


def _product(qtype, rows, cols, seed, salt, x):
    """x . W^T in float64 for the tensor _blocks makes, some rows at a time."""
    blk, nb, step = _blocks(qtype, rows, cols, seed, salt), cols // 256, 8192
    x = x.double()
    return torch.cat([x @ _dequant(qtype, blk[r * nb:(r + step) * nb]).view(-1, cols).t().contiguous()
                      for r in range(0, rows, step)], 1)


def _gelu(g):
    return 0.5 * g * (1.0 + torch.tanh(0.7978845608028654 * g * (1.0 + 0.044715 * g * g)))


def _normed(x, w):
    x = x.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def exact(case, seed):
    b = case["batch"]
    x = _tokens(case, seed, D, 2)
    if case["part"] == "head":
        return _product(N.Q6_K, VOCAB, D, seed, 1, x)
    if case["part"] == "attn":
        k = _product(N.Q4_K, KV_ROWS, D, seed, 5, x)
        out = [_product(N.Q4_K, Q_ROWS, D, seed, 4, x), k,
               _product(N.Q4_K, D, Q_ROWS, seed, 7, _tokens(case, seed, Q_ROWS, 3))]
        if case["v"] == "tied":
            return out if b == 1 else out + [k]
        return out + [_product(TYPES[case["v"]], KV_ROWS, D, seed, 6, x)]
    if case["part"] == "ffn":
        n = _normed(x, _norm_weight(seed, 7)) if b == 1 else x
        h = _gelu(_product(N.Q4_K, F, D, seed, 4, n)) * _product(N.Q4_K, F, D, seed, 5, n)
        # the interface hands h on in fp16 above one token: the down projection's input is that value
        return [h, _product(TYPES[case["down"]], D, F, seed, 6, h.half() if b > 1 else h)]
    y = x
    for i in range(case["layers"]):
        n = _normed(y, _norm_weight(seed, 13 + 4 * i))
        h = _gelu(_product(N.Q4_K, F, D, seed, 10 + 4 * i, n)) * _product(N.Q4_K, F, D, seed, 11 + 4 * i, n)
        y = _product(TYPES[_down_type(i)], D, F, seed, 12 + 4 * i, h)
    return [h, y]
