"""The work that a user of the GGUF linear path has it do, as cases to time and to compare.

A server that runs a GGUF model calls this library in four ways: the linear modules of every
decoder layer at decode (a few rows, captured in a HIP graph, as vLLM captures its decode
step), the same modules at prefill (hundreds to thousands of rows, launched eagerly), the
repack of every weight while the model loads, and the dequantize API.  Layer sizes are the
27B-class ones of this repository's benchmark (hidden 5120, intermediate 17408) or generic;
weights are random valid GGUF blocks whose scales give them the spread of a trained layer.
"""
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "hyperqwen-rtx4080s32_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gguf_hip  # noqa: E402

Q4_0, Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ3_S, IQ4_XS = 2, 6, 8, 10, 11, 12, 13, 14, 20, 21, 23
# GGML type -> (weights per block, bytes per block)
BLOCK = {Q4_0: (32, 18), Q5_0: (32, 22), Q8_0: (32, 34), Q2_K: (256, 84), Q3_K: (256, 110), Q4_K: (256, 144),
         Q5_K: (256, 176), Q6_K: (256, 210), IQ4_NL: (32, 18), IQ3_S: (256, 110), IQ4_XS: (256, 136)}
# byte offset of the block's fp16 scale, of its fp16 min scale (None: none), and their size for
# uniform quantized fields to come out as weights of about 0.02
SCALE = {Q4_0: (0, None, 4e-3, 0), Q5_0: (0, None, 2e-3, 0), Q8_0: (0, None, 2.5e-4, 0), IQ4_NL: (0, None, 3e-4, 0),
         Q2_K: (80, 82, 2.4e-3, 3.6e-3), Q3_K: (108, None, 5e-4, 0), Q4_K: (0, 2, 1.2e-4, 9e-4),
         Q5_K: (0, 2, 6e-5, 9.3e-4), Q6_K: (208, None, 1.5e-5, 0), IQ3_S: (0, None, 1.5e-4, 0),
         IQ4_XS: (0, None, 1.5e-5, 0)}
TYPES = tuple(BLOCK)
# how often each type is drawn: the mixed models of the benchmark are mostly Q4_K, Q5_K, IQ4_XS
WEIGHTS = tuple({Q4_K: 6, Q5_K: 4, IQ4_XS: 4, Q6_K: 3}.get(t, 1) for t in TYPES)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _row_bytes(t, k):
    return k // BLOCK[t][0] * BLOCK[t][1]


def _shards(text):
    """"12:1024,14:512" -> [(type, rows), ...]"""
    return [tuple(int(v) for v in s.split(":")) for s in text.split(",")]


def _modules(case):
    """The linear modules of a case: [(shards, K)].  A decoder layer has four (qkv, o_proj, gate_up, down)."""
    if case["op"] != "layer":
        return [(_shards(case["shards"]), case["k"])]
    h, i, kv = case["hidden"], case["inter"], case["kv"]
    q, k, v, o, g, u, d = (int(t) for t in case["types"].split(","))
    return [([(q, h), (k, kv), (v, kv)], h), ([(o, h)], h), ([(g, i), (u, i)], h), ([(d, h)], i)]


def listed():
    layer = {"op": "layer", "hidden": 5120, "inter": 17408, "kv": 1024, "graph": True}
    gate_up = {"op": "linear", "k": 5120, "x": "bf16", "bias": False}
    down = {"op": "linear", "k": 17408, "x": "bf16", "bias": False}
    return [
        # the smallest call: one small projection for one token, launched eagerly
        {"name": "linear-q8_0-m1", "op": "linear", "shards": "8:4096", "k": 4096, "m": 1, "x": "bf16", "bias": False,
         "graph": False},
        # one decoder layer's weight stream for one token: the step of a single chat
        {"name": "layer-m1", **layer, "m": 1, "types": "12,12,14,12,12,12,14"},
        # the same with eight rows: a few chats, or one with speculative rows; another type mix
        {"name": "layer-m8", **layer, "m": 8, "types": "13,13,14,13,23,23,13"},
        # two streams of eight speculative rows through the largest matrix of a layer
        {"name": "gate_up-q4_k-m16", **gate_up, "shards": "12:17408,12:17408", "m": 16, "graph": True},
        # four streams of eight speculative rows
        {"name": "layer-m32", **layer, "m": 32, "types": "13,13,14,12,12,12,14"},
        # a batch of 64 chats
        {"name": "gate_up-iq4_xs-m64", **gate_up, "shards": "23:17408,23:17408", "m": 64, "graph": True},
        # a larger batch through the long-K matrix
        {"name": "down-q5_k-m128", **down, "shards": "13:5120", "m": 128, "graph": True},
        # a ragged prompt through a ragged mixed-type layer with a bias and fp16 activations
        {"name": "ragged-m333", "op": "linear", "shards": "11:3001,8:517,21:1090", "k": 2816, "m": 333, "x": "fp16",
         "bias": True, "graph": False},
        # a prompt chunk of 2048 tokens (the benchmark's prefill line)
        {"name": "gate_up-q4_k-m2048", **gate_up, "shards": "12:17408,12:17408", "m": 2048, "graph": False},
        # the largest chunk
        {"name": "down-q5_k-m8192", **down, "shards": "13:5120", "m": 8192, "graph": False},
        # the dequantize API on a layer's raw rows (callers that run their own GEMM)
        {"name": "dequantize-q6_k", "op": "dequantize", "shards": "14:34816", "k": 5120, "dtype": "bf16"},
        # model load: the repack of a layer's largest matrix
        {"name": "repack-q4_k", "op": "repack", "shards": "12:34816", "k": 5120},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    t = lambda: rng.choices(TYPES, WEIGHTS)[0]  # noqa: E731
    kind = rng.choices(("linear", "layer", "dequantize", "repack", "dequantize_tiles"), (12, 3, 2, 1, 1))[0]
    if kind == "layer":
        return {"op": "layer", "hidden": 256 * _log(rng, 4, 20), "inter": 256 * _log(rng, 8, 68),
                "kv": _log(rng, 128, 1024), "graph": True, "m": _log(rng, 1, 32),
                "types": ",".join(str(t()) for _ in range(7))}
    k = 256 * _log(rng, 2, 68)
    if kind != "linear":
        n = _log(rng, 512, min(34816, 34816 * 5120 // k))
        return {"op": kind, "shards": "%d:%d" % (t(), n), "k": k,
                **({} if kind == "repack" else {"dtype": rng.choice(("bf16", "bf16", "fp16", "fp32"))})}
    m = _log(rng, 1, 8192)
    count = rng.choice((1, 1, 2, 3))
    most = min(36864, 34816 * 5120 // k, 8192 * 5120 * 17408 // (m * k))
    each = max(64, _log(rng, min(256, most), most) // count)
    types = [t() for _ in range(count)] if rng.random() < 0.5 else [t()] * count
    return {"op": "linear", "shards": ",".join("%d:%d" % (w, max(1, each - rng.randrange(64))) for w in types), "k": k,
            "m": m, "x": rng.choice(("bf16", "bf16", "bf16", "fp16")), "bias": rng.random() < 0.3,
            "graph": m <= 128 and rng.random() < 0.7}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _raw(gen, t, n, k):
    """Raw GGUF rows: uniform quantized fields (every bit pattern is valid), finite fp16 scales."""
    bw, bb = BLOCK[t]
    raw = torch.randint(0, 256, (n, k // bw, bb), dtype=torch.uint8, device="cuda", generator=gen)
    at, at_min, d, dmin = SCALE[t]
    for o, size in ((at, d), (at_min, dmin)):
        if o is not None:
            v = (torch.rand((n, k // bw), device="cuda", generator=gen) + 0.5) * size
            raw[:, :, o:o + 2] = v.to(torch.float16).view(torch.uint8).reshape(n, k // bw, 2)
    return raw.reshape(n, -1)


def _inputs(case, seed):
    """What both sides start from: per module (raw rows of each shard, x, bias)."""
    gen = _gen(seed)
    got = []
    for shards, k in _modules(case):
        raws = [_raw(gen, t, n, k) for t, n in shards]
        x = bias = None
        if "m" in case:
            x = torch.randn((case["m"], k), device="cuda", generator=gen).to(DTYPES[case.get("x", "bf16")])
            if case.get("bias"):
                bias = torch.randn(sum(n for _, n in shards), device="cuda", generator=gen).to(x.dtype)
        got.append((shards, k, raws, x, bias))
    return got


class _Type:
    def __init__(self, weight_type, shard_weight_type):
        self.weight_type = weight_type
        self.shard_weight_type = shard_weight_type


def _linear_layer(shards, raws):
    """A merged linear layer as the plugin's loader leaves it: one weight if its shards have one
    type, else a tensor per shard."""
    layer = torch.nn.Module()
    types = {i: t for i, (t, _) in enumerate(shards)}
    one = len(set(types.values())) == 1
    weight = torch.cat(raws) if one else torch.empty(0, dtype=torch.uint8, device="cuda")
    layer.weight = torch.nn.Parameter(weight, requires_grad=False)
    layer.weight_type = _Type(shards[0][0], types)
    if len(shards) > 1:
        layer.weight.shard_id = list(types)
        if not one:
            layer.gguf_shards = dict(enumerate(raws))
    return layer


def prepare(case, seed):
    got = _inputs(case, seed)
    if case["op"] in ("dequantize", "repack", "dequantize_tiles"):
        shards, k, raws, _, _ = got[0]
        t, n = shards[0]
        w = gguf_hip.repack_tiles(raws[0], n, t) if case["op"] == "dequantize_tiles" else raws[0]
        return {"op": case["op"], "w": w, "type": t, "n": n, "k": k, "dtype": DTYPES[case.get("dtype", "bf16")]}
    method = gguf_hip.GGUFLinearMethod()
    calls = []
    while got:
        shards, k, raws, x, bias = got.pop(0)
        layer = _linear_layer(shards, raws)
        del raws
        method.process_weights_after_loading(layer)
        calls.append((layer, x, bias))
    state = {"op": case["op"], "method": method, "calls": calls}
    if case["graph"]:
        _apply(state)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = _apply(state)
        state["graph"] = graph
    return state


def _apply(state):
    return [state["method"].apply(layer, x, bias) for layer, x, bias in state["calls"]]


def run(state):
    if state["op"] == "dequantize":
        return gguf_hip.ggml_dequantize(state["w"], state["type"], state["n"], state["k"], state["dtype"])
    if state["op"] == "dequantize_tiles":
        return gguf_hip.dequantize_tiles(state["w"], state["n"], state["k"], state["type"], state["dtype"])
    if state["op"] == "repack":
        return gguf_hip.repack_tiles(state["w"], state["n"], state["type"])
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _apply(state)


def work(case):
    nbytes = flops = 0
    for shards, k in _modules(case):
        packed = sum(n * _row_bytes(t, k) for t, n in shards)
        n = sum(n for _, n in shards)
        if case["op"] == "repack":
            nbytes += 2 * packed
        elif case["op"] in ("dequantize", "dequantize_tiles"):
            nbytes += packed + n * k * DTYPES[case["dtype"]].itemsize
        else:
            nbytes += packed + 2 * case["m"] * (k + n)
            flops += 2 * case["m"] * n * k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Decoded weights and repacked bytes are exact.  A product is rounded once to bf16 (1.7e-3
    against 64 bits), and above 16 rows its weights are rounded to bf16 first (2.4e-3); the
    largest single difference seen is one bf16 step of a value plus that noise."""
    return "exact" if case["op"] in ("dequantize", "repack", "dequantize_tiles") else {"rel": 1e-2, "max": 5e-2}


# ---- the same results in 64 bits, in plain torch ---------------------------------------------

KVALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)   # IQ4 values
# IQ3_S grid: 512 words of four magnitudes, a hex digit each
GRID = """
1111 3111 5111 b111 f111 1311 3311 5311 9311 d311 1511 3511 b511 7711 1911 5911 b911 f911 3b11 7b11 1d11 5d11 3f11 9f11 ff11 1131 3131 5131
9131 1331 3331 b331 1531 7531 f531 3731 b731 9931 3d31 bd31 5f31 1151 3151 b151 f151 1351 7351 d351 3551 b551 1751 9751 5951 b951 f951 3b51
7b51 1f51 7f51 7171 3371 b371 1571 5571 3771 7771 d771 9971 1b71 5b71 fd71 3f71 bf71 1191 7391 f391 3591 9591 5791 1991 7991 3b91 1f91 51b1
91b1 15b1 55b1 d5b1 77b1 39b1 b9b1 f9b1 ddb1 7fb1 d1d1 33d1 73d1 37d1 5bd1 3fd1 11f1 51f1 91f1 15f1 55f1 d5f1 77f1 1bf1 9bf1 1113 3113 5113
9113 1313 3313 7313 b313 f313 1513 5513 3713 9713 d713 9b13 db13 3d13 5f13 1133 3133 7133 d133 1333 9333 3533 1733 7733 3933 1b33 5b33 1f33
df33 1153 5353 b353 f353 1553 9553 5753 1953 7953 bb53 1d53 5f53 3173 9173 f173 1373 7373 3573 f573 1773 9773 3973 5d73 1f73 7193 b193 5393
9393 3793 7793 5993 d993 1b93 9b93 31b3 13b3 73b3 35b3 17b3 57b3 3bb3 15d3 95d3 f5d3 99d3 d9d3 31f3 71f3 13f3 53f3 35f3 b7f3 39f3 5df3 1ff3
1115 3115 7115 b115 f115 1315 5315 9315 d315 3515 7515 f515 1715 5715 3915 7915 b915 1b15 5b15 fd15 1f15 7f15 bf15 1135 5135 1335 7335 f335
5535 b535 3735 9735 5935 3b35 3155 9155 f155 3555 7555 1755 f755 3955 7b55 fb55 3f55 9f55 1175 5175 b175 3375 5575 9575 3775 7775 5975 1b75
dd75 3195 f195 1595 7595 5795 b795 3995 5f95 bf95 91b5 33b5 55b5 f7b5 19b5 7bb5 1fb5 11d5 51d5 f1d5 35d5 bbd5 3dd5 b1f5 33f5 d5f5 17f5 79f5
1bf5 5117 3317 7317 b317 f317 5517 3717 7717 b717 5917 9917 f917 3b17 7d17 3f17 3137 7137 b137 9337 3537 7537 1937 1d37 5f37 df37 1157 5357
1557 5757 9757 1b57 3177 1377 9377 3577 7577 f577 1777 3977 7977 f977 bb77 7f77 7197 3397 d397 5597 3797 5b97 1d97 9d97 31b7 13b7 53b7 b5b7
57b7 99b7 dbb7 7fb7 d3d7 39d7 31f7 71f7 15f7 55f7 b7f7 1119 9119 5319 1519 9519 f519 5719 3919 1b19 1f19 5139 f139 3339 7339 5539 1739 b739
7939 3b39 bb39 3159 7159 1359 b359 3559 7759 1959 fb59 5d59 1f59 9179 3379 7379 1579 5579 3779 b779 1199 5199 9599 f799 1999 3f99 b1b9 f1b9
35b9 5db9 73d9 97d9 1dd9 13f9 b3f9 17f9 79f9 3bf9 511b 131b 931b 551b 191b 991b f91b 5b1b dd1b 9f1b 313b 713b b13b 533b 353b 573b 5f3b 115b
335b 755b 175b d75b 7b5b 517b f17b 137b f57b 997b 3b7b bd7b 7f7b 319b 919b 159b 579b d99b 53bb d5bb 3bbb 7bbb 59db 51fb 91fb 55fb 331d 731d
b31d 371d 771d 1d1d 113d 153d f53d 9d3d 535d 975d 595d bb5d 5d5d 1f5d 117d 937d 357d 197d b59d 799d 5d9d 11bd 71bd 97bd 1dbd b1dd 19dd 33fd
73fd 111f 911f f11f 151f 551f d71f 191f 9b1f 5d1f 513f 333f 953f 793f b93f 315f 915f 135f d35f 355f 175f 3b5f 517f 577f b77f 7b7f 319f b19f
739f 159f 1b9f 55bf 59bf 51df 37df 11ff
"""


def _scales_k4(s):
    """The 12 packed scale bytes of Q4_K / Q5_K -> eight 6-bit scales and eight 6-bit mins."""
    low, mid, top = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    return (torch.cat([low & 63, (top & 15) | (low >> 6 << 4)], -1),
            torch.cat([mid & 63, (top >> 4) | (mid >> 6 << 4)], -1))


def _bits(v, width):
    """The width-bit fields of each byte of v (lowest first), a new axis before the last."""
    return torch.stack([(v >> (width * i)) & ((1 << width) - 1) for i in range(8 // width)], -2)


def _dequant(raw, t, n, k):
    """[n, k] weights in 64 bits: d * scale * q - dmin * min of each block."""
    bw, bb = BLOCK[t]
    raw = raw.reshape(n, k // bw, bb)
    b = raw.int()
    half = lambda o: raw[..., o:o + 2].contiguous().view(torch.float16).double()  # noqa: E731
    flat = lambda v: v.reshape(n, k // bw, -1)  # noqa: E731
    kv = torch.tensor(KVALUES, device=raw.device)
    d, minus = half(SCALE[t][0]), None
    sc = torch.ones_like(b[..., :1])
    if t == Q4_0:
        q = flat(_bits(b[..., 2:18], 4)) - 8
    elif t == IQ4_NL:
        q = kv[flat(_bits(b[..., 2:18], 4))]
    elif t == Q5_0:
        high = flat(_bits(b[..., 2:6], 1).transpose(-1, -2))
        q = (flat(_bits(b[..., 6:22], 4)) | high << 4) - 16
    elif t == Q8_0:
        q = raw[..., 2:].view(torch.int8).int()
    elif t == Q2_K:
        q = flat(_bits(b[..., 16:80].reshape(n, -1, 2, 32), 2))
        sc, minus = b[..., 0:16] & 15, half(82) * (b[..., 0:16] >> 4)
    elif t == Q3_K:
        q = flat(_bits(b[..., 32:96].reshape(n, -1, 2, 32), 2)) - 4 + 4 * flat(_bits(b[..., 0:32], 1))
        s = b[..., 96:108]
        sc = (flat(_bits(s[..., 0:8], 4)) | flat(_bits(s[..., 8:12], 2)) << 4) - 32
    elif t in (Q4_K, Q5_K):
        q = flat(_bits(b[..., bb - 128:].reshape(n, -1, 4, 32), 4))
        if t == Q5_K:
            q = q | flat(_bits(b[..., 16:48], 1)) << 4
        sc, m = _scales_k4(b[..., 4:16])
        minus = half(2) * m
    elif t == Q6_K:
        low = flat(_bits(b[..., 0:128].reshape(n, -1, 2, 64), 4))
        q = (low | flat(_bits(b[..., 128:192].reshape(n, -1, 2, 32), 2)) << 4) - 32
        sc = raw[..., 192:208].contiguous().view(torch.int8).int()
    elif t == IQ4_XS:
        q = kv[flat(_bits(b[..., 8:136].reshape(n, -1, 8, 16), 4))]
        low = flat(_bits(b[..., 4:8], 4).transpose(-1, -2))
        sc = (low | flat(_bits(b[..., 2:4], 2).transpose(-1, -2)) << 4) - 32
    else:   # IQ3_S: grid index = byte + a high bit, eight sign bits per eight weights
        grid = torch.tensor([[int(c, 16) for c in w] for w in GRID.split()], device=raw.device)
        at = b[..., 2:66] | flat(_bits(b[..., 66:74], 1).transpose(-1, -2)) << 8
        sign = 1 - 2 * flat(_bits(b[..., 74:106], 1).transpose(-1, -2))
        q = flat(grid[at.long()]) * sign
        sc = 1 + 2 * flat(_bits(b[..., 106:110], 4).transpose(-1, -2))
    w = (d * sc)[..., None] * q.reshape(n, k // bw, sc.shape[-1], -1)
    if minus is not None:
        w = w - minus[..., None]
    return w.reshape(n, k)


def _rows(raw, t, k):
    return torch.cat([_dequant(r, t, r.shape[0], k) for r in raw.split(1024)])


def exact(case, seed):
    if case["op"] == "repack":
        return None
    out = []
    for shards, k, raws, x, bias in _inputs(case, seed):
        if x is None:
            return _rows(raws[0], shards[0][0], k)
        y = torch.cat([x.double() @ _rows(r, t, k).t() for r, (t, _) in zip(raws, shards)], 1)
        out.append(y if bias is None else y + bias.double())
    return out
