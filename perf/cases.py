"""Performance cases of the quantized MoE expert-FFN path: whole layer calls through MoeLayerRunner, as a serving or
prompt-processing program makes them, over the formats, row counts and routers that the path is used with.

A case is a stack of `layers` MoE layers (the layers of a model that one pass goes through; each has its own weights,
router and hidden rows, since what lies between two MoE layers is not this package's), `rows` token rows a layer and:
  path     "decode" (few rows: generation and speculative verify) or "prefill" (the grouped GEMM path)
  tg, td   GGUF types of gate/up and down;  d, E, k, ff: d_model, experts, experts a token, expert intermediate size
  shared   type of an always-on expert of the same shape beside the routed ones ("" for none; td of it is `shared_td`)
  router   "softmax" or "sigmoid" (with a selection bias);  bf16: router weights held as bf16
  zipf     tokens per expert follow Zipf(zipf) through a router logit bias (0: the router's own logits alone)
  lognormal  the rows' L2 norms are log-normal with this sigma (0: N(0, 1) rows)
  graph    the pass was captured into a HIP graph once; a pass copies its rows in and replays it (a serving loop)
"""
import math
import re
from pathlib import Path

import torch

from hyper_amd import moe
from hyper_amd.formats import GType, activations, random_layer, row_bytes, zipf_logit_bias

DEV = "cuda"
# fp16 scale ranges of the synthetic weights, per type (hidden values of ordinary size)
D_RANGE = {"Q4_K": (1e-4, 4e-3), "Q5_K": (1e-4, 4e-3), "Q6_K": (1e-4, 4e-3), "IQ4_NL": (1e-3, 1e-2), "IQ4_XS": (1e-3, 1e-2),
           "IQ2_XS": (1e-3, 1e-2), "Q8_0": (1e-4, 1e-3), "MXFP4": (1e-2, 1e-1)}
_PLAIN = dict(layers=1, shared="", shared_td="", router="softmax", bf16=False, zipf=0.0, lognormal=0.0, graph=False)


def _case(name, path, tg, td, d, E, k, ff, rows, **more):
    return dict(_PLAIN, name=name, path=path, tg=tg, td=td, d=d, E=E, k=k, ff=ff, rows=rows, **more)


def listed():
    return [
        # one token through sixteen small-expert layers, the captured decode step of a serving loop (d 2048, 128
        # experts, top-8, ff 768): launch latency and the chain of dependent kernels
        _case("q4k decode 1, 16 layers", "decode", "Q4_K", "Q4_K", 2048, 128, 8, 768, 1, layers=16, graph=True),
        # one token through four wide layers called eagerly, the router in bf16
        _case("iq4xs decode 1, 4 layers", "decode", "IQ4_XS", "IQ4_XS", 4096, 288, 8, 1536, 1, layers=4, bf16=True),
        # two rows, 8-bit experts behind a sigmoid router with a selection bias, eight layers, eager
        _case("q8_0 decode 2, 8 layers", "decode", "Q8_0", "Q8_0", 2048, 64, 8, 1024, 2, layers=8, router="sigmoid"),
        # a 4-row speculative verify of a wide layer
        _case("iq4nl verify 4", "decode", "IQ4_NL", "IQ4_NL", 4096, 288, 8, 1536, 4),
        # an 8-row verify of a 2-bit large-expert layer with a shared expert
        _case("iq2xs verify 8", "decode", "IQ2_XS", "IQ2_XS", 7168, 384, 6, 2048, 8, shared="Q4_K", shared_td="Q4_K"),
        # a short ragged prompt (or a batch of sequences): most experts get one to three rows
        _case("q4k/q6k prefill 37", "prefill", "Q4_K", "Q6_K", 2048, 128, 8, 768, 37),
        # MXFP4 weights, a medium ragged prompt, fewer experts
        _case("mxfp4 prefill 131", "prefill", "MXFP4", "MXFP4", 2048, 64, 8, 1024, 131),
        # the 512-token prompt with skewed routing
        _case("q4k/q6k prefill 512", "prefill", "Q4_K", "Q6_K", 2048, 128, 8, 768, 512, zipf=1.1),
        # a ragged prompt through a wide layer of 32-value blocks
        _case("iq4nl prefill 509", "prefill", "IQ4_NL", "IQ4_NL", 4096, 288, 8, 1536, 509),
        # a ragged prompt through a wide layer of 256-value 4-bit blocks, skewed routing
        _case("iq4xs prefill 1000", "prefill", "IQ4_XS", "IQ4_XS", 4096, 288, 8, 1536, 1000, zipf=1.1),
        # one chunk of a long prompt: many small experts and a shared one
        _case("q5k/q6k chunk 2048", "prefill", "Q5_K", "Q6_K", 2048, 512, 10, 512, 2048, shared="Q5_K", shared_td="Q6_K",
              zipf=1.1, lognormal=0.5),
        # one chunk of a long prompt through a 2-bit large-expert layer with a shared expert: the largest call
        _case("iq2xs chunk 2048", "prefill", "IQ2_XS", "IQ2_XS", 7168, 384, 6, 2048, 2048, shared="Q4_K", shared_td="Q4_K"),
    ]


# layer families: (d, most experts, ff, format pairs, most rows of a decode call), sizes as the listed ones'
_FAMILIES = [
    (2048, 128, 768, [("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("Q5_K", "Q6_K"), ("IQ4_XS", "Q6_K")], 16),
    (4096, 288, 1536, [("IQ4_NL", "IQ4_NL"), ("IQ4_XS", "IQ4_XS"), ("Q4_K", "Q6_K"), ("IQ2_XS", "IQ4_NL")], 8),
    (7168, 384, 2048, [("IQ2_XS", "IQ2_XS")], 8),
    (2048, 512, 512, [("Q5_K", "Q6_K"), ("Q4_K", "Q4_K")], 16),
    (2048, 64, 1024, [("Q8_0", "Q8_0"), ("MXFP4", "MXFP4"), ("IQ4_NL", "Q6_K"), ("MXFP4", "Q6_K")], 16),
]


def draw(rng):
    d, E, ff, pairs, dec_rows = rng.choice(_FAMILIES)
    tg, td = rng.choice(pairs)
    k = rng.choice([6, 8, 10] if E > 64 else [2, 4, 8])
    if d == 7168:
        k = 6
    E -= rng.choice([0, 0, 1, 7, 28])
    path = "decode" if tg == "Q8_0" else rng.choice(["decode", "prefill", "prefill"])   # (8-bit experts: generation only)
    if path == "decode":
        rows = int(round(math.exp(rng.uniform(0, math.log(dec_rows)))))
    else:
        rows = int(round(math.exp(rng.uniform(math.log(9), math.log(1500 if d == 7168 else 2047)))))
    c = dict(_PLAIN, path=path, tg=tg, td=td, d=d, E=E, k=k, ff=ff, rows=rows, bf16=rng.random() < 0.2)
    if rng.random() < 0.3:
        c["shared"], c["shared_td"] = ("Q4_K", "Q4_K") if d == 7168 or tg.startswith("IQ") else (tg, td)
    elif rng.random() < 0.2:
        c["router"] = "sigmoid"
    if path == "prefill":
        c["zipf"] = rng.choice([0.0, 1.1])
    else:
        c["graph"] = rng.random() < 0.5
        c["layers"] = max(1, min(8, 16 // rows if d == 2048 else 4 // rows))
    return c


# ------------------------------------------------------------------ inputs

def _inputs(case, seed, i):
    """Layer i's raw inputs from the seed: (weights, shared expert or None, router weights, selection bias or None,
    hidden rows, logit bias or None)."""
    c, s = case, 1009 * int(seed) + 31 * i
    g = torch.Generator(device=DEV)
    g.manual_seed(s)
    L = random_layer(GType[c["tg"]], GType[c["td"]], c["E"], c["ff"], c["d"], seed=s + 1, device=DEV, d_range=D_RANGE[c["tg"]],
                     d_range_down=D_RANGE[c["td"]])
    S = None
    if c["shared"]:
        S = random_layer(GType[c["shared"]], GType[c["shared_td"]], 1, c["ff"], c["d"], seed=s + 2, device=DEV,
                         d_range=D_RANGE[c["shared"]], d_range_down=D_RANGE[c["shared_td"]])
    W = torch.randn(c["E"], c["d"], generator=g, device=DEV) * 0.02
    if c["bf16"]:
        W = W.to(torch.bfloat16)
    sel = torch.randn(c["E"], generator=g, device=DEV) * 0.05 if c["router"] == "sigmoid" else None
    x = activations(c["rows"], c["d"], g, DEV, lognormal=c["lognormal"] or None)
    b = zipf_logit_bias(c["rows"], c["E"], c["zipf"], g, DEV) if c["zipf"] else None
    return L, S, W, sel, x, b


class _State:
    pass


def prepare(case, seed):
    c, st = case, _State()
    st.path, st.runners, st.xs, st.biases, st.graph = c["path"], [], [], [], None
    for i in range(c["layers"]):
        L, S, W, sel, x, b = _inputs(c, seed, i)
        dev = moe.MoeDev(L, torch.arange(c["E"], dtype=torch.int32, device=DEV))
        sh = moe.MoeDev(S, torch.zeros(1, dtype=torch.int32, device=DEV)) if S is not None else None
        st.runners.append(moe.MoeLayerRunner(dev, W, c["k"], c["rows"], shared=sh, router=c["router"], router_bias=sel))
        st.xs.append(x)
        st.biases.append(b)
        del L, S
    if c["graph"]:
        # the serving loop's captured step, on rows of its own that every pass writes first
        st.inp = torch.stack(st.xs)
        st.rows = torch.zeros_like(st.inp)
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            st.outs = _layers(st, st.rows)
            side.synchronize()
            st.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st.graph, stream=side):
                st.outs = _layers(st, st.rows)
        torch.cuda.synchronize()
    return st


def _layers(st, xs):
    if st.path == "decode":
        return [r.decode(x, bias=b) for r, x, b in zip(st.runners, xs, st.biases)]
    return [r.prefill(x, bias=b) for r, x, b in zip(st.runners, xs, st.biases)]


def run(st):
    if st.graph is not None:
        st.rows.copy_(st.inp)
        st.graph.replay()
        return st.outs
    return _layers(st, st.xs)


# ------------------------------------------------------------------ what a pass cannot do without

def _expert_bytes(c, tg, td):
    return 2 * c["ff"] * row_bytes(GType[tg], c["d"]) + c["d"] * row_bytes(GType[td], c["ff"])


def _touched(c):
    """expected distinct experts of a layer call: each expert is missed by a row with probability 1 - (its share of k)"""
    E, k, T = c["E"], c["k"], c["rows"]
    if not c["zipf"]:
        return E * (1 - (1 - k / E) ** T)
    p = [1.0 / (r + 1) ** c["zipf"] for r in range(E)]
    t = sum(p)
    return sum(1 - (1 - min(1.0, k * v / t)) ** T for v in p)


def work(case):
    c = case
    T, d, ff = c["rows"], c["d"], c["ff"]
    by = _touched(c) * _expert_bytes(c, c["tg"], c["td"]) + c["E"] * d * (2 if c["bf16"] else 4) + 2 * T * d * 4
    fl = 2.0 * T * (c["k"] * 3 * ff * d + c["E"] * d)
    if c["shared"]:
        by += _expert_bytes(c, c["shared"], c["shared_td"])
        fl += 2.0 * T * 3 * ff * d
    if c["zipf"]:
        by += T * c["E"] * 4
    return {"bytes": c["layers"] * by, "flops": c["layers"] * fl}


def tolerance(case):
    # Weights, activations and block integers are the formats' own and exact; what may differ is the order of 32-bit
    # sums, and through it the rounding of a hidden value to its 8-bit block now and then (one step of 1/127 of the
    # block's largest value).  Against 64 bits throughout, the path is off by 6e-8 (no such step) to 1.7e-3 (a step in
    # a large hidden row of a short prompt) relative over these cases: four times the most seen.
    return {"rel": 6e-3, "max": 0.3}


# ------------------------------------------------------------------ the same in 64 bits, plain torch

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _k4_scales(s):
    """the eight 6-bit scales and mins of a K-quant's 12 bytes s [.., 12]"""
    lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    return torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1), torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1)


_KV = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]   # the IQ4 codebook
_FP4 = [0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12]                    # twice the E2M1 values
_grid_cache = {}


def _iq2xs_grid():
    if not _grid_cache:   # the format's codebook, 512 rows of 8 values, kept in the tree as base-3 numbers
        text = re.sub(r"//.*", "", (Path(__file__).resolve().parents[1] / "hyper_amd/csrc/iq2xs_grid.inc").read_text())
        codes = [int(v) for v in re.findall(r"\d+", text)]
        rows = [[(8, 25, 43)[(code // 3 ** i) % 3] for i in range(8)] for code in codes]
        _grid_cache["g"] = torch.tensor(rows, dtype=torch.float64, device=DEV)
        signs = [[-1.0 if ((i | (bin(i).count("1") & 1) << 7) >> j) & 1 else 1.0 for j in range(8)] for i in range(128)]
        _grid_cache["s"] = torch.tensor(signs, dtype=torch.float64, device=DEV)
    return _grid_cache["g"], _grid_cache["s"]


def _dequant(t, raw, n):
    """rows of GGUF blocks [R, bytes] -> float64 [R, n]"""
    R = raw.shape[0]
    if t in ("IQ4_NL", "Q8_0", "MXFP4"):
        b = raw.view(R, n // 32, -1)
        if t == "Q8_0":
            return (_f16(b[..., 0:2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(R, n)
        at = 1 if t == "MXFP4" else 2
        qs = b[..., at:].long()
        table = torch.tensor(_FP4 if t == "MXFP4" else _KV, dtype=torch.float64, device=raw.device)
        v = table[torch.cat([qs & 15, qs >> 4], -1)]
        s = torch.exp2(b[..., 0:1].double() - 128) if t == "MXFP4" else _f16(b[..., 0:2])
        return (s * v).reshape(R, n)
    b = raw.view(R, n // 256, -1)
    i = b.int()
    if t in ("Q4_K", "Q5_K"):
        sc, mn = _k4_scales(i[..., 4:16])
        qs = i[..., 16 if t == "Q4_K" else 48:].view(R, n // 256, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 3).view(R, n // 256, 8, 32)
        if t == "Q5_K":
            bit = torch.arange(8, device=raw.device, dtype=torch.int32).view(1, 1, 8, 1)
            q = q | (((i[..., None, 16:48] >> bit) & 1) << 4)
        d, dmin = _f16(b[..., 0:2])[..., None], _f16(b[..., 2:4])[..., None]
        return (d * (sc[..., None] * q).double() - dmin * mn[..., None].double()).reshape(R, n)
    if t == "Q6_K":
        ql, qh = i[..., 0:128].view(R, -1, 2, 2, 32), i[..., 128:192].view(R, -1, 2, 32)
        low = torch.stack([ql & 15, ql >> 4], 3)                       # [.., half, nibble, 32-group of the nibble, 32]
        high = torch.stack([(qh >> (2 * j)) & 3 for j in range(4)], 3).view(R, -1, 2, 2, 2, 32)
        q = ((low | (high << 4)) - 32).view(R, -1, 16, 16)
        sc = b[..., 192:208].contiguous().view(torch.int8).int()
        return (_f16(b[..., 208:210])[..., None] * (sc[..., None] * q).double()).reshape(R, n)
    if t == "IQ4_XS":
        sh = i[..., 2] | (i[..., 3] << 8)
        ls = torch.stack([((i[..., 4 + j // 2] >> (4 * (j & 1))) & 15) | (((sh >> (2 * j)) & 3) << 4) for j in range(8)], -1) - 32
        qs = b[..., 8:].long().view(R, -1, 8, 16)
        v = torch.tensor(_KV, dtype=torch.float64, device=raw.device)[torch.cat([qs & 15, qs >> 4], -1)]
        return (_f16(b[..., 0:2])[..., None] * ls[..., None].double() * v).reshape(R, n)
    if t == "IQ2_XS":
        grid, signs = _iq2xs_grid()
        q = b[..., 2:66].contiguous().view(torch.int16).long() & 0xFFFF          # [.., 32] 8-value groups
        v = (grid[q & 511] * signs[q >> 9]).view(R, -1, 16, 16)
        sc = torch.stack([i[..., 66:74] & 15, i[..., 66:74] >> 4], -1).view(R, -1, 16, 1)
        return (_f16(b[..., 0:2])[..., None] * 0.125 * (2 * sc + 1).double() * v).reshape(R, n)
    raise ValueError(t)


def _q8(t, x):
    """float64 rows through the 8-bit activation blocks that weights of type t are multiplied with"""
    R, n = x.shape
    if t in ("IQ4_NL", "Q8_0", "MXFP4"):   # 32 values, scale amax / 127 held in 16 bits
        b = x.view(R, -1, 32)
        a = b.abs().amax(-1, keepdim=True)
        q = torch.round(b * torch.where(a > 0, 127.0 / a, torch.zeros_like(a)))
        return (q * (a / 127.0).to(torch.float16).double()).view(R, n)
    b = x.view(R, -1, 256)                 # 256 values, scale from the value of largest magnitude
    top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    inv = torch.where(top != 0, -127.0 / top, torch.zeros_like(top))
    q = torch.round(b * inv).clamp(max=127)
    return (q * torch.where(top != 0, top / -127.0, torch.zeros_like(top))).view(R, n)


def _ffn(tg, td, gate, up, down, xq, d, ff):
    g, u = xq @ _dequant(tg, gate, d).T, xq @ _dequant(tg, up, d).T
    return _q8(td, g * torch.sigmoid(g) * u) @ _dequant(td, down, ff).T


def exact(case, seed):
    c, outs = case, []
    for i in range(c["layers"]):
        L, S, W, sel, x, b = _inputs(c, seed, i)
        X = x.double()
        logits = X @ W.double().T
        if b is not None:
            logits = logits + b.double()
        p = torch.sigmoid(logits) if sel is not None else torch.softmax(logits, -1)
        ids = torch.topk(p + sel.double() if sel is not None else p, c["k"], -1).indices
        w = p.gather(1, ids)
        w = w / w.sum(-1, keepdim=True)
        out = torch.zeros_like(X)
        xq = _q8(c["tg"], X)
        for e in torch.unique(ids).tolist():
            t, j = (ids == e).nonzero(as_tuple=True)
            y = _ffn(c["tg"], c["td"], L.gate[e], L.up[e], L.down[e], xq[t], c["d"], c["ff"])
            out[t] += w[t, j][:, None] * y
        if S is not None:
            out += _ffn(c["shared"], c["shared_td"], S.gate[0], S.up[0], S.down[0], _q8(c["shared"], X), c["d"], c["ff"])
        outs.append(out)
        del L, S
    return outs
