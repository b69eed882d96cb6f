"""What this framework's users have it compute, as cases that can be timed and checked.

A case is one call (or, for the decode step, one indexer-to-attention sequence) of the sparse-MLA
path through its public entry points in ``smla``, over the sizes of the layer that the package is
for: model width 4096, 64 heads, 512 latent + 64 rope dims, a 128-row window, block-4 compressed
rows, 64 indexer heads of 64 or 128 dims.  The kinds:

* ``linear``       ``mla.linear``: a projection of 1 .. 8192 tokens by one of the layer's weights,
                   bf16 (serving) or fp32 (the reference's own precision).
* ``o_project``    ``mla.o_project``: inverse RoPE, grouped product and output product.
* ``decode``       ``indexer.index_decode`` then ``sparse_attn_two_source``: the decode step's
                   index build and attention over a window ring and a compressed cache.
* ``fp8_rows``     ``sparse_attn_batched`` over e4m3 rows with per-64 scales, ragged sequences.
* ``prompt_attn``  ``prefill_attn``: a prompt's (or a later prompt chunk's) attention.
* ``prompt_index`` indexer scores and top-k selection of every query of a prompt chunk, over keys
                   in the stored fp4 form or e4m3.
* ``compress``     ``compressor_prefill``: projections and gated pooling of a prompt.
* ``layer_prompt`` ``DecodeLayer.prefill``: a whole attention layer over one prompt.
* ``layer_step``   ``DecodeLayer.step``: the layer's decode step for a batch of sequences.

``exact`` restates each in float64 with plain torch.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deepseek-v4-flash-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from smla import compressor, engine, indexer, mla, norm_rope, qat, sparse_attn, workloads  # noqa: E402

DEV = "cuda"
DIM, HEADS, HD, LATENT, ROPE, WINDOW = 4096, 64, 512, 576, 64, 128
GROUPS, RANK = 8, 1024
SCALE = workloads.SCALE_576
YARN, PLAIN = (65536, 160000.0, 16, 32, 1), (0, 10000.0, 40, 32, 1)
# the layer's weights [out, in]: the q down and up projections, the kv projection, the output product
WEIGHTS = {"wq_a": (1024, 4096), "wq_b": (32768, 1024), "wkv": (512, 4096), "wo_b": (4096, 8192)}


def listed():
    return [
        # one token of one sequence through the q down projection: the smallest call of a decode step
        {"name": "linear_token", "kind": "linear", "T": 1, "weight": "wq_a", "dtype": "bf16"},
        # a serving batch of 64 sequences through the output product
        {"name": "linear_batch", "kind": "linear", "T": 64, "weight": "wo_b", "dtype": "bf16"},
        # the attention output path of a 300-token prompt chunk, and of a whole 4096-token prompt
        {"name": "o_project_chunk", "kind": "o_project", "T": 300},
        {"name": "o_project_prompt", "kind": "o_project", "T": 4096},
        # the decode step at 32K context for 8 sequences: 8192 compressed rows, top 2048 and the window
        {"name": "decode_32k", "kind": "decode", "B": 8, "N": 8192, "k": 2048},
        # 64 sequences of 2048 .. 16384 fp8 rows, 2048 of them attended
        {"name": "fp8_rows_64", "kind": "fp8_rows", "B": 64, "lo": 2048, "hi": 16384, "k": 2048},
        # a 4096-token prompt, and a ragged chunk that continues a prompt of 7683 tokens
        {"name": "prompt_attn_4k", "kind": "prompt_attn", "S": 4096, "pos0": 0, "D": 576},
        {"name": "prompt_attn_chunk", "kind": "prompt_attn", "S": 509, "pos0": 7683, "D": 576},
        # the index build of a 1024-token chunk at position 7168: 128-dim fp4 keys, top 512
        {"name": "prompt_index_1k", "kind": "prompt_index", "S": 1024, "pos0": 7168, "Di": 128, "keys": "fp4", "k": 512},
        # the compressor over a 2046-token prompt in the reference's fp32 (a remainder of 2 tokens)
        {"name": "compress_fp32", "kind": "compress", "S": 2046, "dtype": "fp32", "form": "plain"},
        # a ratio-4 attention layer: a 4096-token prompt, and a step of 8 sequences deep in their contexts
        {"name": "layer_prompt_4k", "kind": "layer_prompt", "S": 4096, "ratio": 4},
        {"name": "layer_step_8", "kind": "layer_step", "B": 8, "ratio": 4, "max_pos": 32768},
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "o_project", "decode", "fp8_rows", "prompt_attn", "prompt_index",
                       "compress", "layer_prompt", "layer_step"])
    if kind == "linear":
        dt = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        return {"kind": kind, "T": _logint(rng, 1, 8192 if dt == "bf16" else 2048),
                "weight": rng.choice(sorted(WEIGHTS)), "dtype": dt}
    if kind == "o_project":
        return {"kind": kind, "T": _logint(rng, 1, 4096)}
    if kind == "decode":
        return {"kind": kind, "B": _logint(rng, 1, 32), "N": _logint(rng, 200, 16384), "k": rng.choice([512, 1024, 2048])}
    if kind == "fp8_rows":
        lo = _logint(rng, 256, 4096)
        return {"kind": kind, "B": _logint(rng, 2, 64), "lo": lo, "hi": rng.randint(2 * lo, 4 * lo),
                "k": rng.choice([512, 1024, 2048])}
    if kind == "prompt_attn":
        return {"kind": kind, "S": _logint(rng, 16, 2048), "pos0": rng.choice([0, rng.randint(1, 12000)]),
                "D": rng.choice([512, 576])}
    if kind == "prompt_index":
        return {"kind": kind, "S": _logint(rng, 32, 1024), "pos0": rng.randint(1024, 12000),
                "Di": rng.choice([64, 128]), "keys": rng.choice(["fp4", "fp8"]), "k": rng.choice([256, 512])}
    if kind == "compress":
        return {"kind": kind, "S": _logint(rng, 16, 4096), "dtype": rng.choice(["bf16", "fp32"]),
                "form": rng.choice(["plain", "fp8", "rotate"])}
    if kind == "layer_prompt":
        return {"kind": kind, "S": _logint(rng, 16, 4096), "ratio": rng.choice([0, 4])}
    return {"kind": "layer_step", "B": _logint(rng, 1, 32), "ratio": rng.choice([0, 4, 4, 128]),
            "max_pos": rng.choice([4096, 16384, 32768])}


# ---------------------------------------------------------------------------------------------
# inputs

class _Draw:
    """Seeded tensors made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std).to(dtype)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=torch.int32)

    def around_one(self, *shape):
        return 1.0 + 0.1 * torch.randn(*shape, generator=self.g, device=DEV)


def _layer_weights(r, ratio):
    bf = lambda *s: r.normal(*s, std=0.02, dtype=torch.bfloat16)  # noqa: E731
    w = dict(wq_a=bf(1024, DIM), q_a_norm=r.around_one(1024), wq_b=bf(HEADS * HD, 1024), wkv=bf(HD, DIM),
             kv_a_norm=r.around_one(HD), wo_a=bf(GROUPS * RANK, HEADS * HD // GROUPS), wo_b=bf(DIM, GROUPS * RANK),
             sinks=r.around_one(HEADS))
    if ratio == 4:
        w.update(wkv_c=bf(2 * HD, DIM), wgate_c=bf(2 * HD, DIM), ape=r.normal(4, 2 * HD, std=0.1), norm_c=r.around_one(HD))
    return engine.LayerWeights(**w)


def _nvis(c):
    """Compressed rows visible to each query of a chunk at positions pos0 .. pos0+S-1."""
    return (torch.arange(c["S"], device=DEV, dtype=torch.int32) + c["pos0"] + 1) // 4


def prepare(case, seed):
    c, r, kind = case, _Draw(seed), case["kind"]
    st = {"case": dict(case)}
    bf = torch.bfloat16
    if kind == "linear":
        n, k = WEIGHTS[c["weight"]]
        dt = bf if c["dtype"] == "bf16" else torch.float32
        st.update(x=r.normal(c["T"], k, dtype=dt), w=r.normal(n, k, std=0.02, dtype=dt))
    elif kind == "o_project":
        cos_t, sin_t = norm_rope.rope_tables(ROPE, 65536, *YARN, device=DEV)
        st.update(o=r.normal(c["T"], HEADS, HD, std=0.5, dtype=bf), pos=r.ints(0, 65536, c["T"]), cos=cos_t, sin=sin_t,
                  wo_a=r.normal(GROUPS * RANK, HEADS * HD // GROUPS, std=0.02, dtype=bf),
                  wo_b=r.normal(DIM, GROUPS * RANK, std=0.02, dtype=bf))
    elif kind == "decode":
        B, N = c["B"], c["N"]
        codes, ks = workloads.quant_e4m3_pow2(r.normal(B, N, 64), block=64)
        # queries aligned enough with the rows that the attention weights differ from row to row
        st.update(q=r.normal(B, 1, HEADS, LATENT, std=1.0, dtype=bf), raw=r.normal(B, WINDOW, LATENT, dtype=bf),
                  comp=r.normal(B, N, LATENT, dtype=bf), sink=r.normal(HEADS), q_idx=r.normal(B, 1, 64, 64, dtype=bf),
                  codes=codes, kscale=ks.reshape(B, N), w=r.normal(B, 1, 64), nvis=torch.full((B, 1), N, dtype=torch.int32, device=DEV),
                  pos=r.ints(4 * N - 1, 4 * N + 3, B))
    elif kind == "fp8_rows":
        B, hi, k = c["B"], c["hi"], c["k"]
        lens = r.ints(c["lo"], hi + 1, B)
        codes, scales = workloads.quant_e4m3_pow2(r.normal(B, hi, LATENT))
        # k distinct rows of each sequence in ascending order, all rows (then -1) where it has fewer
        key = torch.rand(B, hi, generator=r.g, device=DEV)
        key[torch.arange(hi, device=DEV)[None] >= lens[:, None]] = 2.0
        top = torch.topk(key, min(k, hi), dim=1, largest=False)
        idx = torch.where(top.values < 1.5, top.indices, torch.full_like(top.indices, hi)).sort(dim=1).values
        idx = torch.where(idx < hi, idx, torch.full_like(idx, -1)).to(torch.int32)
        idx = torch.nn.functional.pad(idx, (0, k - idx.shape[1]), value=-1)
        st.update(q=r.normal(B, 1, HEADS, LATENT, dtype=bf), codes=codes, scales=scales, idx=idx[:, None].contiguous(),
                  sink=r.normal(HEADS))
    elif kind == "prompt_attn":
        n = c["pos0"] + c["S"]
        st.update(q=r.normal(1, c["S"], HEADS, c["D"], dtype=bf), raw=r.normal(1, n, c["D"], dtype=bf),
                  comp=r.normal(1, max(1, n // 4), c["D"], dtype=bf), sink=r.normal(HEADS))
    elif kind == "prompt_index":
        N, Di = (c["pos0"] + c["S"]) // 4, c["Di"]
        k = r.normal(1, N, Di)
        if c["keys"] == "fp4":
            keys, ks = qat.fp4_pack(k)
        else:
            keys, ks = workloads.quant_e4m3_pow2(k, block=Di)
            ks = ks.reshape(1, N)
        st.update(q=r.normal(1, c["S"], 64, Di, dtype=bf), keys=keys, ks=ks, w=r.normal(1, c["S"], 64),
                  nvis=_nvis(c)[None].contiguous())
    elif kind == "compress":
        d = 128 if c["form"] == "rotate" else HD
        dt = bf if c["dtype"] == "bf16" else torch.float32
        st.update(x=r.normal(1, c["S"], DIM, dtype=dt), wkv=r.normal(2 * d, DIM, std=0.02, dtype=dt),
                  wgate=r.normal(2 * d, DIM, std=0.02, dtype=dt), ape=r.normal(4, 2 * d, std=0.1), norm=r.around_one(d), d=d)
    elif kind == "layer_prompt":
        w = _layer_weights(r, c["ratio"])
        st.update(w=w, layer=engine.DecodeLayer(w, 1, c["ratio"], max_pos=8192, device=DEV),
                  xn=r.normal(1, c["S"], DIM, dtype=bf))
    else:  # layer_step: caches as a long decode leaves them, every sequence at a position of its own
        w = _layer_weights(r, c["ratio"])
        layer = engine.DecodeLayer(w, c["B"], c["ratio"], max_pos=c["max_pos"], device=DEV)
        layer.raw.copy_(r.normal(*layer.raw.shape, dtype=bf))
        if c["ratio"] == 4:
            layer.comp.copy_(r.normal(*layer.comp.shape, dtype=bf))
            layer.ring.ring_kv.copy_(r.normal(*layer.ring.ring_kv.shape))
            layer.ring.ring_sc.copy_(r.normal(*layer.ring.ring_sc.shape))
        # not the last position of a block of 4: the step then writes the same rows every time, so
        # that it can be repeated on the same state
        pos = 4 * r.ints(c["max_pos"] // 8, c["max_pos"] // 4, c["B"]) + r.ints(0, 3, c["B"])
        st.update(w=w, layer=layer, xn=r.normal(c["B"], DIM, dtype=bf), pos=pos,
                  raw0=layer.raw.clone(), comp0=layer.comp)
    return st


# ---------------------------------------------------------------------------------------------
# the calls

def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "linear":
        return mla.linear(st["x"], st["w"])
    if kind == "o_project":
        return mla.o_project(st["o"], st["pos"], st["cos"], st["sin"], st["wo_a"], st["wo_b"])
    if kind == "decode":
        ids = indexer.index_decode(st["q_idx"], st["codes"], st["kscale"], st["w"], st["nvis"], c["k"], st["pos"], WINDOW, WINDOW)
        o = sparse_attn.sparse_attn_two_source(st["q"], st["raw"], st["comp"], st["sink"], ids[:, None], SCALE, dv=HD)
        return {"ids": ids, "o": o}
    if kind == "fp8_rows":
        return sparse_attn.sparse_attn_batched(st["q"], st["codes"], st["sink"], st["idx"], SCALE, dv=HD, kv_scale=st["scales"])
    if kind == "prompt_attn":
        return sparse_attn.prefill_attn(st["q"], st["raw"], st["comp"], st["sink"], c["D"] ** -0.5, q_pos0=c["pos0"])
    if kind == "prompt_index":
        if c["keys"] == "fp4":
            s = indexer.indexer_score_fp4(st["q"], st["keys"], st["ks"], None, st["w"], st["nvis"])
        else:
            s = indexer.indexer_score(st["q"], st["keys"], st["ks"], st["w"], st["nvis"])
        return {"scores": s, "ids": indexer.topk(s, c["k"], nvis=st["nvis"])}
    if kind == "compress":
        kv, state = compressor.compressor_prefill(st["x"], st["wkv"], st["wgate"], st["ape"], st["norm"], head_dim=st["d"],
                                                  fp8_sim=c["form"] == "fp8", rotate=c["form"] == "rotate")
        return {"rows": kv, "state": state}
    if kind == "layer_prompt":
        y = st["layer"].prefill(st["xn"])
        return {"y": y, "window": st["layer"].raw, "comp": st["layer"].comp[:, : c["S"] // 4]}
    return {"y": st["layer"].step(st["xn"], st["pos"]), "window": st["layer"].raw}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without

def _pairs(S, pos0, ratio, n_comp):
    p = torch.arange(pos0, pos0 + S)
    n = torch.clamp(p + 1, max=WINDOW)
    return int((n + (torch.clamp((p + 1) // ratio, max=n_comp) if ratio else 0)).sum())


def _w_bytes(ratio):
    n = 1024 * DIM + HEADS * HD * 1024 + HD * DIM + 2 * GROUPS * RANK * DIM + (4 * HD * DIM if ratio == 4 else 0)
    return 2 * n


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        (n, k), es = WEIGHTS[c["weight"]], 2 if c["dtype"] == "bf16" else 4
        return {"bytes": es * (c["T"] * (n + k) + n * k), "flops": 2 * c["T"] * n * k}
    if kind == "o_project":
        T, mid = c["T"], GROUPS * RANK
        return {"bytes": 2 * (T * (HEADS * HD + DIM) + 2 * mid * DIM), "flops": 4 * T * mid * DIM}
    if kind == "decode":
        B, N = c["B"], c["N"]
        rows = WINDOW + min(c["k"], N)
        return {"bytes": B * (N * 68 + 64 * 130 + 4 * (WINDOW + c["k"]) + rows * LATENT * 2 + HEADS * (LATENT + HD) * 2),
                "flops": B * (2 * N * 64 * 64 + 2 * rows * HEADS * (LATENT + HD))}
    if kind == "fp8_rows":
        rows = min(c["k"], (c["lo"] + c["hi"]) // 2)
        return {"bytes": c["B"] * (rows * (LATENT + 36 + 4) + HEADS * (LATENT + HD) * 2),
                "flops": c["B"] * 2 * rows * HEADS * (LATENT + HD)}
    if kind == "prompt_attn":
        S, n, D = c["S"], c["pos0"] + c["S"], c["D"]
        rows = min(n, S + WINDOW - 1) + n // 4
        return {"bytes": 2 * (S * HEADS * (D + HD) + rows * D), "flops": 2 * _pairs(S, c["pos0"], 4, n // 4) * HEADS * (D + HD)}
    if kind == "prompt_index":
        S, N, Di = c["S"], (c["pos0"] + c["S"]) // 4, c["Di"]
        vis = sum((c["pos0"] + i + 1) // 4 for i in range(S))
        key = Di // 2 + Di // 32 if c["keys"] == "fp4" else Di + 4
        return {"bytes": S * (64 * (2 * Di + 4) + 4 * N + 4 * c["k"]) + N * key, "flops": 2 * vis * 64 * Di}
    if kind == "compress":
        es, d = 2 if c["dtype"] == "bf16" else 4, 128 if c["form"] == "rotate" else HD
        return {"bytes": es * DIM * (c["S"] + 4 * d) + 4 * d * (c["S"] // 4), "flops": 2 * c["S"] * 4 * d * DIM}
    if kind == "layer_prompt":
        S, r = c["S"], c["ratio"]
        proj = _w_bytes(r) // 2 * 2 * S
        attn = 2 * _pairs(S, 0, r, S // 4 if r else 0) * HEADS * 2 * HD
        return {"bytes": _w_bytes(r) + 2 * S * 2 * DIM, "flops": proj + attn}
    B, r = c["B"], c["ratio"]
    rows = WINDOW + (3 * c["max_pos"] // 16 if r == 4 else 0)  # positions average three quarters of max_pos
    return {"bytes": _w_bytes(r) + B * (4 * DIM + rows * HD * 2), "flops": B * (_w_bytes(r) + 4 * rows * HEADS * HD)}


# ---------------------------------------------------------------------------------------------
# tolerances: about four times the distance from exact() at these sizes (relative / largest): linear
# 1.7e-3 / 4e-3 (bf16) and 1.6e-6 / 1.4e-5 (fp32), the output path and attention 2.6e-3 / 1.4e-2, the
# plain compressor 1.6e-6 / 1.6e-5, the layer 4.3e-3 / 3.5e-2

def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 7e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 7e-6, "max": 6e-5}
    if kind == "prompt_index":
        return "exact"  # scores are defined as one fixed chain of fp32 operations, ids by exact ranks
    if kind == "compress":
        # quantised rows: a value on a rounding boundary moves by one step of its format (1/16 .. 1/8
        # of it in e4m3, up to half of it in e2m1), which a short prompt's few values show
        return {"plain": {"rel": 7e-6, "max": 7e-5}, "fp8": {"rel": 5e-3, "max": 0.3}, "rotate": {"rel": 2e-2, "max": 0.7}}[case["form"]]
    if kind in ("layer_prompt", "layer_step"):
        return {"rel": 1.7e-2, "max": 0.5}  # the window rows hold e4m3 values, as above
    return {"rel": 1e-2, "max": 6e-2}


# ---------------------------------------------------------------------------------------------
# the same in float64

def _rms64(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    return y if w is None else y * w.double()


def _rope64(x, cos_t, sin_t, inverse=False):
    """Interleaved pairs of the last 64 dims of x [T, heads, d] by tables rows [T, 32]."""
    c, s = cos_t.double()[:, None], sin_t.double()[:, None]
    s = -s if inverse else s
    y = x.clone()
    a, b = x[..., -ROPE::2], x[..., -ROPE + 1::2]
    y[..., -ROPE::2], y[..., -ROPE + 1::2] = a * c - b * s, a * s + b * c
    return y


def _fp8_64(x):
    """The e4m3 round trip of the last dim in blocks of 64 with power-of-two scales."""
    b = x.reshape(*x.shape[:-1], -1, 64)
    s = torch.exp2(torch.ceil(torch.log2(b.abs().amax(-1, keepdim=True).clamp_min(1e-4) / 448.0)))
    return ((b / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s).reshape(x.shape)


def _attn64(q, rows, sink, mask, scale, dv):
    """q [s, h, d], rows [n, d], mask [s, n] -> [s, h, dv]; all float64."""
    s, h, d = q.shape
    x = ((q.reshape(s * h, d) @ rows.t()) * scale).reshape(s, h, -1)
    x = x.masked_fill(~mask[:, None], float("-inf"))
    m = x.amax(-1, keepdim=True)
    p = (x - m).exp()
    den = p.sum(-1, keepdim=True) + (sink.double()[None, :, None] - m).exp()
    return ((p / den).reshape(s * h, -1) @ rows[:, :dv]).reshape(s, h, dv)


def _prompt64(q, raw, comp, sink, pos0, ratio, scale, dv):
    """Every query of a chunk over its window and the compressed rows visible to it."""
    out = []
    for s0 in range(0, q.shape[0], 128):
        p = torch.arange(pos0 + s0, pos0 + min(s0 + 128, q.shape[0]), device=q.device)
        lo = max(0, int(p[0]) - WINDOW + 1)
        r = torch.arange(lo, int(p[-1]) + 1, device=q.device)
        rows, mask = raw[lo:int(p[-1]) + 1], (r[None] <= p[:, None]) & (r[None] > p[:, None] - WINDOW)
        if ratio and comp is not None:
            j = torch.arange(comp.shape[0], device=q.device)
            rows, mask = torch.cat([rows, comp]), torch.cat([mask, j[None] < ((p + 1) // ratio)[:, None]], 1)
        out.append(_attn64(q[s0:s0 + 128].double(), rows.double(), sink, mask, scale, dv))
    return torch.cat(out)


def _pool64(kv, sc, ape, norm, fp8):
    """Gated overlapped pooling of kv, sc [n, 2d] (n a multiple of 4), norm, RoPE, e4m3 round trip."""
    d = kv.shape[1] // 2
    kv, sc = kv.reshape(-1, 4, 2 * d), sc.reshape(-1, 4, 2 * d) + ape.double()
    none = torch.full_like(sc[:1, :, :d], float("-inf"))
    s8 = torch.cat([torch.cat([none, sc[:-1, :, :d]]), sc[:, :, d:]], 1)
    k8 = torch.cat([torch.cat([torch.zeros_like(none), kv[:-1, :, :d]]), kv[:, :, d:]], 1)
    y = _rms64((k8 * torch.softmax(s8, 1)).sum(1), norm)
    cos_t, sin_t = _tables(4 * y.shape[0], YARN)
    y = _rope64(y[:, None], cos_t[::4], sin_t[::4])[:, 0]
    return torch.cat([_fp8_64(y[:, :d - ROPE]), y[:, d - ROPE:]], 1) if fp8 else y


def _tables(n, args):
    """cos, sin [n, 32] of the rotation by position: YaRN frequencies, or the plain ones."""
    orig, base, factor, fast, slow = args
    f = 1.0 / base ** (torch.arange(0, ROPE, 2, dtype=torch.float32) / ROPE)
    if orig:
        corr = lambda r: ROPE * math.log(orig / (r * 2 * math.pi)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(corr(fast)), 0), min(math.ceil(corr(slow)), ROPE - 1)
        ramp = ((torch.arange(ROPE // 2, dtype=torch.float32) - lo) / (hi - lo)).clamp(0, 1)
        f = f / factor * ramp + f * (1 - ramp)
    ang = torch.outer(torch.arange(n, dtype=torch.float32), f)  # the angles themselves are defined in fp32
    return ang.cos().to(DEV), ang.sin().to(DEV)


def _o_project64(o, cos_t, sin_t, wo_a, wo_b):
    o = _rope64(o.double(), cos_t, sin_t, inverse=True).reshape(o.shape[0], GROUPS, -1)
    wa = wo_a.reshape(GROUPS, RANK, -1)
    mid = torch.cat([o[:, g] @ wa[g].double().t() for g in range(GROUPS)], 1)
    return mid @ wo_b.double().t()


def _qkv64(x, w, cos_t, sin_t):
    q = _rms64(x @ w.wq_a.double().t(), w.q_a_norm) @ w.wq_b.double().t()
    q = _rope64(_rms64(q.reshape(-1, HEADS, HD)), cos_t, sin_t)
    kv = _rope64(_rms64(x @ w.wkv.double().t(), w.kv_a_norm)[:, None], cos_t, sin_t)[:, 0]
    return q, torch.cat([_fp8_64(kv[:, :HD - ROPE]), kv[:, HD - ROPE:]], 1)


def exact(case, seed):
    c, kind = case, case["kind"]
    st = prepare(case, seed)
    if kind == "linear":
        return st["x"].double() @ st["w"].double().t()
    if kind == "o_project":
        p = st["pos"].long()
        return _o_project64(st["o"], st["cos"][p], st["sin"][p], st["wo_a"], st["wo_b"])
    if kind == "decode":
        o, key = [], st["codes"].view(torch.float8_e4m3fn).double()
        for b in range(c["B"]):
            s = (st["q_idx"][b, 0].double() @ key[b].t()).clamp_min(0)
            s = (st["w"][b, 0].double() @ s) * st["kscale"][b].double()
            sel = torch.topk(s, min(c["k"], c["N"])).indices
            rows = torch.cat([st["raw"][b], st["comp"][b, sel]]).double()
            o.append(_attn64(st["q"][b].double(), rows, st["sink"], torch.ones(1, rows.shape[0], dtype=torch.bool, device=DEV), SCALE, HD))
        return {"ids": None, "o": torch.stack(o)}
    if kind == "fp8_rows":
        o = []
        for b in range(c["B"]):
            i = st["idx"][b, 0]
            i = i[i >= 0].long()
            rows = workloads.dequant_e4m3(st["codes"][b, i], st["scales"][b, i]).double()
            o.append(_attn64(st["q"][b].double(), rows, st["sink"], torch.ones(1, rows.shape[0], dtype=torch.bool, device=DEV), SCALE, HD))
        return torch.stack(o)
    if kind == "prompt_attn":
        return _prompt64(st["q"][0], st["raw"][0], st["comp"][0], st["sink"], c["pos0"], 4, c["D"] ** -0.5, HD)[None]
    if kind == "prompt_index":
        Di = c["Di"]
        if c["keys"] == "fp4":
            k = st["keys"][0]
            k = torch.stack([k & 15, k >> 4], -1).reshape(k.shape[0], Di)
            mag = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=DEV)[(k & 7).long()]
            k = torch.where(k >= 8, -mag, mag) * torch.exp2(st["ks"][0].double() - 127).repeat_interleave(32, 1)
        else:
            k = st["keys"][0].view(torch.float8_e4m3fn).double() * st["ks"][0].double()[:, None]
        out = []
        for s0 in range(0, c["S"], 128):
            q = st["q"][0, s0:s0 + 128].double()
            d = (q.reshape(-1, Di) @ k.t()).clamp_min(0).reshape(q.shape[0], 64, -1)
            out.append((d * st["w"][0, s0:s0 + 128].double()[..., None]).sum(1))
        s = torch.cat(out)
        return {"scores": s.masked_fill(torch.arange(k.shape[0], device=DEV)[None] >= st["nvis"][0][:, None], float("-inf"))[None],
                "ids": None}
    if kind == "compress":
        x = st["x"][0].double()
        kv, sc = x @ st["wkv"].double().t(), x @ st["wgate"].double().t()
        cut = c["S"] - c["S"] % 4
        state = {"kv": kv[None, cut - 4:cut], "score": (sc[cut - 4:cut] + st["ape"].double())[None]}
        if c["S"] % 4:
            state["kv_rem"] = kv[None, cut:]
        # quantised rows have no one right value where the unquantised one lies on a rounding boundary
        rows = _pool64(kv[:cut], sc[:cut], st["ape"], st["norm"], False)[None] if c["form"] == "plain" else None
        return {"rows": rows, "state": state}
    w, ratio = st["w"], c["ratio"]
    if kind == "layer_prompt":
        x, S = st["xn"][0].double(), c["S"]
        cos_t, sin_t = _tables(S, YARN if ratio else PLAIN)
        q, kv = _qkv64(x, w, cos_t, sin_t)
        comp = None
        if ratio == 4 and S >= 4:
            cut = S - S % 4
            comp = _pool64((x @ w.wkv_c.double().t())[:cut], (x @ w.wgate_c.double().t())[:cut], w.ape, w.norm_c, True)
        o = _prompt64(q, kv, comp, w.sinks, 0, ratio, HD ** -0.5, HD)
        return {"y": _o_project64(o, cos_t, sin_t, w.wo_a, w.wo_b)[None], "window": None, "comp": None}
    pos = st["pos"].long()
    cos_t, sin_t = (t[pos] for t in _tables(c["max_pos"], YARN if ratio else PLAIN))
    q, kv = _qkv64(st["xn"].double(), w, cos_t, sin_t)
    ring, o = st["raw0"].double(), []
    for b in range(c["B"]):
        ring[b, pos[b] % WINDOW] = kv[b]
        rows = torch.cat([ring[b], st["comp0"][b, :(int(pos[b]) + 1) // 4].double()]) if ratio == 4 else ring[b]
        o.append(_attn64(q[b:b + 1], rows, w.sinks, torch.ones(1, rows.shape[0], dtype=torch.bool, device=DEV), HD ** -0.5, HD))
    return {"y": _o_project64(torch.cat(o), cos_t, sin_t, w.wo_a, w.wo_b), "window": None}
