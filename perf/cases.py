"""Performance cases: the calls a program that serves a Qwen3(-MoE) model makes.

Each case is one call (or one captured decode step) through the package's
public entry points on synthetic data of the real shapes.  Sizes are the
repository's own: the Qwen3-30B-A3B layer (hidden 2048, 128 experts, top-8,
intermediate 768, 32 query and 4 kv heads of 128), the Qwen3-235B-A22B MoE
block (hidden 4096, intermediate 1536) and the dense MLP of the same
configuration (intermediate 6144).

Kinds: ``moe`` (the sparse block), ``linear`` (a W4A16 projection), ``mlp``
(the dense SwiGLU MLP), ``decode_attn`` / ``chunk_attn`` (paged attention, one
or several query rows), ``causal_attn`` (the initial prefill's attention) and
``model`` (a step of a shortened model, logits out).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "nano-vllm-metal_amd"))

from nano_vllm_metal_amd import (Moe, Qwen3Model, QuantizedWeights, paged_attention,  # noqa: E402
                                 quantized_linear, qwen3_30b_a3b_config)
from nano_vllm_metal_amd.attention import causal_attention  # noqa: E402
from nano_vllm_metal_amd.qwen3 import DenseMLP  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
MOE_SHAPES = {"30b": (2048, 768, 128, 8), "235b": (4096, 1536, 128, 8)}
# in, out: stacked q/k/v, attention output, dense gate or up, dense down
PROJECTIONS = [(2048, 5120), (4096, 2048), (2048, 6144), (6144, 2048)]
VOCAB = 151936
PAGE = 16


def listed():
    return [
        # one request decoding: the smallest call, latency
        {"name": "moe_decode_1", "kind": "moe", "shape": "30b", "T": 1, "dtype": "bf16", "group": 64},
        # the benchmark's decode batch
        {"name": "moe_decode_32", "kind": "moe", "shape": "30b", "T": 32, "dtype": "bf16", "group": 64},
        # many requests decoding, or a short prompt, in fp16
        {"name": "moe_batch_150_f16", "kind": "moe", "shape": "30b", "T": 150, "dtype": "f16", "group": 64},
        # the benchmark's prefill
        {"name": "moe_prefill_4096", "kind": "moe", "shape": "30b", "T": 4096, "dtype": "bf16", "group": 64},
        # a medium prompt through the larger block
        {"name": "moe_235b_700", "kind": "moe", "shape": "235b", "T": 700, "dtype": "bf16", "group": 64},
        # the attention input projection of a decode step, an odd batch
        {"name": "linear_qkv_17", "kind": "linear", "M": 17, "n_in": 2048, "n_out": 5120, "dtype": "bf16", "group": 64},
        # the attention output projection of a ragged prompt, fp16, groups of 128
        {"name": "linear_o_1500_f16", "kind": "linear", "M": 1500, "n_in": 4096, "n_out": 2048, "dtype": "f16", "group": 128},
        # the dense MLP of a small decode batch
        {"name": "mlp_decode_5", "kind": "mlp", "M": 5, "dtype": "bf16", "group": 64},
        # decode attention of the benchmark's batch, contexts up to 1280
        {"name": "attn_decode_32", "kind": "decode_attn", "B": 32, "ctx": 1280, "kv": "bf16"},
        # the same over int8 pages, fewer requests with longer contexts
        {"name": "attn_decode_int8_8", "kind": "decode_attn", "B": 8, "ctx": 3000, "kv": "int8"},
        # the initial prefill's attention
        {"name": "attn_causal_5x1001", "kind": "causal_attn", "B": 5, "L": 1001, "dtype": "bf16"},
        # a decode step of the model, captured once and replayed as the server does
        {"name": "model_decode_8", "kind": "model", "layers": 4, "B": 8, "L": 1, "ctx": 500, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "linear", "linear", "mlp", "decode_attn", "decode_attn",
                       "chunk_attn", "causal_attn", "model"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "moe":
        shape = rng.choice(["30b", "30b", "235b"])
        return {"kind": kind, "shape": shape, "T": _log(rng, 1, 4096 if shape == "30b" else 1000),
                "dtype": dtype, "group": 64}
    if kind == "linear":
        n_in, n_out = rng.choice(PROJECTIONS + [(2048, VOCAB)])
        return {"kind": kind, "M": _log(rng, 1, 64 if n_out == VOCAB else 4096), "n_in": n_in,
                "n_out": n_out, "dtype": dtype, "group": rng.choice([64, 64, 128])}
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 1, 2048), "dtype": dtype, "group": rng.choice([64, 64, 128])}
    if kind == "decode_attn":
        return {"kind": kind, "B": _log(rng, 1, 64), "ctx": _log(rng, 32, 4096),
                "kv": rng.choice(["bf16", "bf16", "f16", "int8"])}
    if kind == "chunk_attn":
        L = _log(rng, 2, 256)
        return {"kind": kind, "B": rng.randint(1, 4), "L": L, "ctx": L + _log(rng, 16, 1024),
                "kv": rng.choice(["bf16", "f16"])}
    if kind == "causal_attn":
        return {"kind": kind, "B": rng.randint(1, 8), "L": _log(rng, 16, 1024), "dtype": dtype}
    if rng.random() < 0.5:
        return {"kind": kind, "layers": rng.randint(2, 4), "B": _log(rng, 1, 32), "L": 1,
                "ctx": _log(rng, 64, 1024), "dtype": "bf16"}
    return {"kind": kind, "layers": rng.randint(2, 4), "B": 1, "L": _log(rng, 16, 1024), "ctx": 0,
            "dtype": "bf16"}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _qw(g, dtype, group, *shape, std=0.02):
    """A 4-bit weight whose groups look like quantised N(0, std) values."""
    *lead, n_out, n_in = shape
    words = torch.randint(-2**31, 2**31 - 1, (*lead, n_out, n_in // 8), dtype=torch.int32,
                          device="cuda", generator=g)
    s = (torch.rand((*lead, n_out, n_in // group), device="cuda", generator=g) * 0.5 + 0.75) * (
        std * 6.0 / 15.0)
    return QuantizedWeights(s.to(dtype), (-7.5 * s).to(dtype), group, 4, words)


def _lens(case, g):
    """Context lengths spread over the upper half of the range."""
    B, ctx = case["B"], case["ctx"]
    lens = torch.randint(max(1, ctx // 2), ctx + 1, (B,), device="cuda", generator=g)
    lens[0] = ctx
    return lens.clamp_(min=case.get("L", 1)).to(torch.int32)


def _pages(case, g):
    B, width = case["B"], -(-case["ctx"] // PAGE)
    shape = (B * width, 4, PAGE, 128)
    bt = torch.randperm(B * width, device="cuda", generator=g).to(torch.int32).reshape(B, width)
    if case["kv"] == "int8":
        kp, vp = (torch.randint(-127, 128, shape, device="cuda", generator=g, dtype=torch.int8)
                  for _ in range(2))
        ks, vs = (torch.rand((*shape[:3], 1), device="cuda", generator=g) * 0.02 + 0.01
                  for _ in range(2))
        return bt, kp, vp, ks, vs
    dt = DTYPES[case["kv"]]
    kp, vp = (torch.randn(shape, device="cuda", generator=g).to(dt) for _ in range(2))
    return bt, kp, vp, None, None


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("decode_attn", "chunk_attn"):
        bt, kp, vp, ks, vs = _pages(case, g)
        q = torch.randn((case["B"], 32, case.get("L", 1), 128), device="cuda", generator=g)
        return {"kind": kind, "q": q, "kp": kp, "vp": vp, "ks": ks, "vs": vs, "bt": bt,
                "lens": _lens(case, g), "out": torch.bfloat16 if case["kv"] != "f16" else torch.float16}
    dt = DTYPES[case["dtype"]]
    if kind == "causal_attn":
        # values of the activation dtype held in float32, as the q/k norm leaves them
        q, k, v = (torch.randn((case["B"], case["L"], h, 128), device="cuda", generator=g).to(dt).float()
                   for h in (32, 4, 4))
        return {"kind": kind, "q": q, "k": k, "v": v, "dt": dt}
    if kind == "model":
        return _prepare_model(case, g, seed, dt)
    gs = case["group"]
    if kind == "moe":
        H, I, E, k = MOE_SHAPES[case["shape"]]
        block = Moe(_qw(g, dt, gs, E, H), _qw(g, dt, gs, E, I, H), _qw(g, dt, gs, E, I, H),
                    _qw(g, dt, gs, E, H, I), num_experts_per_tok=k, norm_topk_prob=True)
        x = torch.randn((case["T"], H), device="cuda", generator=g).to(dt)
    elif kind == "linear":
        block = _qw(g, dt, gs, case["n_out"], case["n_in"])
        x = torch.randn((case["M"], case["n_in"]), device="cuda", generator=g).to(dt)
    else:
        block = DenseMLP(_qw(g, dt, gs, 6144, 2048), _qw(g, dt, gs, 6144, 2048),
                         _qw(g, dt, gs, 2048, 6144))
        x = torch.randn((case["M"], 2048), device="cuda", generator=g).to(dt)
    return {"kind": kind, "block": block, "x": x}


def _prepare_model(case, g, seed, dt):
    cfg = qwen3_30b_a3b_config(case["layers"])
    cfg.max_position_embeddings = 4096
    model = Qwen3Model.random(cfg, device="cuda", dtype=dt, seed=seed)
    B, L, ctx = case["B"], case["L"], case["ctx"]
    cache = model.create_kv_cache(B * (-(-(ctx + L) // PAGE)), PAGE)
    for pool in cache.key_pages + cache.value_pages:
        pool.normal_(generator=g)
    for s in range(B):
        cache.add(s)
        cache.reserve(s, ctx)
        cache.advance([s], ctx)
    step = model.prepare(cache, list(range(B)), L)
    tokens = torch.randint(0, VOCAB, (B, L), device="cuda", generator=g)
    state = {"kind": "model", "model": model, "cache": cache, "step": step, "tokens": tokens,
             "graph": None}
    if L == 1:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.run(tokens, step, cache)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["logits"] = model.run(tokens, step, cache)
    return state


def run(state):
    kind = state["kind"]
    if kind in ("moe", "mlp"):
        return state["block"](state["x"])
    if kind == "linear":
        return quantized_linear(state["x"], state["block"])
    if kind == "causal_attn":
        return causal_attention(state["q"], state["k"], state["v"], 128 ** -0.5, state["dt"],
                                out_dtype=state["dt"])
    if kind == "model":
        if state["graph"] is not None:
            state["graph"].replay()
            return state["logits"]
        return state["model"].run(state["tokens"], state["step"], state["cache"])
    return paged_attention(state["q"], state["kp"], state["vp"], state["bt"], state["lens"], PAGE,
                           key_scales=state["ks"], value_scales=state["vs"], mask="causal",
                           out_dtype=state["out"])


# -------------------------------------------------------- what a pass needs


def _w_bytes(n_out, n_in, group):
    return n_out * n_in // 2 + 4 * n_out * (n_in // group)


def _moe_work(H, I, E, k, T, group):
    touched = E * (1.0 - (1.0 - k / E) ** T)
    by = touched * (2 * _w_bytes(I, H, group) + _w_bytes(H, I, group)) + _w_bytes(E, H, group)
    return by + 4 * T * H, 2.0 * T * k * 3 * H * I + 2.0 * T * H * E


def work(case):
    kind = case["kind"]
    if kind == "moe":
        H, I, E, k = MOE_SHAPES[case["shape"]]
        by, fl = _moe_work(H, I, E, k, case["T"], case["group"])
    elif kind == "linear":
        M, n, o = case["M"], case["n_in"], case["n_out"]
        by, fl = _w_bytes(o, n, case["group"]) + 2 * M * (n + o), 2.0 * M * n * o
    elif kind == "mlp":
        M, H, I = case["M"], 2048, 6144
        by = 2 * _w_bytes(I, H, case["group"]) + _w_bytes(H, I, case["group"]) + 4 * M * H
        fl = 6.0 * M * H * I
    elif kind == "causal_attn":
        B, L = case["B"], case["L"]
        by, fl = B * L * 128 * (40 * 4 + 32 * 2), 4.0 * B * 32 * (L * (L + 1) / 2) * 128
    elif kind in ("decode_attn", "chunk_attn"):
        B, L = case["B"], case.get("L", 1)
        ctx = case["ctx"] * 0.75
        row = 4 * 128 * (1 if case["kv"] == "int8" else 2) + (16 if case["kv"] == "int8" else 0)
        by = B * ctx * row * 2 + B * L * 32 * 128 * 6
        fl = 4.0 * B * L * 32 * max(ctx - L / 2, L / 2) * 128
    else:
        n, B, L, ctx = case["layers"], case["B"], case["L"], case["ctx"]
        T = B * L
        by, fl = _moe_work(2048, 768, 128, 8, T, 64)
        by += _w_bytes(5120, 2048, 64) + _w_bytes(2048, 4096, 64) + B * (ctx + L) * 2048
        fl += 2.0 * T * (5120 * 2048 + 2048 * 4096) + 4.0 * T * 32 * (ctx + (L + 1) / 2) * 128
        by = n * by + _w_bytes(VOCAB, 2048, 64) + 2 * B * VOCAB
        fl = n * fl + 2.0 * B * VOCAB * 2048
    return {"bytes": float(by), "flops": float(fl)}


def tolerance(case):
    kind = case["kind"]
    if kind == "model":
        # a near-tie in one layer's routing picks another expert: GEMV against
        # GEMM products in the blocks alone move the logits by up to 0.07
        return {"rel": 0.25}
    if kind in ("moe", "mlp"):
        return {"rel": 0.02 if case["dtype"] == "bf16" else 0.003}
    # one rounding of the output to the activation dtype
    return {"rel": 0.0012 if "f16" in (case.get("dtype"), case.get("kv")) else 0.007}


# ------------------------------------------------------------ 64-bit results


def _dequant(w, e=None):
    wq, s, b = (t if e is None else t[e] for t in (w.weight, w.scales, w.biases))
    shifts = torch.arange(0, 32, 4, device=wq.device, dtype=torch.int32)
    q = (wq[..., None] >> shifts) & 15
    q = q.reshape(wq.shape[0], s.shape[1], w.group_size).double()
    return (q * s.double()[..., None] + b.double()[..., None]).reshape(wq.shape[0], -1)


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_moe(block, x):
    act, k, xd = x.dtype, block.num_experts_per_tok, x.double()
    # the routing is defined on logits and probabilities of the activation
    # dtype, ties to the lower expert
    logits = (xd @ _dequant(block.w_router).T).to(act).double()
    probs = torch.softmax(logits, dim=-1).to(act)
    p, ids = torch.sort(probs.double(), dim=-1, descending=True, stable=True)
    p, ids = p[:, :k], ids[:, :k]
    score = (p / p.sum(-1, keepdim=True).to(act).double()).to(act).double()
    y = torch.zeros_like(xd)
    for e in range(block.w_router.weight.shape[0]):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            xe = xd[t]
            h = _silu(xe @ _dequant(block.w_gate, e).T) * (xe @ _dequant(block.w_up, e).T)
            y.index_add_(0, t, (h @ _dequant(block.w_down, e).T) * score[t, j][:, None])
    return y


def _attend(q, k, v, first):
    """q [Hq, L, D], k and v [Hkv, n, D]; row i sees keys up to first + i."""
    r = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(r, 0), v.repeat_interleave(r, 0)
    s = torch.matmul(q, k.transpose(1, 2)) * 128 ** -0.5
    j = torch.arange(k.shape[1], device=q.device)
    i = torch.arange(q.shape[1], device=q.device)
    s = s.masked_fill(j[None, :] > first + i[:, None], -math.inf)
    return torch.matmul(torch.softmax(s, dim=-1), v)


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return None  # a model's rounding travels through its layers
    st = prepare(case, seed)
    if kind == "moe":
        return _exact_moe(st["block"], st["x"])
    if kind == "linear":
        return st["x"].double() @ _dequant(st["block"]).T
    if kind == "mlp":
        m, x = st["block"], st["x"].double()
        h = _silu(x @ _dequant(m.w_gate).T) * (x @ _dequant(m.w_up).T)
        return h @ _dequant(m.w_down).T
    if kind == "causal_attn":
        return torch.stack([
            _attend(*(st[n][b].double().transpose(0, 1) for n in "qkv"), 0).transpose(0, 1)
            for b in range(case["B"])])
    out = []
    for b in range(case["B"]):
        n = int(st["lens"][b])
        pages = st["bt"][b, :-(-n // PAGE)].long()

        def rows(pool, scale):
            x = pool[pages].double()
            if scale is not None:
                x = x * scale[pages].double()
            return x.transpose(0, 1).reshape(4, -1, 128)[:, :n]

        q = st["q"][b].double()
        out.append(_attend(q, rows(st["kp"], st["ks"]), rows(st["vp"], st["vs"]), n - q.shape[1]))
    return torch.stack(out)
