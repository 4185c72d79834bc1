#!/usr/bin/env python
"""Benchmark of the Qwen3 sparse-MoE block on one MI355X.

Headline: MoE-layer tokens/s at the Qwen3-30B-A3B shape (hidden 2048, 128
experts, top-8 with renormalisation, moe_intermediate 768, MLX-affine int4
with group 64 and bf16 scale/bias), decode batch of 32 tokens.  One step is
one full MoE layer (route -> dispatch -> gate/up+SwiGLU -> down -> combine)
over one batch whose activations are already resident in HBM.  Eight distinct
layers of weights (2.7 GB packed) are cycled so the 256 MB MALL cannot hold
them.  The decode value is timed over HIP-graph replays of the layer calls;
per-kernel durations come from HIP events around each stage in an eager pass.

Also reported: decode batches 1/8/64, prefill of 4096 tokens with uniform and
Zipf(1.1) routing (MFMA roofline), the Qwen3-235B-A22B-shaped MoE layer
(decode 32, prefill 2048), the dense W4A16 projections of the same
model through quantized_matmul (q/k/o and the lm head, 1/32/4096 rows), paged
decode attention, the full 48-layer model through LLM.generate (32 x 1024-token
prompts, 256 greedy tokens: end-to-end decode tokens/s), and the CPU baseline (the C restatement of the reference algorithm in oracle/,
timed on a bounded sample).

Prints one JSON line on stdout; progress goes to stderr.  The line carries
the headline and each workload's main figures; ``--record FILE`` writes every
timing.
"""

from __future__ import annotations

import argparse
import ctypes
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT / "nano-vllm-metal_amd"))

HBM_PEAK_GBS = 8000.0            # MI355X HBM3E
MFMA_BF16_PEAK_TFLOPS = 2500.0   # dense bf16 MFMA
MI355X_XCDS, MI355X_SIMDS = 8, 1024  # 256 CUs of 4 SIMDs in 8 XCDs
METRIC = "MoE-layer tokens/s + HBM GB/s, 30B-A3B shape, decode B=32 / prefill 4K"
SHAPE = dict(H=2048, E=128, I=768, k=8, gs=64)
# Qwen3-235B-A22B's MoE layer (also reported: decode B=32, prefill 2048)
SHAPE_235B = dict(H=4096, E=128, I=1536, k=8, gs=64)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def bytes_per_expert(H, I, gs):
    """Packed int4 codes plus bf16 scale and bias, split (gate+up, down)."""
    gateup = 2 * (I * H // 2 + 2 * 2 * I * (H // gs))
    down = H * I // 2 + 2 * 2 * H * (I // gs)
    return gateup, down


def router_bytes(H, E, gs):
    return E * H // 2 + 2 * 2 * E * (H // gs)


def make_layers(n_layers, H, E, I, gs, dev, seed=1234, zipf_s=None, k=None):
    import torch
    from nano_vllm_metal_amd import Moe, QuantizedWeights, quantize

    gen = torch.Generator(device=dev)
    layers = []
    for li in range(n_layers):
        gen.manual_seed(seed + li)

        def q(shape, std=0.02, router_bias=None):
            w = (torch.randn(shape, generator=gen, device=dev) * std)
            if router_bias is not None:
                # one 64-wide activation group is held at 1.0 by the Zipf
                # inputs; these router columns then add log-popularity offsets
                w[:, :64] = (router_bias / 64.0)[:, None]
            wq, s, b = quantize(w.to(torch.bfloat16), gs, 4)
            return QuantizedWeights(s, b, gs, 4, wq)

        bias = None
        if zipf_s is not None:
            ranks = torch.arange(1, E + 1, device=dev, dtype=torch.float32)
            p = ranks ** (-zipf_s)
            bias = torch.log(p / p.sum())
        moe = Moe(q((E, H), router_bias=bias), q((E, I, H)), q((E, I, H)), q((E, H, I)),
                  num_experts_per_tok=k or SHAPE["k"], norm_topk_prob=True)
        layers.append(moe)
    torch.cuda.synchronize()
    return layers


def make_inputs(n, T, H, dev, seed=99, zipf=False):
    import torch

    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    xs = []
    for _ in range(n):
        x = torch.randn((T, H), generator=gen, device=dev)
        if zipf:
            x[:, :64] = 1.0
        xs.append(x.to(torch.bfloat16))
    return xs


class Stages:
    """Stage-level calls of the block (the kernels nvm_moe_forward runs)."""

    def __init__(self, moe, T, dev):
        import torch
        from nano_vllm_metal_amd import _lib

        self.lib = _lib.load()
        self.L = _lib
        self.moe = moe
        self.dev = dev
        E = moe.w_router.weight.shape[0]
        H = moe.w_router.weight.shape[1] * 8
        I = moe.w_gate.weight.shape[1]
        k = moe.num_experts_per_tok
        self.T, self.H, self.I, self.E, self.k = T, H, I, E, k
        N = T * k
        bf = torch.bfloat16
        self.ids = torch.empty((T, k), dtype=torch.int32, device=dev)
        self.scores = torch.empty((T, k), dtype=bf, device=dev)
        self.offsets = torch.empty(E + 1, dtype=torch.int32, device=dev)
        self.sorted = torch.empty(N, dtype=torch.int32, device=dev)
        self.h = torch.empty((N, I), dtype=bf, device=dev)
        self.down = torch.empty((N, H), dtype=bf, device=dev)
        self.y = torch.empty((T, H), dtype=bf, device=dev)
        size = ctypes.c_size_t()
        self.L.check(self.lib.nvm_route_dispatch_workspace_size(T, H, E, k, ctypes.byref(size)))
        self.rws = torch.empty(max(size.value, 1), dtype=torch.uint8, device=dev)

    def launch(self, stage, x):
        """One stage alone, on the routing its last run() left (route,
        gateup, down or combine)."""
        lib, L, m = self.lib, self.L, self.moe
        st = L.stream_of(self.dev)
        T, H, I, E, k = self.T, self.H, self.I, self.E, self.k
        gs = m.w_gate.group_size
        r, g, u, d = m.w_router, m.w_gate, m.w_up, m.w_down
        if stage == "route":
            L.check(lib.nvm_moe_route_dispatch(
                x.data_ptr(), T, H, r.weight.data_ptr(), r.scales.data_ptr(),
                r.biases.data_ptr(), E, gs, 4, k, 1, 1, None, self.ids.data_ptr(),
                self.scores.data_ptr(), self.offsets.data_ptr(), self.sorted.data_ptr(),
                self.rws.data_ptr(), self.rws.numel(), st))
        elif stage == "gateup":
            L.check(lib.nvm_moe_expert_gateup(
                x.data_ptr(), T, H, I, E, k, gs, 4, 1, g.weight.data_ptr(), g.scales.data_ptr(),
                g.biases.data_ptr(), u.weight.data_ptr(), u.scales.data_ptr(),
                u.biases.data_ptr(), self.offsets.data_ptr(), self.sorted.data_ptr(),
                self.h.data_ptr(), 0, st))
        elif stage == "down":
            L.check(lib.nvm_moe_expert_down(
                self.h.data_ptr(), T * k, H, I, E, gs, 4, 1, d.weight.data_ptr(),
                d.scales.data_ptr(), d.biases.data_ptr(), self.offsets.data_ptr(),
                self.sorted.data_ptr(), self.down.data_ptr(), 0, st))
        else:
            L.check(lib.nvm_moe_combine(self.down.data_ptr(), self.scores.data_ptr(), T, k, H, 1,
                                        self.y.data_ptr(), st))

    def run(self, x, events=None):
        lib, L, m = self.lib, self.L, self.moe
        st = L.stream_of(self.dev)
        T, H, I, E, k = self.T, self.H, self.I, self.E, self.k
        gs = m.w_gate.group_size
        r, g, u, d = m.w_router, m.w_gate, m.w_up, m.w_down
        ev = events or [None] * 5

        def rec(i):
            if ev[i] is not None:
                ev[i].record()

        rec(0)
        L.check(lib.nvm_moe_route_dispatch(
            x.data_ptr(), T, H, r.weight.data_ptr(), r.scales.data_ptr(), r.biases.data_ptr(), E,
            gs, 4, k, 1, 1, None, self.ids.data_ptr(), self.scores.data_ptr(),
            self.offsets.data_ptr(), self.sorted.data_ptr(), self.rws.data_ptr(), self.rws.numel(),
            st))
        rec(1)
        L.check(lib.nvm_moe_expert_gateup(
            x.data_ptr(), T, H, I, E, k, gs, 4, 1, g.weight.data_ptr(), g.scales.data_ptr(),
            g.biases.data_ptr(), u.weight.data_ptr(), u.scales.data_ptr(), u.biases.data_ptr(),
            self.offsets.data_ptr(), self.sorted.data_ptr(), self.h.data_ptr(), 0, st))
        rec(2)
        L.check(lib.nvm_moe_expert_down(
            self.h.data_ptr(), T * k, H, I, E, gs, 4, 1, d.weight.data_ptr(),
            d.scales.data_ptr(), d.biases.data_ptr(), self.offsets.data_ptr(),
            self.sorted.data_ptr(), self.down.data_ptr(), 0, st))
        rec(3)
        L.check(lib.nvm_moe_combine(self.down.data_ptr(), self.scores.data_ptr(), T, k, H, 1,
                                    self.y.data_ptr(), st))
        rec(4)
        return self.y


class ForwardStages:
    """The launches of nvm_moe_forward one stage at a time
    (nvm_moe_forward_stage: 0 routing, 1 gate/up, 2 down, 3 combine), on a
    workspace of their own: the kernels the layer runs, timed apart."""

    def __init__(self, moe, T, dev):
        import torch
        from nano_vllm_metal_amd import _lib

        self.lib, self.L, self.moe, self.dev = _lib.load(), _lib, moe, dev
        E = moe.w_router.weight.shape[0]
        H = moe.w_router.weight.shape[1] * 8
        I = moe.w_gate.weight.shape[1]
        k = moe.num_experts_per_tok
        self.T, self.H, self.I, self.E, self.k = T, H, I, E, k
        size = ctypes.c_size_t()
        self.L.check(self.lib.nvm_moe_workspace_size(T, H, I, E, k, ctypes.byref(size)))
        self.ws = torch.empty(size.value, dtype=torch.uint8, device=dev)
        self.y = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
        self.ops = moe._operands()

    def launch(self, stage, x):
        L, m = self.L, self.moe
        flat = [t.data_ptr() for trio in self.ops for t in trio]
        L.check(self.lib.nvm_moe_forward_stage(
            stage, x.data_ptr(), self.T, self.H, self.I, self.E, self.k,
            int(bool(m.norm_topk_prob)), m.w_gate.group_size, m.w_gate.bits,
            L.dtype_code(x.dtype), *flat, self.y.data_ptr(), None, None,
            L.REGIME_AUTO, self.ws.data_ptr(), self.ws.numel(), L.stream_of(self.dev)))

    def run(self, x, upto=4, seq=None):
        """Stages 0 .. upto-1, or the stages of `seq` in order."""
        for s in (range(upto) if seq is None else seq):
            self.launch(s, x)
        return self.y


def forward_plan(moe, T, regime=0):
    """1 when nvm_moe_forward runs both products of this batch as one launch
    (stage 4 of nvm_moe_forward_stage), else 0."""
    from nano_vllm_metal_amd import _lib

    lib = _lib.load()
    E = moe.w_router.weight.shape[0]
    H = moe.w_router.weight.shape[1] * 8
    I = moe.w_gate.weight.shape[1]
    out = ctypes.c_int(0)
    _lib.check(lib.nvm_moe_forward_plan(T, H, I, E, moe.num_experts_per_tok,
                                        moe.w_gate.group_size, regime, ctypes.byref(out)))
    return out.value


def forward_stage_us(layers, xs, stage, n=64, before=None):
    """Duration (us) of one stage of the layer's own launch sequence: a HIP
    graph of `n` back-to-back launches of that stage (weight sets cycled, each
    set's earlier stages run beforehand), timed with HIP events on the stream
    the graph's kernels run on; the mean per launch, the figure that
    `rocprofv3 --kernel-trace` reports as the kernel's average."""
    import torch

    T = xs[0].shape[0]
    fs = [ForwardStages(m, T, layers[0].w_gate.weight.device) for m in layers]
    # (each set's stages before this one: a later stage may overwrite what
    # this one reads, as the down product overwrites the fp16 copy of x)
    for i, f in enumerate(fs):
        f.run(xs[i % len(xs)], upto=stage, seq=before)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for i, f in enumerate(fs):
            f.launch(stage, xs[i % len(xs)])
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(n):
            fs[i % len(fs)].launch(stage, xs[i % len(fs) % len(xs)])
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    g.replay()
    e1.record()
    torch.cuda.synchronize()
    del fs
    return e0.elapsed_time(e1) * 1e3 / n


def in_layer_stage_us(layers, xs, stage, n=64, seq=None):
    """Duration (us) of one stage where the layer runs it, after its own
    earlier stages (their outputs just written, as in the layer): a HIP graph
    of `n` runs of stages 0..stage minus a graph of `n` runs of stages
    0..stage-1 (with `seq`: of the stages seq[:stage + 1] minus seq[:stage]),
    over the same weight sets, timed with HIP events on the stream the
    graphs' kernels run on."""
    import torch

    T = xs[0].shape[0]
    fs = [ForwardStages(m, T, layers[0].w_gate.weight.device) for m in layers]

    def graph_us(upto):
        sq = None if seq is None else seq[:upto]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for i, f in enumerate(fs):
                f.run(xs[i % len(xs)], upto=upto, seq=sq)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for i in range(n):
                fs[i % len(fs)].run(xs[i % len(fs) % len(xs)], upto=upto, seq=sq)
        g.replay()
        torch.cuda.synchronize()
        best = None
        for _ in range(3):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            g.replay()
            e1.record()
            torch.cuda.synchronize()
            t = e0.elapsed_time(e1) * 1e3
            best = t if best is None else min(best, t)
        del g
        return best

    with_stage = graph_us(stage + 1)
    before = graph_us(stage)
    del fs
    return (with_stage - before) / n


# route = routing and dispatch (nvm_moe_route_dispatch)
STAGE_NAMES = ["route", "gateup", "down", "combine"]


def eager_stage_pass(layers, xs, steps, warmup, dev):
    """Per-stage HIP-event durations (us) and touched-expert counts per step."""
    import torch

    T = xs[0].shape[0]
    stages = [Stages(m, T, dev) for m in layers]
    for i in range(warmup):
        stages[i % len(layers)].run(xs[i % len(xs)])
    torch.cuda.synchronize()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(5)] for _ in range(steps)]
    touched = []
    ids_snap = []
    for i in range(steps):
        s = stages[i % len(layers)]
        s.run(xs[i % len(xs)], evs[i])
        ids_snap.append(s.ids.clone())
    torch.cuda.synchronize()
    dur = {n: 0.0 for n in STAGE_NAMES}
    total = 0.0
    for i in range(steps):
        for j, n in enumerate(STAGE_NAMES):
            dur[n] += evs[i][j].elapsed_time(evs[i][j + 1]) * 1e3
        total += evs[i][0].elapsed_time(evs[i][4]) * 1e3
    for i in range(steps):
        touched.append(int(torch.unique(ids_snap[i]).numel()))
    return {n: v / steps for n, v in dur.items()}, total / steps, touched, ids_snap


def timed_steps(layers, xs, steps, warmup, dev):
    """Exactly `steps` layer calls, timed as one region: `warmup` untimed calls,
    then one HIP graph holding the `steps` calls (weight sets and inputs
    cycled, as consecutive layers of a model run) replayed once between two
    synchronisations.  Returns the mean layer time (us)."""
    import torch

    L = len(layers)
    for i in range(max(warmup, 1)):
        layers[i % L](xs[i % len(xs)])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(steps):
            layers[i % L](xs[i % len(xs)])
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    g.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e3 / steps


def median_steps(layers, xs, n, warmup=10):
    """Median and mean layer time (us) over `n` individually timed layer calls
    (one HIP graph per weight set, replayed in turn with an event between
    consecutive replays), after `warmup` untimed replays."""
    import statistics

    import torch

    L = len(layers)
    graphs = []
    for i in range(L):
        layers[i](xs[i % len(xs)])
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            layers[i](xs[i % len(xs)])
        graphs.append(g)
    for i in range(warmup):
        graphs[i % L].replay()
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(n + 1)]
    ev[0].record()
    for i in range(n):
        graphs[i % L].replay()
        ev[i + 1].record()
    torch.cuda.synchronize()
    d = [ev[i].elapsed_time(ev[i + 1]) * 1e3 for i in range(n)]
    return statistics.median(d), sum(d) / n


def stage_kernel_us(stages, xs, stage, n=64):
    """Duration (us) of one stage's launch: a HIP graph of `n` back-to-back
    launches of that stage alone (weight sets cycled, routing of each set
    computed beforehand), timed with events; the mean per launch.  This is
    the kernel's own time plus the short gap between graph kernels, the figure
    that `rocprofv3 --kernel-trace` reports as the kernel's average."""
    import torch

    for i, s in enumerate(stages):
        s.run(xs[i % len(xs)])
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for i, s in enumerate(stages):
            s.launch(stage, xs[i % len(xs)])
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(n):
            stages[i % len(stages)].launch(stage, xs[i % len(stages) % len(xs)])
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    g.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e3 / n


def eager_fused_pass(layers, xs, steps, warmup, dev):
    import torch

    L = len(layers)
    for i in range(warmup):
        layers[i % L](xs[i % len(xs)])
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for i in range(steps):
        layers[i % L](xs[i % len(xs)])
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e3 / steps


def decode_bench(layers, T, steps, warmup, dev, use_graph=True, shape=None, n_median=100):
    """Decode layer at T tokens.  `layer_us` is the mean of exactly `steps`
    layer calls in one timed region (a HIP graph of the calls); the median
    (and mean) over max(n_median, steps) individually timed layer calls is
    reported beside it, as is each stage's kernel time from back-to-back
    launches of that stage (the roofline's duration)."""
    H, E, I, k, gs = ((shape or SHAPE)[n] for n in ("H", "E", "I", "k", "gs"))
    xs = make_inputs(8, T, H, dev)
    stage_us, eager_layer_us, touched, _ = eager_stage_pass(layers, xs, min(steps, 64),
                                                            warmup, dev)
    fused_us = eager_fused_pass(layers, xs, min(steps, 64), warmup, dev)
    if use_graph:
        layer_us = timed_steps(layers, xs, steps, warmup, dev)
        med_us, mean_us = median_steps(layers, xs, max(n_median, steps))
    else:
        layer_us, med_us, mean_us = fused_us, None, None
    stages = [Stages(m, T, dev) for m in layers]
    graph_kernel_us = {n: stage_kernel_us(stages, xs, n) for n in ("gateup", "down")}
    del stages
    fwd_kernel_us = {n: forward_stage_us(layers, xs, i) for i, n in enumerate(STAGE_NAMES)}
    in_layer_us = {n: in_layer_stage_us(layers, xs, i) for i, n in ((1, "gateup"), (2, "down"))}
    # both products as the layer launches them (stage 4: one launch where the
    # forward fuses them)
    fused_products = forward_plan(layers[0], T)
    in_layer_us["products"] = in_layer_stage_us(layers, xs, 1, seq=[0, 4])
    fwd_kernel_us["products"] = forward_stage_us(layers, xs, 4, before=[0])
    gu_b, dn_b = bytes_per_expert(H, I, gs)
    avg_touched = sum(touched) / len(touched)
    layer_bytes = avg_touched * (gu_b + dn_b) + router_bytes(H, E, gs) + 2 * T * H * 2
    gateup_bytes = avg_touched * gu_b + T * H * 2
    products_bytes = avg_touched * (gu_b + dn_b) + T * H * 2
    return {
        "tokens": T,
        "tokens_per_s": T / (layer_us * 1e-6),
        "layer_us": layer_us,
        "timing": (f"one HIP-graph replay of exactly {steps} layer calls" if use_graph
                   else "eager"),
        "layer_us_median": med_us,
        "layer_us_mean_individual": mean_us,
        "median_samples": max(n_median, steps) if use_graph else 0,
        "tokens_per_s_median": T / (med_us * 1e-6) if med_us else None,
        "eager_layer_us": fused_us,
        "eager_staged_layer_us": eager_layer_us,
        "kernel_us": stage_us,
        "kernel_us_back_to_back": graph_kernel_us,
        "forward_kernel_us": fwd_kernel_us,
        "forward_kernel_us_note": "the layer's own launches one stage at a time "
                                  "(nvm_moe_forward_stage: route = partial logits, gateup = "
                                  "gate/up with the routing finalised in its prologue), each a "
                                  "HIP graph of 64 back-to-back launches timed with events",
        "in_layer_kernel_us": in_layer_us,
        "in_layer_kernel_us_note": "the stage where the layer runs it, after its own earlier "
                                   "stages: a HIP graph of 64 runs of stages 0..s minus one of "
                                   "stages 0..s-1 (nvm_moe_forward_stage), timed with events; "
                                   "products = both products as the layer launches them "
                                   "(stages 0, 4 minus stage 0)",
        "fused_products": bool(fused_products),
        "touched_experts_avg": avg_touched,
        "layer_algorithmic_bytes": layer_bytes,
        "hbm_gbs": layer_bytes / (layer_us * 1e-6) / 1e9,
        "gateup_algorithmic_bytes": gateup_bytes,
        "products_algorithmic_bytes": products_bytes,
        "in_layer_products_gbs": products_bytes / (in_layer_us["products"] * 1e-6) / 1e9,
        "forward_products_gbs": products_bytes / (fwd_kernel_us["products"] * 1e-6) / 1e9,
        "gateup_gbs": gateup_bytes / (graph_kernel_us["gateup"] * 1e-6) / 1e9,
        "forward_gateup_gbs": gateup_bytes / (fwd_kernel_us["gateup"] * 1e-6) / 1e9,
        "in_layer_gateup_gbs": gateup_bytes / (in_layer_us["gateup"] * 1e-6) / 1e9,
        "down_gbs": avg_touched * dn_b / (graph_kernel_us["down"] * 1e-6) / 1e9,
    }


def prefill_bench(layers, T, steps, warmup, dev, zipf, shape=None):
    import torch

    H, E, I, k, gs = ((shape or SHAPE)[n] for n in ("H", "E", "I", "k", "gs"))
    xs = make_inputs(2, T, H, dev, seed=7 if zipf else 5, zipf=zipf)
    # the layer: Moe's forward (nvm_moe_forward), which hands the prefill
    # GEMMs fp16 activations converted once; the per-stage times come from the
    # stage entry points, whose GEMMs convert their staged rows themselves
    stage_us, stage_layer_us, touched, ids = eager_stage_pass(layers, xs, steps, warmup, dev)
    layer_us = eager_fused_pass(layers, xs, steps, warmup, dev)
    fwd_us = {n: forward_stage_us(layers, xs, i, n=16) for i, n in enumerate(STAGE_NAMES)}
    in_layer_us = {n: in_layer_stage_us(layers, xs, i, n=16) for i, n in ((1, "gateup"), (2, "down"))}
    N = T * k
    gateup_flops = 2.0 * N * H * 2 * I
    down_flops = 2.0 * N * I * H
    layer_flops = gateup_flops + down_flops + 2.0 * T * H * E
    counts = torch.bincount(ids[0].reshape(-1).long(), minlength=E).float()
    return {
        "tokens": T,
        "routing": "zipf(1.1)" if zipf else "uniform",
        "tokens_per_s": T / (layer_us * 1e-6),
        "layer_us": layer_us,
        "timing": "eager: HIP events around the layer calls (nvm_moe_forward)",
        "stage_layer_us": stage_layer_us,
        "kernel_us": stage_us,
        "kernel_us_note": "stage entry points (route+dispatch, gate/up, down, combine), "
                          "each timed with HIP events",
        "forward_kernel_us": fwd_us,
        "forward_kernel_us_note": "the layer's own launches one stage at a time "
                                  "(nvm_moe_forward_stage; the GEMMs on the fp16 copies of x "
                                  "and h), each a HIP graph of 16 back-to-back launches timed "
                                  "with events",
        "in_layer_kernel_us": in_layer_us,
        "in_layer_kernel_us_note": "the stage where the layer runs it, after its own earlier "
                                   "stages: a HIP graph of 16 runs of stages 0..s minus one of "
                                   "stages 0..s-1 (nvm_moe_forward_stage), timed with events",
        "in_layer_gateup_tflops": gateup_flops / (in_layer_us["gateup"] * 1e-6) / 1e12,
        "in_layer_down_tflops": down_flops / (in_layer_us["down"] * 1e-6) / 1e12,
        "forward_gateup_tflops": gateup_flops / (fwd_us["gateup"] * 1e-6) / 1e12,
        "forward_down_tflops": down_flops / (fwd_us["down"] * 1e-6) / 1e12,
        "layer_tflops": layer_flops / (layer_us * 1e-6) / 1e12,
        "gateup_tflops": gateup_flops / (stage_us["gateup"] * 1e-6) / 1e12,
        "down_tflops": down_flops / (stage_us["down"] * 1e-6) / 1e12,
        "layer_mfma_frac": layer_flops / (layer_us * 1e-6) / 1e12 / MFMA_BF16_PEAK_TFLOPS,
        "expert_load_max_over_mean": float(counts.max() / counts.mean()),
        "experts_touched": int((counts > 0).sum()),
    }


def shape_235b_bench(dev, steps):
    """The Qwen3-235B-A22B MoE layer (hidden 4096, 128 experts, top-8,
    intermediate 1536, int4 g64): decode batch 32 and prefill 2048 tokens,
    over 3 distinct layers of weights (1.2 GB each)."""
    import torch

    sh = SHAPE_235B
    layers = make_layers(3, sh["H"], sh["E"], sh["I"], sh["gs"], dev, seed=2350, k=sh["k"])
    d = decode_bench(layers, 32, max(steps // 2, 16), 10, dev, True, shape=sh)
    p = prefill_bench(layers, 2048, max(steps // 20, 8), 3, dev, False, shape=sh)
    log(f"[bench] 235B decode B=32: {d['layer_us']:.1f} us/layer, {d['hbm_gbs']:.0f} GB/s; "
        f"prefill 2048: {p['layer_us']:.1f} us/layer, {p['layer_tflops']:.0f} TFLOP/s")
    del layers
    torch.cuda.empty_cache()
    return {"decode_32": d, "prefill_2048": p}


# Dense W4A16 projections of the same model (quantized_linear): name, in, out.
DENSE_SHAPES = (("q_proj", 2048, 4096), ("k_proj", 2048, 512), ("o_proj", 4096, 2048),
                ("lm_head", 2048, 151936))


def dense_bench(dev, rows=(1, 32, 4096)):
    """Kernel time of quantized_matmul per call (HIP-graph replay, _graph_us)
    for the 30B-A3B dense projection shapes."""
    import torch
    from nano_vllm_metal_amd import quantized_matmul

    gs = 64
    out = {}
    for name, N, K in DENSE_SHAPES:
        g = torch.Generator(device=dev).manual_seed(N + K)
        w = torch.randint(-2**31, 2**31 - 1, (K, N // 8), dtype=torch.int32, device=dev,
                          generator=g)
        sc = (torch.rand(K, N // gs, device=dev, generator=g) * 0.01).to(torch.bfloat16)
        bi = (torch.rand(K, N // gs, device=dev, generator=g) * -0.04).to(torch.bfloat16)
        wbytes = K * N // 2 + 2 * 2 * K * (N // gs)
        res = {"in": N, "out": K, "weight_bytes": wbytes}
        for M in rows:
            if name == "lm_head" and M > 32:
                continue
            a = torch.randn(M, N, device=dev, generator=g).to(torch.bfloat16)
            us = _graph_us(lambda: quantized_matmul(sc, bi, gs, 4, a, w, True))
            res[str(M)] = {"us": us, "weight_gbs": wbytes / us / 1e3,
                           "tflops": 2.0 * M * N * K / us / 1e6}
        out[name] = res
        del w, sc, bi
    return out


# Paged decode attention of the same model: 32 query heads over 4 kv heads of
# dim 128, bf16 pages of 16 slots; (requests, context positions).
ATTN_SHAPE = dict(Hq=32, Hkv=4, D=128, page=16)
ATTN_CASES = ((32, 1280), (1, 4096), (64, 2048))


def _graph_us(fn, reps=20, n=10):
    """Kernel time per call: HIP-graph replay of `reps` calls, `n` replays."""
    import torch

    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        for _ in range(3):
            fn()
    torch.cuda.current_stream().wait_stream(st)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(reps):
            fn()
    graph.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(n):
        graph.replay()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e3 / (n * reps)


def attention_bench(dev):
    """Paged decode attention: kernel time per call and K/V bytes read per
    second (each request's context read once per kv head)."""
    import torch
    from nano_vllm_metal_amd import paged_attention

    Hq, Hkv, D, ps = (ATTN_SHAPE[n] for n in ("Hq", "Hkv", "D", "page"))
    out = {}
    for B, ctx in ATTN_CASES:
        g = torch.Generator(device=dev).manual_seed(B * 7 + ctx)
        mp = (ctx + ps - 1) // ps
        P = B * mp
        q = torch.randn(B, Hq, 1, D, device=dev, generator=g)
        kp = torch.randn(P, Hkv, ps, D, device=dev, generator=g).to(torch.bfloat16)
        vp = torch.randn(P, Hkv, ps, D, device=dev, generator=g).to(torch.bfloat16)
        bt = torch.randperm(P, device=dev, generator=g).to(torch.int32).reshape(B, mp)
        lens = torch.full((B,), ctx, dtype=torch.int32, device=dev)
        us = _graph_us(lambda: paged_attention(q, kp, vp, bt, lens, ps))
        kv_bytes = 2 * B * ctx * Hkv * D * 2
        out[f"B{B}_ctx{ctx}"] = {"us": us, "kv_bytes": kv_bytes, "gbs": kv_bytes / us / 1e3,
                                 "frac_hbm": kv_bytes / us / 1e3 / HBM_PEAK_GBS}
        del q, kp, vp, bt
    # the initial-prefill causal attention at the e2e shape: 8 requests x 1024
    # tokens (flops of the visible half: 2 products of 2 L^2/2 D per head)
    from nano_vllm_metal_amd.attention import causal_attention

    B, L = 8, 1024
    g = torch.Generator(device=dev).manual_seed(11)
    q = torch.randn(B, L, Hq, D, device=dev, generator=g).to(torch.bfloat16).float()
    k = torch.randn(B, L, Hkv, D, device=dev, generator=g).to(torch.bfloat16).float()
    v = torch.randn(B, L, Hkv, D, device=dev, generator=g).to(torch.bfloat16).float()
    us = _graph_us(lambda: causal_attention(q, k, v, D ** -0.5, torch.bfloat16,
                                            out_dtype=torch.bfloat16))
    flops = 2.0 * B * Hq * L * (L + 1) * D * 2 / 2
    out[f"prefill_causal_B{B}_L{L}"] = {"us": us, "tflops": flops / us / 1e6,
                                        "frac_mfma": flops / us / 1e6 / MFMA_BF16_PEAK_TFLOPS}
    del q, k, v
    # chunked prefill / prefill after a prefix on the paged cache: 4 requests
    # of 256 new rows over 1024 cached positions (causal; the matrix-core
    # multi-query kernel); flops of the visible scores and values
    B, L, ctx = 4, 256, 1280
    g = torch.Generator(device=dev).manual_seed(13)
    mp = (ctx + ps - 1) // ps
    P = B * mp
    q = torch.randn(B, Hq, L, D, device=dev, generator=g)
    kp = torch.randn(P, Hkv, ps, D, device=dev, generator=g).to(torch.bfloat16)
    vp = torch.randn(P, Hkv, ps, D, device=dev, generator=g).to(torch.bfloat16)
    bt = torch.randperm(P, device=dev, generator=g).to(torch.int32).reshape(B, mp)
    lens = torch.full((B,), ctx, dtype=torch.int32, device=dev)
    us = _graph_us(lambda: paged_attention(q, kp, vp, bt, lens, ps, mask="causal"))
    vis = sum(ctx - L + i + 1 for i in range(L))  # visible positions per (request, head)
    flops = 2.0 * 2 * B * Hq * vis * D
    out[f"prefill_chunk_B{B}_L{L}_ctx{ctx}"] = {
        "us": us, "tflops": flops / us / 1e6, "frac_mfma": flops / us / 1e6 / MFMA_BF16_PEAK_TFLOPS,
        "note": "query scores on three act-dtype parts of the float32 query (3 MFMAs a product)"}
    del q, kp, vp, bt
    return out


def e2e_bench(dev, n_seqs=32, prompt_len=1024, gen=256, layers=48):
    """Full Qwen3-30B-A3B-shaped model (random int4 weights) through
    LLM.generate with the paged KV cache: n_seqs concurrent requests of
    prompt_len random tokens, gen greedy tokens each (no early stop)."""
    import numpy as np
    import torch
    from nano_vllm_metal_amd import LLM, Qwen3Model, SamplingParams, qwen3_30b_a3b_config

    cfg = qwen3_30b_a3b_config(layers)
    log(f"[bench] e2e: building a {layers}-layer 30B-A3B-shaped model (random int4 weights)")
    model = Qwen3Model.random(cfg, device=dev, seed=7)
    llm = LLM(model, max_num_seqs=n_seqs, max_model_len=prompt_len + gen + 16, page_size=16,
              prefill_step=8 * prompt_len)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, cfg.vocab_size, prompt_len).tolist() for _ in range(n_seqs)]
    llm.generate([p[:32] for p in prompts[:4]], SamplingParams(max_tokens=4))  # warm-up
    from nano_vllm_metal_amd.llm import GenerateStats

    llm.stats = GenerateStats()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    outs = llm.generate(prompts, SamplingParams(max_tokens=gen, ignore_eos=True))
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    st = llm.stats
    assert all(len(o.token_ids) == gen for o in outs)
    res = {"layers": layers, "seqs": n_seqs, "prompt_len": prompt_len, "gen_tokens": gen,
           "decode_tokens_per_s": st.decode_tokens / st.decode_s,
           "decode_step_ms": st.decode_s / st.decode_steps * 1e3,
           "prefill_tokens_per_s": st.prefill_tokens / st.prefill_s,
           "wall_s": wall, "generated_tokens_per_s": n_seqs * gen / wall}
    # the run checked at its own size (as tests/test_gpu_e2e_config5.py does):
    # every page free afterwards, and requests re-run alone reproducing the
    # batch's greedy tokens up to a near-tie (recomputed logits, bf16 ulps of
    # the row's largest logit)
    pages_free = llm.cache.free_pages == llm.cache.num_pages
    del llm
    solo = LLM(model, max_num_seqs=1, max_model_len=prompt_len + gen + 16, page_size=16,
               prefill_step=8 * prompt_len)
    checks = []
    for i in (0, n_seqs - 1):
        alone = solo.generate([prompts[i]], SamplingParams(max_tokens=gen, ignore_eos=True))
        alone = alone[0].token_ids
        batch = outs[i].token_ids
        d = next((j for j in range(gen) if batch[j] != alone[j]), gen)
        j = min(d, gen - 1)
        cache = model.create_kv_cache(-(-(prompt_len + gen) // 16), page_size=16)
        cache.add(0)
        lg = model.forward(torch.tensor([prompts[i] + alone[:j]], device=dev), cache, [0])[0]
        lg = lg.float()
        ulp = 2.0 ** (np.floor(np.log2(float(lg.abs().max().clamp_min(2.0 ** -100)))) - 7)
        checks.append({"request": i, "same_tokens": d,
                       "batch_token_gap_ulps": float(lg.max() - lg[batch[j]]) / ulp,
                       "logits_finite": bool(torch.isfinite(lg).all())})
        del cache
    res["check"] = {"all_pages_free": pages_free, "requests_rerun_alone": checks,
                    "bar": "tokens equal, or the batch's token within 4 ulps of the lone "
                           "run's maximum logit where they part"}
    del solo, model
    torch.cuda.empty_cache()
    return res


def host_cpus():
    """The host's CPU model, its logical/physical cores and the cores this
    process may use (affinity and cgroup quota)."""
    info = {"nproc": os.cpu_count(), "affinity_cpus": len(os.sched_getaffinity(0))}
    model, cores = None, set()
    try:
        phys = core = None
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            key, _, val = line.partition(":")
            key, val = key.strip(), val.strip()
            if key == "model name" and model is None:
                model = val
            elif key == "physical id":
                phys = val
            elif key == "core id":
                core = val
            elif not line.strip() and phys is not None:
                cores.add((phys, core))
                phys = core = None
    except OSError:
        pass
    info["cpu_model"] = model
    info["physical_cores"] = len(cores) or None
    quota = None
    try:
        q, per = Path("/sys/fs/cgroup/cpu.max").read_text().split()[:2]
        if q != "max":
            quota = int(q) / int(per)
    except (OSError, ValueError):
        pass
    info["cgroup_cpu_quota"] = quota
    usable = info["affinity_cpus"]
    if quota:
        usable = min(usable, max(1, int(quota)))
    if info["physical_cores"]:
        usable = min(usable, info["physical_cores"])
    info["usable_cores"] = usable
    return info


def cpu_baseline(layer, T, seconds, dev, runs=10, warmup=2):
    """The C restatement of the reference path (oracle/moe_ref.c) on the host
    cores: one decode layer of T tokens, median of `runs` timed runs after
    `warmup`, at 1 thread and at all usable cores (affinity and cgroup
    quota, at most one thread per physical core)."""
    import statistics

    import numpy as np
    import torch

    sys.path.insert(0, str(ROOT))
    from oracle import moe_ref as R

    R.build()
    host = host_cpus()
    ops = []
    for w in (layer.w_router, layer.w_gate, layer.w_up, layer.w_down):
        ops += [w.weight.cpu().numpy().view(np.uint32),
                w.scales.view(torch.int16).cpu().numpy().view(np.uint16),
                w.biases.view(torch.int16).cpu().numpy().view(np.uint16)]
    cl = R.Layer.from_arrays(ops, "bfloat16")
    xs = make_inputs(4, T, SHAPE["H"], dev, seed=31)
    xb = [x.view(torch.int16).cpu().numpy().view(np.uint16) for x in xs]
    # routing agreement of the CPU restatement and the GPU path on the sample
    _, gids, _ = layer.forward(xs[0], return_routing=True)
    torch.cuda.synchronize()

    def timed(nthreads):
        R.threads(nthreads)
        cids = None
        for i in range(warmup):
            _, ids, _ = R.forward(xb[i % len(xb)], cl, SHAPE["k"], True, SHAPE["gs"])
            cids = ids if cids is None else cids
        d = []
        t_start = time.perf_counter()
        for i in range(runs):
            t0 = time.perf_counter()
            R.forward(xb[i % len(xb)], cl, SHAPE["k"], True, SHAPE["gs"])
            d.append(time.perf_counter() - t0)
            if len(d) >= 3 and time.perf_counter() - t_start > seconds:
                break  # bounded sample: at least three runs
        med = statistics.median(d)
        return {"tokens_per_s": T / med, "median_s": med, "runs": len(d),
                "threads": R.threads(0)}, cids

    one, cids = timed(1)
    allc, _ = timed(host["usable_cores"])
    return {
        "value": allc["tokens_per_s"],
        "unit": "tokens/s",
        "cores": allc["threads"],
        "kind": "port",
        "sample": f"decode layers of {T} tokens at the 30B-A3B shape (one weight set, 4 inputs "
                  f"cycled), median of {allc['runs']} runs after {warmup} warm-ups at "
                  f"{allc['threads']} threads; OpenMP over routed pairs",
        "single_thread": one,
        "all_cores": allc,
        "host": host,
        "routing_matches_gpu": bool(np.array_equal(cids, gids.cpu().numpy())),
    }


TRAFFIC_JSON = ROOT / "profiles" / "traffic.json"
COPY_PROBE_BYTES = 256 << 20

# rocprofv3 kernel names (regular expressions) -> the product kernels
# reported in the JSON line.  decode_gateup_fused is the gate/up product that
# finalises the routing in its prologue (inside nvm_moe_forward);
# decode_gateup is the product alone (nvm_moe_expert_gateup).
KERNEL_KEYS = (
    # both decode products in one launch (expert-major blocks, each over one
    # half of the down reduction): the layer's products launch from two
    # routed rows per expert on average
    ("decode_products", r"gemv3_kernel<1, true, \d+, true, true, false, [1-9]"),
    ("decode_gateup_fused", r"gemv3_kernel<1, true, \d+, true,"),
    ("decode_gateup", r"gemv3_kernel<1, true, \d+, false,|gemv_kernel<1, true"),
    # the down product with the combine in its epilogue (decode batches of at
    # most 16 pairs)
    ("decode_down_combine", r"gemv3_kernel<1, false, \d+, false, false, true>"),
    ("decode_down", r"gemv3_kernel<1, false|gemv_kernel<1, false"),
    # prefill GEMMs of the forward (activations converted to fp16 once, by
    # act_to_f16) and of the stage entry points (converting their own rows)
    ("prefill_gateup", r"gemm_dma_kernel<true>|gemm_kernel<1, true, true>"),
    ("prefill_down", r"gemm_dma_kernel<false>|gemm_kernel<1, false, true>"),
    ("prefill_gateup_stage", r"gemm_kernel<1, true, false>"),
    ("prefill_down_stage", r"gemm_kernel<1, false, false>"),
    ("prefill_act_f16", r"act_to_f16_kernel"),
    ("route_partial", r"route_mfma_kernel<1|route_i8_kernel<1"),
    ("route_i8_fin", r"route_i8_fin_kernel<1"),
    ("dispatch_hist", r"dispatch_hist_kernel"),
    ("route_finalize_dispatch", r"route_finalize_dispatch_kernel<1"),
    ("route_finalize", r"route_finalize_kernel<1"),
    ("dispatch_count", r"dispatch_count_kernel"),
    ("dispatch_scatter", r"dispatch_scatter_kernel"),
    ("dispatch", r"dispatch_kernel"),
    ("combine", r"combine_kernel<1|combine_narrow_kernel<1"),
    # attention (the model port)
    ("attn_causal_prefill", r"causal_prefill_kernel<"),
    ("attn_paged_prefill", r"paged_prefill_kernel<"),
    ("attn_paged_decode", r"paged_decode_kernel<"),
    ("attn_paged_combine", r"paged_combine_kernel"),
)


PROFILE_DECODE = ROOT / "profiles" / "decode_b32_kernel_trace.txt"
PROFILE_PREFILL = ROOT / "profiles" / "prefill_4096_kernel_trace.txt"


def read_rocprof_us(key, path=PROFILE_DECODE):
    """A kernel's (average, median) duration in us from a committed rocprofv3
    summary (the `<key> calls=... avg=... us ... med=... us` lines written by
    --rocprof-summary); the median is None in summaries without one."""
    import re

    if not path.exists():
        return None, None
    for line in path.read_text().splitlines():
        m = re.match(rf"\s*{re.escape(key)}\s+calls=\s*\d+\s+avg=\s*([0-9.]+) us", line)
        if m:
            med = re.search(r"med=\s*([0-9.]+)", line)
            return float(m.group(1)), (float(med.group(1)) if med else None)
    return None, None


def rocprof_check(key, work, achieved, peak, path=PROFILE_DECODE):
    """The roofline recomputed from the committed rocprof figures of the same
    kernel at the same workload, beside the live figure: the average over the
    profiled launches that directly follow the layer's previous stage (the
    `key@layer` line), the launches the live in-layer figure times.  `work`
    is bytes (achieved in GB/s) or flops (achieved in TFLOP/s)."""
    avg, med = read_rocprof_us(key + "@layer", path)
    if avg is None:
        return {"rocprof_avg_us": None}
    rate = work / (avg * 1e-6) / (1e9 if peak == HBM_PEAK_GBS else 1e12)
    return {"rocprof_avg_us": avg, "rocprof_median_us": med,
            "rocprof_calls": f"{key}@layer",
            "rocprof_profile": str(path.relative_to(ROOT)),
            "frac_from_rocprof": rate / peak,
            "live_vs_rocprof": achieved / rate}


def read_traffic(name):
    """HBM bytes per launch of a kernel, from the committed counter summary."""
    if not TRAFFIC_JSON.exists():
        return None
    try:
        rec = json.loads(TRAFFIC_JSON.read_text()).get(name)
    except (ValueError, OSError):
        return None
    return None if rec is None else rec.get("hbm_bytes_per_launch")


def rocprof_summary(root: Path, write_traffic: bool) -> str:
    """Summarise rocprofv3 CSV output (kernel stats, FETCH_SIZE / WRITE_SIZE runs).

    Counters are KiB per dispatch.  Each is scaled by what it reads for the
    256 MiB device copy of ``--copy-probe`` (the largest copy dispatch):
    factor = 256 MiB / (counter KiB * 1024).
    """
    import csv
    from collections import defaultdict

    import re
    import statistics

    def key_of(name):
        for key, pat in KERNEL_KEYS:
            if re.search(pat, name):
                return key
        return "copy" if "copyBuffer" in name else None

    lines = []
    stats = {}
    durs = defaultdict(list)
    # the layer's own launch of a product: the dispatch that directly follows
    # the layer's previous stage (gate/up after the routing, down after gate/up)
    in_layer = {"decode_gateup_fused": ("route_partial",),
                "decode_products": ("route_partial",),
                "prefill_gateup": ("dispatch_hist",),
                "decode_down": ("decode_gateup_fused",),
                "prefill_down": ("prefill_gateup",)}
    for f in sorted(root.rglob("*kernel_trace.csv")):
        with open(f) as fh:
            rows = sorted(csv.DictReader(fh), key=lambda r: int(r["Start_Timestamp"]))
        prev = None
        for r in rows:
            k = key_of(r["Kernel_Name"])
            if k and k != "copy":
                d = (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3
                durs[k].append(d)
                if prev in in_layer.get(k, ()):
                    durs[k + "@layer"].append(d)
            prev = k
    for k, d in durs.items():
        stats[k] = {"calls": len(d), "avg_us": sum(d) / len(d), "med_us": statistics.median(d),
                    "min_us": min(d), "max_us": max(d)}
    # kernel_stats.csv (--stats): the whole run's kernels by total time
    for f in sorted(root.rglob("*kernel_stats.csv")):
        with open(f) as fh:
            rows = list(csv.DictReader(fh))
        if not rows:
            continue
        tot = sum(float(r["TotalDurationNs"]) for r in rows)
        calls = sum(int(r["Calls"]) for r in rows)
        lines.append(f"kernel stats ({f.name}): total kernel time {tot / 1e6:.1f} ms over "
                     f"{calls} launches")
        lines.append(" total ms   calls    avg us  kernel")
        for r in sorted(rows, key=lambda r: -float(r["TotalDurationNs"]))[:30]:
            name = r["Name"].replace("nvm::(anonymous namespace)::", "")
            name = re.sub(r"\((?!anonymous).*", "", name).replace("void ", "")
            lines.append(f"{float(r['TotalDurationNs']) / 1e6:9.1f} {int(r['Calls']):7d} "
                         f"{float(r['AverageNs']) / 1e3:9.2f}  {name[:90]}")
    if stats:
        lines.append("kernel trace (rocprofv3 --kernel-trace; per key: all calls; key@layer: "
                     "the calls that directly follow the layer's previous stage)")
        for k, s in stats.items():
            lines.append(f"  {k:16s} calls={s['calls']:5d} avg={s['avg_us']:8.2f} us "
                         f"med={s['med_us']:8.2f} us min={s['min_us']:8.2f} max={s['max_us']:8.2f}")
    counters = defaultdict(lambda: defaultdict(list))
    for f in sorted(root.rglob("*counter_collection.csv")):
        with open(f) as fh:
            for r in csv.DictReader(fh):
                k = key_of(r["Kernel_Name"])
                if k:
                    counters[r["Counter_Name"]][k].append(float(r["Counter_Value"]))
    traffic = {}
    factors = {}
    for cname in ("FETCH_SIZE", "WRITE_SIZE"):
        per = counters.get(cname)
        if not per or not per.get("copy"):
            continue
        probe_kib = max(per["copy"])
        factors[cname] = COPY_PROBE_BYTES / (probe_kib * 1024.0)
        lines.append(f"{cname}: 256 MiB copy reads {probe_kib:.0f} KiB -> factor "
                     f"{factors[cname]:.3f}")
        for k, vals in per.items():
            if k == "copy":
                continue
            kib = sum(vals) / len(vals)
            b = kib * 1024.0 * factors[cname]
            traffic.setdefault(k, {})[cname.lower() + "_bytes"] = b
            lines.append(f"  {k:16s} n={len(vals):5d} {kib:12.1f} KiB -> {b / 1e6:9.2f} MB per launch")
    # the other counters: per key, the median per dispatch; the MFMA busy
    # fraction where SQ_VALU_MFMA_BUSY_CYCLES and GRBM_GUI_ACTIVE come from one
    # run (GRBM_GUI_ACTIVE counts the dispatch's cycles once per XCD,
    # SQ_VALU_MFMA_BUSY_CYCLES sums the busy cycles of every SIMD)
    other = sorted(c for c in counters if c not in ("FETCH_SIZE", "WRITE_SIZE"))
    keys = sorted({k for c in other for k in counters[c] if k != "copy"})
    if keys:
        lines.append("counters (rocprofv3 --pmc; per key: median per dispatch):")
    for k in keys:
        vals = {c: statistics.median(counters[c][k]) for c in other if counters[c].get(k)}
        n = max(len(counters[c][k]) for c in other if counters[c].get(k))
        lines.append(f"  {k} (n={n}):")
        for c, v in vals.items():
            lines.append(f"    {c:28s} {v:16.0f}")
        waves = vals.get("SQ_WAVES")
        if waves:
            for c in ("SQ_INSTS_VALU", "SQ_INSTS_MFMA", "SQ_INSTS_LDS"):
                if c in vals:
                    lines.append(f"    per wavefront {c:14s} {vals[c] / waves:10.1f}")
        if "SQ_VALU_MFMA_BUSY_CYCLES" in vals and vals.get("GRBM_GUI_ACTIVE"):
            cycles = vals["GRBM_GUI_ACTIVE"] / MI355X_XCDS
            busy = vals["SQ_VALU_MFMA_BUSY_CYCLES"] / (cycles * MI355X_SIMDS)
            lines.append(f"    MFMA busy {100 * busy:.1f}% = SQ_VALU_MFMA_BUSY_CYCLES / "
                         f"(GRBM_GUI_ACTIVE / {MI355X_XCDS} XCDs x {MI355X_SIMDS} SIMDs); "
                         f"{cycles:.0f} cycles per dispatch")
    for k, rec in traffic.items():
        if k in stats:
            rec["avg_us"] = stats[k]["avg_us"]
    text = "\n".join(lines)
    if write_traffic and traffic:
        # merged per kernel and counter: the FETCH_SIZE and WRITE_SIZE runs
        # each add their own figure to the kernel's record
        old = json.loads(TRAFFIC_JSON.read_text()) if TRAFFIC_JSON.exists() else {}
        for k, rec in traffic.items():
            old.setdefault(k, {}).update(rec)
            cur = old[k]
            if "fetch_size_bytes" in cur and "write_size_bytes" in cur:
                cur["hbm_bytes_per_launch"] = cur["fetch_size_bytes"] + cur["write_size_bytes"]
        old["_factors"] = {**old.get("_factors", {}), **factors}
        TRAFFIC_JSON.parent.mkdir(exist_ok=True)
        TRAFFIC_JSON.write_text(json.dumps(old, indent=1, sort_keys=True) + "\n")
    return text


# The figures of each workload that the printed line carries (what a reader of
# one line compares); the whole record goes to the file of --record.
LINE_FIELDS = {
    "decode": ("layer_us", "layer_us_median", "tokens_per_s", "hbm_gbs"),
    "prefill": ("layer_us", "tokens_per_s", "layer_tflops", "in_layer_gateup_tflops",
                "in_layer_down_tflops"),
    "moe_235b": ("layer_us", "tokens_per_s", "hbm_gbs", "layer_tflops"),
    "dense": ("us",),
    "attention": ("us", "gbs", "tflops"),
    "e2e": ("decode_tokens_per_s", "decode_step_ms", "prefill_tokens_per_s",
            "generated_tokens_per_s"),
    "cpu_baseline": ("value", "unit", "cores", "kind", "sample", "tokens_per_s",
                     "routing_matches_gpu"),
    "roofline": ("kernel", "bound", "achieved", "peak", "unit", "frac", "avg_launch_us",
                 "algorithmic_bytes_per_launch", "traffic", "rocprof_avg_us",
                 "frac_from_rocprof"),
    "prefill_roofline": ("kernel", "bound", "achieved", "peak", "unit", "frac", "avg_launch_us",
                         "layer_frac", "traffic", "rocprof_avg_us", "frac_from_rocprof"),
}


def line_of(record: dict) -> str:
    """The JSON line of a record: every field of the headline, the chosen
    figures of the rest, numbers to six significant digits.  (The whole
    record is some 15 KB, longer than what a log's tail keeps of a line.)"""

    def digits(v):
        if isinstance(v, float):
            return float(f"{v:.6g}")
        if isinstance(v, dict):
            return {k: digits(x) for k, x in v.items()}
        return v

    def pick(v, fields):
        kept = {k: pick(x, fields) if isinstance(x, dict) else x for k, x in v.items()
                if isinstance(x, dict) or k in fields or k == "error"}
        return {k: x for k, x in kept.items() if x != {}}

    headline = ("value", "ms_per_step")  # as measured
    return json.dumps({k: v if k in headline else digits(pick(v, LINE_FIELDS[k]))
                       if k in LINE_FIELDS and isinstance(v, dict) else digits(v)
                       for k, v in record.items()})


def main():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=400)
    ap.add_argument("--warmup", type=int, default=40)
    ap.add_argument("--batch", type=int, default=32)
    ap.add_argument("--layers", type=int, default=8, help="distinct weight sets cycled")
    ap.add_argument("--no-extra", action="store_true", help="headline decode line only")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--no-graph", action="store_true")
    ap.add_argument("--copy-probe", action="store_true",
                    help="also run a plain 256 MiB device copy (calibrates HBM byte counters)")
    ap.add_argument("--prefill-only", action="store_true",
                    help="measure only the 4096-token prefill with uniform routing")
    ap.add_argument("--dense-only", action="store_true",
                    help="measure only the dense W4A16 projections (quantized_matmul)")
    ap.add_argument("--attention-only", action="store_true",
                    help="measure only paged decode attention")
    ap.add_argument("--moe-235b-only", action="store_true",
                    help="measure only the 235B-A22B-shaped MoE layer (decode 32, prefill 2048)")
    ap.add_argument("--e2e", action="store_true",
                    help="measure only the full 48-layer model through LLM.generate "
                         "(32 x 1024-token prompts, 256 greedy tokens)")
    ap.add_argument("--record", metavar="FILE",
                    help="write the whole record (every timing, with notes) to FILE as JSON")
    ap.add_argument("--rocprof-summary", metavar="DIR",
                    help="summarise rocprofv3 CSV output under DIR and exit (no GPU)")
    ap.add_argument("--write-traffic", action="store_true",
                    help="with --rocprof-summary: store HBM bytes per launch in profiles/traffic.json")
    args = ap.parse_args()

    if args.rocprof_summary:
        print(rocprof_summary(Path(args.rocprof_summary), args.write_traffic))
        return

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the MoE block is benchmarked on a single MI355X "
              "(expert/tensor sharding across GPUs is not implemented); run with --gpus 1",
              file=sys.stderr)
        sys.exit(2)

    import torch

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    H, E, I, k, gs = (SHAPE[n] for n in ("H", "E", "I", "k", "gs"))
    if args.copy_probe:
        src = torch.empty(256 << 20, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    if args.moe_235b_only:
        print(json.dumps({"moe_235b": shape_235b_bench(dev, args.steps)}), flush=True)
        return
    if args.e2e:
        r = e2e_bench(dev)
        log(f"[bench] e2e: decode {r['decode_tokens_per_s']:.0f} tok/s "
            f"({r['decode_step_ms']:.2f} ms/step), prefill {r['prefill_tokens_per_s']:.0f} tok/s")
        print(json.dumps({"e2e": r}), flush=True)
        return
    if args.attention_only:
        log("[bench] paged decode attention")
        print(json.dumps({"attention": attention_bench(dev)}), flush=True)
        return
    if args.dense_only:
        log("[bench] dense W4A16 projections")
        print(json.dumps({"dense": dense_bench(dev)}), flush=True)
        return
    if args.prefill_only:
        log("[bench] building 2 layers of 30B-A3B MoE weights")
        layers = make_layers(2, H, E, I, gs, dev)
        r = prefill_bench(layers, 4096, max(args.steps // 20, 8), 3, dev, False)
        log(f"[bench] prefill {r['routing']}: {r['layer_us']:.1f} us/layer, "
            f"{r['layer_tflops']:.0f} TFLOP/s, kernels {r['kernel_us']}")
        print(json.dumps({
            "metric": METRIC, "value": r["tokens_per_s"], "unit": "tokens/s", "n_gpus": 1,
            "steps": max(args.steps // 20, 8), "warmup": 3, "ms_per_step": r["layer_us"] / 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
            "data": "synthetic", "prefill": r,
            "config": {"workload": "Qwen3-30B-A3B-shaped MoE layer, prefill 4096 tokens, "
                                   "uniform routing", "tokens": 4096}}), flush=True)
        return
    log(f"[bench] building {args.layers} layers of 30B-A3B MoE weights")
    layers = make_layers(args.layers, H, E, I, gs, dev)

    log(f"[bench] decode B={args.batch}: {args.steps} steps, {args.warmup} warmup")
    head = decode_bench(layers, args.batch, args.steps, args.warmup, dev, not args.no_graph)
    log(f"[bench] decode B={args.batch}: {head['layer_us']:.1f} us/layer, "
        f"{head['hbm_gbs']:.0f} GB/s, kernels {head['kernel_us']}")

    gu_b, _ = bytes_per_expert(H, I, gs)
    fused = head["fused_products"]
    # the dominant kernel of the layer: both products in one launch where the
    # forward fuses them (B = 32 at this shape), else the gate/up product
    achieved = head["in_layer_products_gbs"] if fused else head["in_layer_gateup_gbs"]
    gateup_alone = {
        "kernel": "gemv3_kernel<bf16, gate/up+SwiGLU, routing finalised in the prologue, "
                  "K=2048> (nvm_moe_forward_stage 1)",
        "avg_launch_us": head["in_layer_kernel_us"]["gateup"],
        "algorithmic_bytes_per_launch": head["gateup_algorithmic_bytes"],
        "achieved": head["in_layer_gateup_gbs"],
        "frac": head["in_layer_gateup_gbs"] / HBM_PEAK_GBS,
        "traffic": read_traffic("decode_gateup_fused"),
        "back_to_back": {"avg_launch_us": head["forward_kernel_us"]["gateup"],
                         "achieved": head["forward_gateup_gbs"],
                         "frac": head["forward_gateup_gbs"] / HBM_PEAK_GBS},
        **rocprof_check("decode_gateup_fused", head["gateup_algorithmic_bytes"],
                        head["in_layer_gateup_gbs"], HBM_PEAK_GBS),
    }
    out = {
        "metric": METRIC,
        "value": head["tokens_per_s"],
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": head["layer_us"] / 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: seeded N(0,1) bf16 activations, N(0,0.02) weights MLX-affine "
                f"int4 g64 with bf16 scale/bias, {args.layers} distinct layers cycled",
        "config": {"workload": f"Qwen3-30B-A3B-shaped MoE layer, decode batch {args.batch}",
                   "tokens": args.batch, "hidden": H, "experts": E, "top_k": k,
                   "moe_intermediate": I, "group_size": gs, "bits": 4,
                   "weight_sets": args.layers, "timing": head["timing"]},
        "hbm_gbs": head["hbm_gbs"],
        # the published GPU timing protocol of the reference's figures: the
        # median of >= 100 individually timed layer calls after 10 warm-ups,
        # weight sets rotated
        "median_protocol": {"layer_us": head["layer_us_median"],
                            "tokens_per_s": head["tokens_per_s_median"],
                            "samples": head["median_samples"],
                            "hbm_gbs": head["layer_algorithmic_bytes"]
                            / (head["layer_us_median"] * 1e-6) / 1e9
                            if head["layer_us_median"] else None},
        "roofline": ({
            "kernel": "gemv3_kernel<bf16, gate/up+SwiGLU then down over one half of its "
                      "reduction, routing finalised in the prologue, K=2048> (the layer's "
                      "products launch, nvm_moe_forward_stage 4)",
            "bound": "hbm",
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": read_traffic("decode_products"),
            "algorithmic_bytes_per_launch": head["products_algorithmic_bytes"],
            "avg_launch_us": head["in_layer_kernel_us"]["products"],
            "timing": "HIP events: a graph of 64 runs of the layer's routing and products "
                      "stages minus a graph of 64 runs of its routing stage (8 weight sets "
                      "cycled), per launch",
            "back_to_back": {"avg_launch_us": head["forward_kernel_us"]["products"],
                             "achieved": head["forward_products_gbs"],
                             "frac": head["forward_products_gbs"] / HBM_PEAK_GBS},
            **rocprof_check("decode_products", head["products_algorithmic_bytes"], achieved,
                            HBM_PEAK_GBS),
            # the gate/up product alone as the forward's stage 1 runs it
            # (the layer's launch at batches that do not fuse the products)
            "gateup_alone": gateup_alone,
        } if fused else {
            **gateup_alone,
            "bound": "hbm",
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "timing": "HIP events: a graph of 64 runs of the layer's routing and gate/up stages "
                      "minus a graph of 64 runs of its routing stage (8 weight sets cycled), "
                      "per launch",
        }) | {
            # the same product without the routing in its prologue (the stage
            # entry point nvm_moe_expert_gateup), beside it
            "stage_entry_point": {
                "kernel": "gemv3_kernel<bf16, gate/up+SwiGLU, K=2048> (nvm_moe_expert_gateup)",
                "avg_launch_us": head["kernel_us_back_to_back"]["gateup"],
                "achieved": head["gateup_gbs"], "frac": head["gateup_gbs"] / HBM_PEAK_GBS,
                "traffic": read_traffic("decode_gateup")},
        },
        "layer_roofline": {"bound": "hbm", "achieved": head["hbm_gbs"], "peak": HBM_PEAK_GBS,
                           "unit": "GB/s", "frac": head["hbm_gbs"] / HBM_PEAK_GBS,
                           "algorithmic_bytes": head["layer_algorithmic_bytes"]},
        "decode": {str(args.batch): head},
    }
    if not args.no_extra:
        for T in (1, 8, 64):
            log(f"[bench] decode B={T}")
            r = decode_bench(layers, T, max(args.steps // 2, 16), args.warmup // 2, dev,
                             not args.no_graph)
            out["decode"][str(T)] = r
            log(f"[bench] decode B={T}: {r['layer_us']:.1f} us/layer, {r['hbm_gbs']:.0f} GB/s")
        out["prefill"] = {}
        psteps = max(args.steps // 20, 8)
        for zipf in (False, True):
            lay = layers if not zipf else make_layers(2, H, E, I, gs, dev, seed=777, zipf_s=1.1)
            log(f"[bench] prefill 4096 {'zipf' if zipf else 'uniform'}: {psteps} steps")
            r = prefill_bench(lay, 4096, psteps, 3, dev, zipf)
            out["prefill"][r["routing"]] = r
            log(f"[bench] prefill {r['routing']}: {r['layer_us']:.1f} us/layer, "
                f"{r['layer_tflops']:.0f} TFLOP/s, kernels {r['kernel_us']}")
            if zipf:
                del lay
        # the other reported workloads: a failure in one is recorded in its
        # field and does not take the headline line down with it
        extras = (("moe_235b", "235B-A22B-shaped MoE layer", lambda: shape_235b_bench(dev, args.steps)),
                  ("dense", "dense W4A16 projections", lambda: dense_bench(dev)),
                  ("attention", "paged decode attention", lambda: attention_bench(dev)),
                  ("e2e", "48-layer model through LLM.generate", lambda: e2e_bench(dev)))
        for key, what, fn in extras:
            log(f"[bench] {what}")
            try:
                out[key] = fn()
            except Exception as e:  # noqa: BLE001 - reported in the JSON line
                log(f"[bench] {what} failed: {e!r}")
                out[key] = {"error": repr(e)}
                torch.cuda.synchronize()
        if "decode_tokens_per_s" in out["e2e"]:
            log(f"[bench] e2e: decode {out['e2e']['decode_tokens_per_s']:.0f} tok/s, "
                f"prefill {out['e2e']['prefill_tokens_per_s']:.0f} tok/s")
        u = out["prefill"]["uniform"]
        out["prefill_roofline"] = {
            "kernel": "gemm_dma_kernel<gate/up+SwiGLU, fp16 copy of x staged by direct-to-LDS "
                      "loads> (the layer's gate/up launch at 4096 tokens, "
                      "nvm_moe_forward_stage 1)",
            "bound": "mfma", "achieved": u["in_layer_gateup_tflops"],
            "peak": MFMA_BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
            "frac": u["in_layer_gateup_tflops"] / MFMA_BF16_PEAK_TFLOPS,
            "avg_launch_us": u["in_layer_kernel_us"]["gateup"],
            "timing": "HIP events: a graph of 16 runs of the layer's routing and gate/up stages "
                      "minus a graph of 16 runs of its routing stage, per launch",
            "back_to_back": {"avg_launch_us": u["forward_kernel_us"]["gateup"],
                             "achieved": u["forward_gateup_tflops"],
                             "frac": u["forward_gateup_tflops"] / MFMA_BF16_PEAK_TFLOPS},
            "traffic": read_traffic("prefill_gateup"),
            "layer_frac": u["layer_mfma_frac"],
        }
        fl = 2.0 * 4096 * SHAPE["k"] * SHAPE["H"] * 2 * SHAPE["I"]
        out["prefill_roofline"].update(rocprof_check(
            "prefill_gateup", fl, u["in_layer_gateup_tflops"], MFMA_BF16_PEAK_TFLOPS,
            PROFILE_PREFILL))
    if not args.no_cpu:
        log(f"[bench] CPU baseline (~{args.cpu_seconds:.0f} s)")
        out["cpu_baseline"] = cpu_baseline(layers[0], args.batch, args.cpu_seconds, dev)
        cb = out["cpu_baseline"]
        log(f"[bench] CPU baseline: {cb['value']:.0f} tokens/s on {cb['cores']} threads, "
            f"{cb['single_thread']['tokens_per_s']:.0f} tokens/s on 1 thread "
            f"({cb['host']['cpu_model']})")
    if args.record:
        Path(args.record).write_text(json.dumps(out, indent=1) + "\n")
    print(line_of(out), flush=True)


if __name__ == "__main__":
    main()
