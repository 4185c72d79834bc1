"""The JSON line that bench.py prints: the contract's fields as measured, and
short enough (8 KB) that the tail of a log holds it whole.  No GPU."""

from __future__ import annotations

import importlib.util
import json
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def _bench():
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_line_holds_the_contract_and_fits_a_log():
    bench = _bench()
    # every timing a workload records: some thirty figures and long notes
    figures = {f"figure_{i}_us": 1.0 / 3 + i for i in range(30)}
    work = {"tokens": 32, "tokens_per_s": 1e6 / 3, "layer_us": 100 / 3, "us": 10 / 3,
            "hbm_gbs": 1e3 / 3, "note": "how it was timed " * 20, **figures}
    head = {"metric": bench.METRIC, "value": 1e6 / 3, "unit": "tokens/s", "n_gpus": 1,
            "steps": 400, "warmup": 40, "ms_per_step": 0.1 / 3, "higher_is_better": True,
            "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
            "config": {"workload": "decode batch 32", "tokens": 32}}
    record = {**head, "hbm_gbs": 1e4 / 3,
              "roofline": {"kernel": "gemv3_kernel", "frac": 1 / 3, "gateup_alone": dict(work),
                           **figures},
              "decode": {b: dict(work) for b in ("1", "8", "32", "64")},
              "prefill": {r: dict(work) for r in ("uniform", "zipf(1.1)")},
              "moe_235b": {w: dict(work) for w in ("decode_32", "prefill_2048")},
              "dense": {p: {"in": 2048, **{m: dict(work) for m in ("1", "32", "4096")}}
                        for p in ("q_proj", "k_proj", "o_proj", "lm_head")},
              "attention": {c: dict(work) for c in "abcde"},
              "e2e": {"error": "out of memory"},
              "cpu_baseline": {"value": 1e3 / 3, "host": dict(work)}}
    assert len(json.dumps(record)) > 16000
    line = bench.line_of(record)
    assert "\n" not in line and len(line) < 8000
    got = json.loads(line)
    assert {k: got[k] for k in head} == head
    assert list(got) == list(record)
    assert got["decode"]["8"] == {"tokens_per_s": 333333.0, "layer_us": 33.3333,
                                  "hbm_gbs": 333.333}
    assert got["dense"]["q_proj"]["32"] == {"us": 3.33333}
    assert got["roofline"]["frac"] == 0.333333
    assert got["e2e"] == {"error": "out of memory"}
