"""Paged decode over a token table whose split pair cuts the table into items: batches of so few requests that equal parts fill no more
than the chip run the pair of equal parts, which the search keeps beside it."""

import dataclasses
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import cleave_amd
import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.dynamic.paging import PagingSpec
from cleave_amd.frontend.paged import trace_paged
from cleave_amd.pipeline import ScheduleConfig, load
from cleave_amd.pipeline.dynamic import PagedKernel, calibrate_dispatch
from cleave_amd.runtime.autotune import WorkloadCandidate
from oracle import paged_oracle
from tests.test_gpu_chunk_tokens import token_table

RULE = {"min_tiles": 25, "lone_tiles": 11, "few_requests": 9, "kv_tile": 32, "page_size": 1}
SOURCES = {"split": "// items", "single": "// one", "fixed": "// parts"}


def operator(dispatch, sources):
    attention = trace_paged(C.paged_decode_op(32, 8, 128, 1, dtype=cl.bf16, name="op")).attention()
    return PagedKernel(attention, attention.paging_spec(), "// main", label="L", variant="solo", latency_us=1.0, dispatch=dispatch, dispatch_sources=sources)


def test_the_rule(tmp_path):
    kernel = operator({**RULE, "fixed": {"requests": 4, "until_tiles": 85, "label": "parts"}}, SOURCES)
    for k in (kernel, load(kernel.save(tmp_path / "k"))):
        assert k.dispatch_sources == SOURCES
        role = k.dispatch_role
        assert [role(n, 1) for n in (1, 320, 321, 84 * 32, 84 * 32 + 1, 10 ** 5)] == ["single", "single", "fixed", "fixed", "split", "split"]
        assert role(2882, 3) == role(3 * 84 * 32, 3) == role(3 * 84 * 32, 4) == "fixed" and role(2882, 1) == role(3 * 85 * 32, 4) == "split"
        assert role(2882, 5) == role(2882, 64) == role(2882) == "split" and role(300, 5) == "single"
    # without the pair's source, or without a rule for it (a directory saved before there was one): items or the single kernel
    for k in (operator(kernel.dispatch, {k: v for k, v in SOURCES.items() if k != "fixed"}), operator(RULE, SOURCES)):
        assert k.dispatch_role(2882, 3) == "split" and k.dispatch_role(320, 1) == "single"


@pytest.mark.parametrize("kv_heads,parts,requests", [(8, 8, 4), (4, 8, 8), (32, 8, 1), (64, 8, None)])
def test_the_calibration(monkeypatch, kv_heads, parts, requests):
    """Times of a lone request at 10, 100, 2000 and 16000 tokens: the equal parts ahead of the items up to the third."""
    lengths = {"a": 10, "b": 100, "c": 2000, "d": 16000}
    us = {"items": [8.1, 8.2, 9.3, 20.0], "one": [3.5, 6.7, 30.0, 200.0], "parts": [6.2, 6.3, 8.5, 28.0]}

    def factory(keep):
        return lambda: ((key, [torch.tensor([0, n])], []) for key, n in lengths.items())

    def timed(candidates, workloads, ramp_seconds):
        for i, (key, *_) in enumerate(workloads()):
            for c in candidates:
                c.latency_us[key] = us[c.label][i]

    monkeypatch.setattr("cleave_amd.runtime.autotune.benchmark_over_workloads", timed)
    monkeypatch.setattr("cleave_amd.pipeline.dynamic.lone_request", lambda kernel, inputs, expected, at: (inputs, expected))
    spec = PagingSpec(num_qo_heads=64, num_kv_heads=kv_heads)
    table = SimpleNamespace(params=[SimpleNamespace(name=f"PlaceHolder_{spec.indptr_input}", role="input")])
    pair, one, fixed = (WorkloadCandidate(label=n, source=n, kernel=table, split=parts, tiling=SimpleNamespace(kv_tile=32)) for n in us)
    one = dataclasses.replace(one, split=None)
    rule = calibrate_dispatch(pair, one, factory, spec, fixed)
    assert "fixed" not in calibrate_dispatch(pair, one, factory, spec)
    if requests is None:
        assert "fixed" not in rule
        return
    kept = rule["fixed"]
    assert kept["requests"] == requests and 63 < kept["until_tiles"] < 500 and kept["label"] == "parts"


@pytest.mark.gpu
def test_every_role_of_a_searched_operator(tmp_path):
    op = C.paged_decode_op(32, 8, 128, 1, dtype=cl.bf16, name="few_requests_op")
    mix = cl.workloads.paged_decode(batch=(1, 40), kv_len=(40, 6000), samples=3)
    kernel = cleave_amd.compile(op, schedule=ScheduleConfig(topk=1), split=cl.Split("kv_len", (8,)), workloads=mix, max_workloads=3)
    sources = kernel.dispatch_sources
    assert {"split", "single"} <= set(sources) and ("fixed" in sources) == ("fixed" in kernel.dispatch)
    for lens in ([5], [1500], [600, 2500, 40], [900, 3000, 2000, 1], [70] * 9, [33, 4000] * 10):
        args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in token_table(lens, sum(lens) + 9, dtype=torch.bfloat16)]
        want, want_lse = paged_oracle.decode(*[a.float().cpu() if i < 3 else a.cpu() for i, a in enumerate(args[:5])], lens, 1, args[-1], out_dtype="bfloat16")
        print(f"few requests {lens[:4]} x {len(lens)}: {kernel.dispatch_role(max(lens), len(lens))}", flush=True)
        for k in (kernel, load(kernel.save(tmp_path / f"k{len(lens)}_{lens[0]}"))):
            out, lse = k(*args, longest=max(lens))
            np.testing.assert_allclose(out.float().cpu().numpy(), want, rtol=1e-2, atol=1e-2)
            np.testing.assert_allclose(lse.cpu().numpy(), want_lse, rtol=1e-3, atol=1e-3)
