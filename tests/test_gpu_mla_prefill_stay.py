"""Paged MLA prefill on workgroups that stay (they draw items one after the other) against the numpy oracle and, bit for bit, against the
form of one workgroup an item, which does the same arithmetic: items of one to many steps, items cut by request boundaries, requests
without queries or keys, tokens that see no key, more than 64 requests, two head groups, narrower latent rows, more items than
the chip holds at once and fewer; where the rule between the two forms lies."""

import dataclasses

import numpy as np
import pytest
import torch

from cleave_amd.codegen import HipCodeGen, parse_manifest
from cleave_amd.dynamic import reference as dref
from cleave_amd.dynamic.paging import MLA_PAGED_PREFILL_CAUSAL, DenseMLA, MLASpec
from cleave_amd.dynamic.paging.apply import _mla_outputs, _mla_params, _mla_plan
from cleave_amd.runtime.compile import _compile, _load_main_kernel_from_code, eval_extent
from oracle import paged_oracle


def source(heads, ckv, dtype, few=None):
    spec = MLASpec(num_qo_heads=heads, kind=MLA_PAGED_PREFILL_CAUSAL, causal=True)
    dense = DenseMLA(heads, ckv, 64, dtype, dtype)
    params, ops = _mla_params(spec, dense)
    outs, out_ops = _mla_outputs(spec, dense)
    plan = _mla_plan(spec, dense, "main", params + outs, {**ops, **out_ops}, tok=4, duo=True)
    return HipCodeGen().gen(plan if few is None else dataclasses.replace(plan, tiling={**plan.tiling, "FEW": few}))


def kernel(heads, ckv, dtype, few):
    loaded = _load_main_kernel_from_code(source(heads, ckv, dtype, few))
    return _compile(loaded, loaded.manifest["out_idx"])


def inputs(q_lens, kv_lens, heads, ckv, dtype, scale):
    tq, tk = sum(q_lens), sum(kv_lens)
    args = dref.mla_paged_prefill_inputs((heads, ckv, 64, 2 * tk + 64, tk + 3, tq), q_lens, kv_lens, device="cpu", dtype=getattr(torch, dtype), scale=scale)
    args[6][tk:] = 2 ** 30
    return args


MIXED = [(37 * i * i) % 230 for i in range(44)]
CASES = {"ragged": ([1, 4, 5, 33, 0, 40, 7], [1, 4, 40, 33, 9, 300, 3]), "no keys": ([6, 0, 3], [0, 5, 3]), "long": ([90], [700]),
         "masked": ([3, 9], [2, 5]), "many": ([1] * 70, [1 + 3 * i for i in range(70)]), "halves": ([2, 2, 2], [16, 17, 65])}
LARGE = {"mixed": (MIXED, [q + (53 * i) % 200 - (q // 2 if i % 9 == 4 else 0) for i, q in enumerate(MIXED)]),
         "small requests": ([30 + i % 30 for i in range(90)], [30 + i % 30 + (i % 4) * 9 for i in range(90)]),
         "steps": ([4] * 40 + [600, 3], [1 + 25 * i for i in range(40)] + [600, 3])}


@pytest.mark.gpu
@pytest.mark.parametrize("heads,ckv,dtype,scale", [(16, 512, "bfloat16", 0.05), (32, 256, "bfloat16", -0.05), (16, 128, "float16", 0.3)])
@pytest.mark.parametrize("case", CASES)
def test_against_the_oracle(case, heads, ckv, dtype, scale):
    q_lens, kv_lens = CASES[case]
    args = inputs(q_lens, kv_lens, heads, ckv, dtype, scale)
    print(f"mla prefill stay {case} heads={heads} ckv={ckv} {dtype}", flush=True)
    out, lse = kernel(heads, ckv, dtype, 0)(*[a.cuda() if isinstance(a, torch.Tensor) else a for a in args])
    torch.cuda.synchronize()
    got_o, got_l = out.float().cpu().numpy(), lse.cpu().numpy()
    want_o, want_l = paged_oracle.mla_prefill(*args[:7], q_lens, kv_lens, args[7])
    # one rounding of the weights and one of the result (2^-9 relative in bf16, 2^-12 in f16)
    np.testing.assert_allclose(got_o, want_o, rtol=1e-2, atol=2e-2)
    live = np.isfinite(want_l)
    np.testing.assert_allclose(got_l[live], want_l[live], rtol=1e-5, atol=2e-4)
    assert np.all(np.isneginf(got_l[~live])) and np.all(got_o[~live.any(axis=1)] == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,ckv,scale", [(16, 512, 0.05), (16, 512, 0.6), (48, 128, 0.05)])
@pytest.mark.parametrize("case", LARGE)
def test_bit_for_bit_with_one_workgroup_an_item(case, heads, ckv, scale):
    args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in inputs(*LARGE[case], heads, ckv, "bfloat16", scale)]
    print(f"mla prefill stay {case} heads={heads} ckv={ckv} scale={scale} tokens={sum(LARGE[case][0])}", flush=True)
    want = kernel(heads, ckv, "bfloat16", 1 << 30)(*args)
    stay = kernel(heads, ckv, "bfloat16", 0)
    for _ in range(3):
        got = stay(*args)
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("heads", [16, 32])
def test_one_of_the_two_forms_is_launched(heads):
    manifest = parse_manifest(source(heads, 512, "bfloat16"))
    assert [l["entry"] for l in manifest["launches"]] == ["main_kernel", "main_kernel_tickets", "main_kernel_stay"]
    assert all(l["optional"] for l in manifest["launches"])

    def grids(tokens, batch):
        return [eval_extent(l["grid"][0], dict(total_q=tokens, batch=batch)) for l in manifest["launches"]]

    per_group = 768 // (heads // 16)
    assert grids(4 * (per_group - 8), 8) == [per_group, 0, 0] and grids(4 * (per_group - 8) + 1, 8) == [0, 1, 256]
    assert grids(1, 1) == [8, 0, 0] and grids(0, 0) == [0, 0, 0]
    scratch = next(p for p in manifest["params"] if p["role"] == "scratch")
    assert [eval_extent(scratch["shape"][0], dict(total_q=t, batch=8)) for t in (64, 8192)] == [0, 64]


@pytest.mark.parametrize("ckv,launches", [(128, 1), (256, 3), (384, 3), (512, 3)])
def test_rows_of_which_a_unit_holds_two_workgroups_run_one_an_item(ckv, launches):
    manifest = parse_manifest(source(16, ckv, "bfloat16"))
    assert len(manifest["launches"]) == launches and any(p["role"] == "scratch" for p in manifest["params"]) == (launches > 1)
    if launches == 1:
        assert not manifest["launches"][0].get("optional")
        assert eval_extent(manifest["launches"][0]["grid"][0], dict(total_q=40000, batch=8)) == 10008


@pytest.mark.gpu
def test_calls_that_share_their_scratch_need_none():
    """Overlapping calls through the fixed array would draw items from one counter: they run one workgroup an item."""
    args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in inputs(*LARGE["mixed"], 16, 512, "bfloat16", 0.05)]
    loaded = _load_main_kernel_from_code(source(16, 512, "bfloat16", 0))
    want = _compile(loaded, loaded.manifest["out_idx"])(*args)
    caller = _compile(loaded, None)
    assert caller.fixed_scratch_layout(dict(total_q=1 << 20, batch=44)) == ({}, 0)
    got = [torch.full_like(t, float("nan")) for t in want]
    caller.call_fixed_scratch(*args, *got)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_launches_are_named_by_their_place_in_the_manifest():
    """Also where a call leaves one out ahead of them."""
    loaded = _load_main_kernel_from_code(source(16, 512, "bfloat16"))
    kernel = _compile(loaded, None)
    few, many = dict(total_q=64, batch=2), dict(total_q=8192, batch=2)
    assert list(kernel._grids(few)) == [0] and list(kernel._grids(many)) == [1, 2] and list(kernel._grids(many, shared=True)) == [0]
    assert kernel._chosen(few, [0]) == [0] and kernel._chosen(many, [2]) == kernel._chosen(many, [-1]) == [1] and kernel._chosen(many, [2, 1]) == [1, 0]
    for dims, only in ((many, [0]), (few, [2]), (few, [0, 1])):
        with pytest.raises(ValueError, match="leaves out main_kernel"):
            kernel._chosen(dims, only)
    with pytest.raises(IndexError):
        kernel._chosen(many, [3])


@pytest.mark.gpu
def test_the_launch_that_was_asked_for_is_timed():
    args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in inputs([700] * 6, [900] * 6, 16, 512, "bfloat16", 0.05)]
    loaded = _load_main_kernel_from_code(source(16, 512, "bfloat16"))
    timed = _compile(loaded, loaded.manifest["out_idx"])
    print("mla prefill stay: one launch timed", flush=True)
    stay, clear = (timed.time(*args, warmup=4, iters=20, only=[i]) for i in (2, 1))
    assert stay > 4 * clear                                  # (well over 50 us, and a few)
    with pytest.raises(ValueError, match="leaves out main_kernel$"):
        timed.time(*args, only=[0])
