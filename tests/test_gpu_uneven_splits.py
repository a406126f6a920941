"""Split-KV decode over key counts that the split factor does not divide: whole 32-key steps are dealt out,
ceil(steps / factor) to a range, so the last ranges are short or empty.  Key counts at the edges: one key, one
range only, one step more than whole ranges, and a count far from any multiple; GQA and MLA (16 heads
too, whose combine has no wave grid of its own).  Against the numpy oracle at 1e-2 / 1e-2."""

import numpy as np
import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.lower.stages import split_stages
from cleave_amd.core.errors import LoweringRejected
from cleave_amd.pipeline.direct import kernel_for, stage_graph
from oracle import program_oracle

pytestmark = pytest.mark.gpu


def _check(prog, args, **kw):
    print(f"case {prog.name} {[tuple(a.shape) for a in args]} {kw}", flush=True)
    got = kernel_for(prog, **kw)(*[a.cuda() for a in args])
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, args)[0]
    np.testing.assert_allclose(got.float().cpu().numpy().reshape(want.shape), want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("skv", [1, 31, 33, 289, 1043])
@pytest.mark.parametrize("tiling", [dict(WAVES=1), dict(WAVES=2, SKEW=30), dict(WAVES=4)], ids=["w1", "w2skew", "w4"])
def test_gqa_decode(skv, tiling):
    shapes = dict(HQ=8, HKV=8, SQ=1, SKV=skv, D=128)
    _check(C.gqa_decode_exact.trace(cl.f16, **shapes), C.inputs_c3(shapes), template="attn_decode", tiling=tiling, split=8)


@pytest.mark.parametrize("skv", [1, 33, 289, 613])
@pytest.mark.parametrize("heads,tiling", [(16, dict(WAVES=1)), (64, dict(WAVES=4)), (64, dict(DUO=1))], ids=["h16", "h64", "duo"])
def test_mla_decode(heads, tiling, skv):
    shapes = dict(B=1, H=heads, D=512, PE=64, SKV=skv)
    _check(C.mla_decode.trace(cl.bf16, **shapes), C.inputs_c4(shapes), template="mla_decode", tiling=tiling, split=8)


@pytest.mark.parametrize("skv", [1, 33, 289, 613])
def test_many_row_attention(skv):
    """The kernel whose waves share the keys: softmax, keys wider than values, QK-norm, and plain sums (their scale as in the
    chained tests: outputs follow the number of keys)."""
    shared = dict(template="attn_prefill", tiling=dict(SHARED=1), split=8)
    for fn, dtype, shapes in ((C.gqa_decode_exact, cl.f16, dict(HQ=8, HKV=2, SQ=70, SKV=skv, D=64)),
                              (C.mla_prefill, cl.bf16, dict(H=2, SQ=100, SKV=skv, DK=192, DV=128)),
                              (C.qknorm, cl.f16, dict(HQ=4, HKV=2, SQ=70, SKV=skv, D=128))):
        prog = fn.trace(dtype, **shapes)
        _check(prog, prog.random_inputs(seed=skv, device="cpu"), **shared)
    prog = C.matmul_matmul.trace(cl.f16, H=2, SQ=70, SKV=skv, D=64)
    first, *rest = prog.random_inputs(seed=skv, device="cpu")
    _check(prog, [(first.float() / (8 * skv)).to(first.dtype), *rest], **shared)


@pytest.mark.parametrize("skv", [33, 289])
def test_gqa_decode_of_narrow_heads_in_groups(skv):
    shapes = dict(HQ=64, HKV=8, SQ=1, SKV=skv, D=64)
    for waves in (1, 4):
        _check(C.gqa_decode_exact.trace(cl.f16, **shapes), C.inputs_c3(shapes), template="attn_decode", tiling=dict(WAVES=waves), split=16)


def test_factors_that_are_neither_divisors_nor_powers_of_two_are_still_refused():
    g = stage_graph(C.gqa_decode_exact.trace(cl.f16, HQ=8, HKV=8, SQ=1, SKV=289, D=128))
    for factor in (3, 6, 12):
        with pytest.raises(LoweringRejected, match="does not divide"):
            split_stages(g, factor)
