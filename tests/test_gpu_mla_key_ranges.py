"""Latent attention whose keys are dealt out to ranges inside an unsplit operator: key counts at the edges of a step and of a range,
workgroups of 16 heads and of score and value waves, one and two head blocks to a range, batches that are and are not whole eights, and
both forms of the combine (up to 16 ranges one thread adds up, above that groups of threads).  The combine of an operator of 16 or 32
heads is a kernel by itself."""

import numpy as np
import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.codegen import HipCodeGen
from cleave_amd.lower.stages import split_stages
from cleave_amd.pipeline.direct import kernel_for, stage_graph
from cleave_amd.runtime.compile import _compile, _load_main_kernel_from_code
from cleave_amd.schedule import apply_tiling, search_tiling
from cleave_amd.schedule.policy import combine_groups
from oracle import program_oracle


@pytest.mark.gpu
@pytest.mark.parametrize("skv,ranges", [(33, 2), (64, 2), (65, 3), (289, 8), (1043, 5), (1043, 33), (703, 22)])
@pytest.mark.parametrize("batch,heads,tiling", [(3, 16, dict(WAVES=1, STAGES=2)), (1, 32, dict(WAVES=2)), (2, 64, dict(DUO=1)),
                                                (3, 128, dict(DUO=1, LDS_AHEAD=4, S_PANELS=4)), (8, 64, dict(DUO=1))],
                         ids=["h16", "h32", "duo", "duo128", "duo8"])
def test_ranges(batch, heads, tiling, skv, ranges):
    shapes = dict(B=batch, H=heads, D=512, PE=64, SKV=skv)
    prog = C.mla_decode.trace(cl.bf16, **shapes)
    args = prog.random_inputs(seed=skv, device="cpu")
    print(f"mla ranges {shapes} {tiling} {ranges}", flush=True)
    got = kernel_for(prog, template="mla_decode", tiling=dict(tiling, KEYS=ranges))(*[a.cuda() for a in args])
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, args)[0]
    got = got.float().cpu().numpy().reshape(want.shape)
    # weights rounded to 8 bits (2^-9 each, of either sign) and one rounding of the result (2^-9)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2.0 ** -7
    np.testing.assert_allclose(got, want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("heads", [16, 32, 64])
def test_the_combine_is_a_kernel_by_itself(heads):
    graph = stage_graph(C.mla_decode.trace(cl.bf16, B=2, H=heads, D=512, PE=64, SKV=640))
    combine = split_stages(graph, 8)[1]
    source = HipCodeGen().gen(apply_tiling(search_tiling(combine)[0]))
    assert _compile(_load_main_kernel_from_code(source), None).stats[0]["spilled_vgprs"] == 0


def test_search_proposes_them_where_workgroups_are_few():
    def ranges(**shapes):
        return [c.tiling["KEYS"] for c in search_tiling(stage_graph(C.mla_decode.trace(cl.bf16, D=512, PE=64, **shapes)), topk=8) if "KEYS" in c.tiling]

    assert ranges(B=3, H=16, SKV=7233) == [57, 38] and ranges(B=24, H=16, SKV=2869) == [18, 10, 5]
    assert ranges(B=6, H=128, SKV=7649) == [20, 10] and ranges(B=32, H=128, SKV=8192)[:1] == [4]
    assert ranges(B=2, H=16, SKV=32) == [] and ranges(B=32, H=16, SKV=40) == [2]
    assert combine_groups(48, 512, 57) == 8 and combine_groups(48, 64, 17) == 16
    assert combine_groups(48, 512, 16) == combine_groups(384, 512, 18) == combine_groups(48, 96, 57) == 1


@pytest.mark.parametrize("heads,halved", [(16, False), (32, False), (64, True), (80, False), (128, True)])
def test_the_cost_of_a_split_has_the_bytes_its_partials_are(heads, halved, monkeypatch):
    from cleave_amd.lower.stages import partial_buffers
    from cleave_amd.schedule import policy

    graph = stage_graph(C.mla_decode.trace(cl.bf16, B=2, H=heads, D=512, PE=64, SKV=4096))
    assert (partial_buffers(graph.lowered, 8)[2][2] == "bfloat16") == halved
    partial = split_stages(graph, 8)[0]
    cost = {c.key(): c.score for c in search_tiling(partial)}
    monkeypatch.setattr(policy, "mla_po_elem", lambda heads: True)
    for c in search_tiling(partial):
        if "DUO" not in c.tiling:
            assert (cost[c.key()] == c.score) == halved and cost[c.key()] >= c.score


@pytest.mark.gpu
@pytest.mark.parametrize("heads,width,tiling", [(16, 128, dict(WAVES=1, STAGES=2)), (48, 256, dict(WAVES=1, STAGES=3)), (32, 64, dict(WAVES=2)), (64, 256, dict(DUO=1))],
                         ids=lambda v: str(v) if isinstance(v, int) else "duo" if "DUO" in v else "w")
@pytest.mark.parametrize("skv,ranges", [(65, 2), (640, 5), (1043, 17), (1043, 33)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_ranges_of_other_widths(dtype, skv, ranges, heads, width, tiling):
    """Latent rows of 64 to 256 features, whose combine has 8 or 16 thread groups above 16 ranges."""
    prog = C.mla_decode.trace(getattr(cl, dtype), B=3, H=heads, D=width, PE=64, SKV=skv)
    args = prog.random_inputs(seed=skv + heads, device="cpu")
    print(f"mla ranges {dtype} h={heads} d={width} {tiling} {skv} / {ranges}", flush=True)
    got = kernel_for(prog, template="mla_decode", tiling=dict(tiling, KEYS=ranges))(*[a.cuda() for a in args]).float().cpu().numpy()
    want = program_oracle.evaluate(prog, args)[0]
    # weights and result rounded once each, to 2^-9 (bf16) or 2^-12 (f16), of either sign
    assert np.linalg.norm(got.reshape(want.shape) - want) / np.linalg.norm(want) < (2.0 ** -7 if dtype == "bf16" else 2.0 ** -10)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,batch", [(16, 3), (32, 2), (48, 1), (64, 2)])
@pytest.mark.parametrize("split,skv", [(4, 640), (8, 1043), (8, 97)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_the_split_form(dtype, split, skv, heads, batch):
    """Partial and combine in one kernel's launches and as two kernels: f32 value partials, or (64 heads) element ones normalised per
    split, which are rounded once more."""
    prog = C.mla_decode.trace(getattr(cl, dtype), B=batch, H=heads, D=512, PE=64, SKV=skv)
    args = prog.random_inputs(seed=heads, device="cpu")
    print(f"mla split {dtype} h={heads} {split} x {skv}", flush=True)
    cuda = [a.cuda() for a in args]
    fused = kernel_for(prog, split=split)(*cuda)
    partial, combine = (apply_tiling(search_tiling(g)[0]) for g in split_stages(stage_graph(prog), split))
    first, second = (_load_main_kernel_from_code(HipCodeGen().gen(p)) for p in (partial, combine))
    parts = _compile(first, first.manifest["out_idx"])(*cuda)
    assert parts[2].dtype == (prog.dtype.torch if heads == 64 else torch.float32)
    apart = _compile(second, second.manifest["out_idx"])(*parts)
    want = program_oracle.evaluate(prog, args)[0]
    for got in (fused, apart):
        got = got.float().cpu().numpy().reshape(want.shape)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < (2.0 ** -7 if dtype == "bf16" else 2.0 ** -10)
