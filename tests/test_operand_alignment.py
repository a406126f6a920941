"""Which inputs of a kernel have to start at a multiple of 16 bytes: those that its templates move straight into LDS.  The
call copies one that does not (a view one element into a buffer); what goes through registers is taken as it is."""

import pytest

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.codegen import ALIGN16, HipCodeGen
from cleave_amd.dynamic import OPERATORS
from cleave_amd.dynamic.paging import MLA_PAGED_PREFILL_CAUSAL, DenseMLA, MLASpec
from cleave_amd.dynamic.paging.apply import _mla_outputs, _mla_params, _mla_plan
from cleave_amd.pipeline.direct import source_for
from cleave_amd.runtime.compile import CompiledKernel, _load_main_kernel_from_code


def aligned(source):
    return {name.replace("PlaceHolder_", "") for name in CompiledKernel(_load_main_kernel_from_code(source), None, b"").aligned_inputs}


def mla_prefill_source(duo):
    spec, dense = MLASpec(num_qo_heads=16, kind=MLA_PAGED_PREFILL_CAUSAL, causal=True), DenseMLA(16, 512, 64, "bfloat16", "bfloat16")
    (params, ops), (outs, out_ops) = _mla_params(spec, dense), _mla_outputs(spec, dense)
    return HipCodeGen().gen(_mla_plan(spec, dense, "main", params + outs, {**ops, **out_ops}, tok=4, duo=duo))


def dense_source(fn, dtype, shapes, **kw):
    return source_for(fn.trace(dtype, **shapes), **kw)


def test_score_wave_mla_prefill_reads_its_queries_past_the_registers_too():
    assert aligned(mla_prefill_source(duo=False)) == {"CKV", "KPE"}
    assert aligned(mla_prefill_source(duo=True)) == {"QN", "QP", "CKV", "KPE"}


@pytest.mark.parametrize("tiling,want", [(dict(DUO=1), 4), (dict(WAVES=4), 2)], ids=["duo", "waves"])
def test_dense_mla(tiling, want):
    source = dense_source(C.mla_decode, cl.bf16, dict(B=1, H=64, D=512, PE=64, SKV=64), template="mla_decode", tiling=tiling)
    assert len(aligned(source)) == want


def test_matmuls_and_attention():
    shapes = dict(M=64, N=64, K=72)
    assert len(aligned(dense_source(C.matmul, cl.f16, shapes, template="gemm", tiling=dict(BM=64, BN=64, BK=64, WM=2, WN=2, DMA=1)))) == 2
    assert not aligned(dense_source(C.matmul, cl.f16, shapes, template="gemm", tiling=dict(BM=64, BN=64, BK=64, WM=2, WN=2)))
    assert len(aligned(dense_source(C.swiglu, cl.f16, dict(M=64, N=128, K=128), template="gemm_dma",
                                    tiling=dict(BM=64, BN=128, BK=64, WM=2, WN=2, SWIGLU=1)))) == 3
    attention = dict(HQ=8, HKV=8, SQ=128, SKV=128, D=128)
    assert len(aligned(dense_source(C.gqa_decode_exact, cl.f16, attention, template="attn_prefill", tiling=dict(SHARED=1)))) == 2
    assert not aligned(dense_source(C.gqa_decode_exact, cl.f16, {**attention, "SQ": 1}, template="attn_decode", tiling=dict(WAVES=1)))


def test_registry_operators_take_queries_and_tables_as_they_are():
    for name, op in OPERATORS.items():
        want = {"CKV", "KPE"} if name.startswith("mla_paged_decode") else {"CKV_CACHE", "KPE_CACHE"} if name.startswith("mla") else \
            set() if "decode" in name else {"K_CACHE", "V_CACHE"} if "paged" in name else {"K", "V"}
        assert aligned(op.kernel_source()) == want, name


def test_a_saved_source_without_the_line_is_read_for_its_loads():
    old = "\n".join(line for line in mla_prefill_source(duo=True).splitlines() if not line.startswith(ALIGN16))
    assert aligned(old) == {"QN", "QP", "CKV", "KPE"}
