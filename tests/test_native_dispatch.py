"""The native call path refuses (``NotImplemented``: the Python path takes the call and says what is wrong) every tensor
that is not plain device memory, and malformed extent programs.  Fake tensors stand in for device memory, so nothing
is launched; launching itself is tested on the GPU."""

import pytest
import torch

from cleave_amd.runtime import dispatch

TENSOR, CONST, DIM, ADD, NEG = dispatch.TENSOR, dispatch.CONST, dispatch.DIM, dispatch.ADD, dispatch.NEG


def plan(grid=((CONST, 1), (CONST, 1), (CONST, 1))):
    return dispatch.native().make_plan([(TENSOR, "float16", [4, -1], 16)], 1, [], [("float16", [(CONST, 4)])], [],
                                       [(0, [list(g) for g in grid], (64, 1, 1), 0, [(0, 0), (1, 0)])], 2, None, lambda i: 0, 0, 0)


def test_tensors_without_plain_memory_are_refused_not_thrown_over():
    from torch._subclasses.fake_tensor import FakeTensorMode

    call = plan()
    with FakeTensorMode(allow_non_fake_inputs=True):
        fake = torch.empty(4, 8, dtype=torch.float16, device="cuda")
        assert call(fake) is NotImplemented
    assert call(fake) is NotImplemented
    assert call(torch.empty(4, 8, dtype=torch.float16)) is NotImplemented
    assert call(torch.empty(4, 8, dtype=torch.float16, device="meta")) is NotImplemented
    assert call() is NotImplemented and call(None) is NotImplemented and call(3.0) is NotImplemented
    seen = []
    torch.func.vmap(lambda x: (seen.append(call(x)), x)[1])(torch.empty(2, 4, 8, dtype=torch.float16, device="meta"))
    assert seen == [NotImplemented]


@pytest.mark.parametrize("program", [(), (NEG, CONST, 1), (ADD,), (CONST,), (CONST, 1, CONST, 2), (DIM, 7), (CONST, 1, 99)])
def test_malformed_extent_programs_are_refused(program):
    with pytest.raises(ValueError):
        plan((program, (CONST, 1), (CONST, 1)))


def test_a_paged_operator_without_its_query_names_it():
    from cleave_amd.frontend.paged import trace_paged
    from cleave_amd import examples
    from cleave_amd.pipeline.dynamic import PagedKernel

    attention = trace_paged(examples.paged_decode_op(32, 8, 128, 64), None).attention()
    kernel = PagedKernel(attention, attention.paging_spec(), "")
    args = [None] * len(attention.inputs)
    with pytest.raises(TypeError, match="missing input"):
        kernel(*args)
    with pytest.raises(TypeError, match="missing input"):
        kernel(*args, longest=3)


def _kernels():
    """A compiled kernel, a chain and a paged operator whose checked calls only say that they ran."""
    from types import SimpleNamespace

    import cleave_amd.lang as cl
    from cleave_amd import examples
    from cleave_amd.dynamic import OPERATORS
    from cleave_amd.frontend.paged import trace_paged
    from cleave_amd.pipeline.direct import source_for
    from cleave_amd.pipeline.dynamic import PagedKernel
    from cleave_amd.pipeline.kernel import Kernel, Param, Stage
    from cleave_amd.runtime.compile import CompiledKernel, _load_main_kernel_from_code

    def compiled(source, out_idx):
        kernel = CompiledKernel(_load_main_kernel_from_code(source), out_idx, b"")
        kernel._module = SimpleNamespace(function=lambda entry: 0)
        return kernel

    source = source_for(examples.matmul.trace(cl.f16, M=64, N=64, K=128), template="gemm", tiling=dict(BM=64, BN=64, BK=64, WM=2, WN=2))
    one = compiled(source, [-1])
    inputs = [p for p in one.params if p.role == "input"]
    stage = Stage("main", source, [-1], [Param(p.name, "input", i, p.shape) for i, p in enumerate(inputs)])
    chain = Kernel([stage], name="chain", input_names=["a", "b"], input_shapes=[p.shape for p in inputs], output_shapes=[(64, 64)])
    chain._callables = [compiled(source, [-1])]
    attention = trace_paged(examples.paged_decode_op(32, 8, 128, 64, dtype=cl.bf16)).attention()
    paged = PagedKernel(attention, attention.paging_spec(), "")
    paged._compiled = compiled(OPERATORS["gqa_paged_decode_h32_kv8_d128_ps64"].kernel_source(), None)
    for kernel in (one, chain, paged):
        kernel._checked_call = lambda *a, **k: "ran"
    query = torch.empty(1, 32, 128)
    calls = [lambda: one(0, 0), lambda: chain(0, 0), lambda: paged(query, *[0] * (len(attention.inputs) - 1))]
    plans = [lambda: one._plan, lambda: chain._plan, lambda: paged._plans.get(None)]
    return [(one, one), (chain, chain._callables[0]), (paged, paged._compiled)], calls, plans


@pytest.mark.parametrize("at", range(3), ids=["compiled", "chain", "paged"])
def test_kernels_without_a_native_plan_stay_on_the_checked_path(at, monkeypatch):
    """Beyond a plan's limits (nine launches), an extent it has no operator for, a module that is not there or does not
    load: the first call has run, and every call does."""
    def leaves(change, value):
        _, calls, plans = (made := _kernels())
        change(made[0][at][1])
        for _ in range(2):
            assert calls[at]() == "ran"
        assert plans[at]() is False if value is False else plans[at]()

    leaves(lambda k: None, True)
    leaves(lambda k: k.manifest.update(launches=k.manifest["launches"] * 9), False)
    leaves(lambda k: k.manifest["launches"][0].update(grid=["1 << 2", "1", "1"]), False)
    monkeypatch.setattr(dispatch, "_native", None)
    for name in ("absent.so", "libcleave_hip.so"):          # (the second has no such module in it)
        monkeypatch.setattr(dispatch, "MODULE_NAME", name)
        with pytest.warns(RuntimeWarning, match="step by step"):
            leaves(lambda k: None, False)


def test_a_stage_parameter_the_kernel_does_not_have_leaves_no_plan():
    (_, (chain, _), _), calls, plans = _kernels()
    from cleave_amd.pipeline.kernel import Param

    chain.stages[0].params.append(Param("PlaceHolder_unread", "input", 1, (4, 4)))
    assert calls[1]() == "ran" and plans[1]() is False
