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
