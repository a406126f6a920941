"""Outputs of native calls come from torch's own allocator whether or not the call passes torch's dispatcher: counted, given back,
usable on other streams, inference tensors in inference mode; under a profiler or a dispatch mode the allocation is seen there."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.pipeline.direct import kernel_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def call():
    prog = C.matmul.trace(cl.f16, M=256, N=512, K=128)
    kernel, args = kernel_for(prog), prog.random_inputs(seed=1)
    want = kernel(*args).clone()                       # (the first call makes the native plan)
    return lambda: kernel(*args), want


def test_outputs_are_counted_and_given_back(call):
    run, want = call
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = run()
    assert out.device.type == "cuda" and out.is_contiguous() and not out.requires_grad
    assert torch.cuda.memory_allocated() - before == 256 * 512 * 2
    assert torch.equal(out, want)
    out.record_stream(torch.cuda.Stream())
    del out
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    out = run()
    out.resize_(512, 512)
    assert out.shape == (512, 512)


def test_inference_mode(call):
    run, want = call
    with torch.inference_mode():
        out = run()
    assert out.is_inference() and torch.equal(out.clone(), want) and not run().is_inference()


def test_profiler_and_modes_see_the_allocation(call):
    run, want = call
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as seen:
        run()
    assert any(e.key == "aten::empty" for e in seen.key_averages())

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))

    names = []
    with Names():
        out = run()
    assert any("empty" in n for n in names) and torch.equal(out, want)


def test_graph_capture_uses_the_pool_of_the_graph(call):
    run, want = call
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = run()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
