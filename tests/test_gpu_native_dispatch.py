"""The native call path (``csrc/dispatch.cpp``) against the checked Python path it stands in for: same
results bit for bit for fused pairs, chains of stages, caller-owned outputs and paged operators with
run-time extents; the same errors where arguments do not fit; scratch of calls on different streams
and threads kept apart."""

import threading

import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd import pipeline as P
from cleave_amd.dynamic import reference as dref
from cleave_amd.dynamic.paging import PAGED_DECODE_SLAB, CombineTiling, DenseAttention, PagingSpec, build_split_decode
from cleave_amd.codegen import HipCodeGen
from cleave_amd.pipeline.direct import kernel_for
from cleave_amd.runtime.compile import _compile, _load_main_kernel_from_code

pytestmark = pytest.mark.gpu
SHAPES = dict(M=16, K=512, N=384)


def _split_kernel():
    kernel = kernel_for(C.rmsnorm_matmul.trace(cl.f16, **SHAPES), template="skinny", tiling=dict(WAVES_N=1, WAVES_K=2), split=4)
    args = [t.cuda() for t in C.inputs_c2(SHAPES)]
    want = kernel(*args)                       # (the first call goes the checked way and leaves a plan)
    assert kernel._plan
    return kernel, args, want


def test_fused_pair_and_its_errors():
    kernel, args, want = _split_kernel()
    assert torch.equal(kernel(*args), want) and torch.equal(kernel._checked_call(*args), want)
    with pytest.raises(TypeError, match="expects 3 arguments"):
        kernel(*args[:2])
    with pytest.raises(TypeError, match="dtype"):
        kernel(args[0].float(), *args[1:])
    with pytest.raises(ValueError, match="contiguous"):
        kernel(args[0].t().contiguous().t(), *args[1:])
    with pytest.raises(ValueError, match="shape"):
        kernel(args[0][:8], *args[1:])
    with pytest.raises(ValueError, match="only run on the GPU"):
        kernel(args[0].cpu(), *args[1:])
    with pytest.raises(TypeError, match="torch tensor"):
        kernel(None, *args[1:])


def test_chain_of_stages_is_one_plan(cache_root):
    kernel = P.compile(C.rmsnorm_matmul, shapes=SHAPES, dtype=cl.f16, split=cl.Split("K", (4,)), cache_kernels=False,
                       schedule=P.ScheduleConfig(topk=2, split_k=(4,)), eval=P.EvalConfig(warmup=1, iters=3, max_parallel=0))
    chain = next(k for k in (kernel, *kernel.report.contenders(top=8, within=100.0)) if len(k.stages) == 2)
    args = [t.cuda() for t in C.inputs_c2(SHAPES)]
    want = chain(*args)
    assert chain._plan and torch.equal(chain(*args), want) and torch.equal(chain(x=args[0], gamma=args[1], w=args[2]), want)
    with pytest.raises(ValueError, match="expected"):
        chain(args[0][:8], *args[1:])


def test_paged_pair_with_caller_owned_outputs_and_run_time_extents():
    spec = PagingSpec(num_qo_heads=32, num_kv_heads=8, kind=PAGED_DECODE_SLAB, page_size=64)
    dense = DenseAttention(16, 32, 128, 512, "float16", "float16", waves=8, chunk_pages=-1, lockstep=True)
    source = HipCodeGen().gen(build_split_decode(spec, dense, 8, CombineTiling(split=8)))
    kernel = _compile(_load_main_kernel_from_code(source), None)
    for lens in ([1], [70, 500, 64], [3000, 1, 200, 65, 64, 1000, 129]):
        pages = sum(-(-n // 64) for n in lens)
        args = dref.gqa_paged_decode_inputs((len(lens), 32, 8, 128, pages + 3, pages), lens, page_size=64, dtype=torch.float16)
        got, checked = ([torch.full((len(lens), 32, 128), float("nan"), dtype=torch.float16, device="cuda"),
                         torch.full((len(lens), 32), float("nan"), device="cuda")] for _ in range(2))
        assert kernel._checked_call(*args, *checked) is None and kernel(*args, *got) is None
        assert torch.equal(got[0], checked[0]) and torch.equal(got[1], checked[1]) and bool(torch.isfinite(got[1]).all())
    assert kernel._plan
    with pytest.raises(ValueError, match="conflicts"):
        kernel(*args, got[0][:2], got[1])


def test_threads_on_their_own_streams_do_not_share_scratch():
    kernel, args, _ = _split_kernel()
    inputs = [[t + 0 for t in args] for _ in range(4)]
    for i, ins in enumerate(inputs):
        ins[0] = ins[0] * (i + 1) + i
    wants = [kernel(*ins) for ins in inputs]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            outs = [kernel(*inputs[i]) for _ in range(50)]
            torch.cuda.current_stream().synchronize()
        wrong.extend(i for o in outs if not torch.equal(o, wants[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_operands_between_two_16_byte_pieces_are_copied_for_the_direct_to_lds_kernels():
    """A view one element into a buffer: the checked path and the native one give what the aligned operand gives."""
    shapes = dict(M=66, N=136, K=200)
    kernel = kernel_for(C.matmul.trace(cl.f16, **shapes), template="gemm", tiling=dict(BM=64, BN=64, BK=64, WM=2, WN=2, DMA=1))
    a, b = (torch.randn(*s, dtype=torch.float16, device="cuda") for s in ((66, 200), (200, 136)))
    want = kernel(a, b)
    moved = []
    for t in (a, b):
        buffer = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        moved.append(buffer[1:].view(t.shape).copy_(t))
    assert kernel._plan and kernel._plan(*moved) is NotImplemented
    assert torch.equal(kernel(*moved), want) and torch.equal(kernel._checked_call(*moved), want)


def _direct_to_lds_cases():
    from cleave_amd.dynamic.paging import MLA_PAGED_PREFILL_CAUSAL, DenseMLA, MLASpec
    from cleave_amd.dynamic.paging.apply import _mla_outputs, _mla_params, _mla_plan

    def mla_prefill(duo):
        spec, dense = MLASpec(num_qo_heads=16, kind=MLA_PAGED_PREFILL_CAUSAL, causal=True), DenseMLA(16, 512, 64, "bfloat16", "bfloat16")
        (params, ops), (outs, out_ops) = _mla_params(spec, dense), _mla_outputs(spec, dense)
        loaded = _load_main_kernel_from_code(HipCodeGen().gen(
            _mla_plan(spec, dense, "main", params + outs, {**ops, **out_ops}, tok=4, duo=duo)))
        q_lens, kv_lens = [3, 9], [40, 9]
        return _compile(loaded, loaded.manifest["out_idx"]), dref.mla_paged_prefill_inputs((16, 512, 64, 96, 49, 12), q_lens, kv_lens)

    def mla(tiling):
        shapes = dict(B=1, H=64, D=512, PE=64, SKV=70)
        return kernel_for(C.mla_decode.trace(cl.bf16, **shapes), template="mla_decode", tiling=tiling), C.inputs_c4(shapes)

    def attention():
        shapes = dict(HQ=8, HKV=8, SQ=130, SKV=70, D=128)
        return kernel_for(C.gqa_decode_exact.trace(cl.f16, **shapes), template="attn_prefill", tiling=dict(SHARED=1)), C.inputs_c3(shapes)

    return {"mla_prefill_duo": lambda: mla_prefill(True), "mla_prefill": lambda: mla_prefill(False), "mla_duo": lambda: mla(dict(DUO=1)),
            "mla": lambda: mla(dict(WAVES=4)), "attention": attention}


@pytest.mark.parametrize("case", _direct_to_lds_cases())
def test_operands_between_two_16_byte_pieces(case):
    """Every 16-bit operand in turn as a view one element into a buffer: the same bits as from the aligned one."""
    kernel, args = _direct_to_lds_cases()[case]()
    args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in args]

    def run(ins):
        got = kernel(*ins)
        return list(got) if isinstance(got, (list, tuple)) else [got]

    want = run(args)
    for i, t in enumerate(args):
        if isinstance(t, torch.Tensor) and t.element_size() == 2:
            buffer = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
            ins = [*args[:i], buffer[1:].view(t.shape).copy_(t), *args[i + 1:]]
            print(f"{case}: operand {i} {tuple(t.shape)} one element into its buffer", flush=True)
            assert all(torch.equal(a, b) for a, b in zip(run(ins), want)), i


@pytest.mark.parametrize("k", [128, 200], ids=["whole_steps", "partly_filled"])
def test_timed_and_allocation_free_calls_take_such_operands_too(k):
    shapes = dict(M=66, N=136, K=k)
    tile = dict(BM=64, BN=64, BK=64, WM=2, WN=2)
    kernel = kernel_for(C.matmul.trace(cl.f16, **shapes), **(dict(template="gemm", tiling=dict(tile, DMA=1)) if k % 64 else
                                                            dict(template="gemm_dma", tiling=tile)))
    owned = _compile(kernel.loaded, None)
    a, b = (torch.randn(*s, dtype=torch.float16, device="cuda") for s in ((66, k), (k, 136)))
    want = kernel(a, b)
    moved = [torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view(t.shape).copy_(t) for t in (a, b)]
    out = torch.zeros_like(want)
    owned.call_fixed_scratch(*moved, out)
    assert torch.equal(out, want)
    out.zero_()
    owned.time(*moved, out, warmup=1, iters=2, rotate=[(*moved, out)])
    assert torch.equal(out, want)
    kernel.time(*moved, warmup=1, iters=2)
    assert torch.equal(kernel.last_timed_outputs[0], want)


@pytest.mark.parametrize("change,error,text", [(dict(lds=1 << 20), "LdsExceeded", "LDS limit exceeded"), (dict(block=[2048, 1, 1]), "HipError", "1024 threads")])
def test_a_launch_the_library_refuses_raises_what_the_checked_path_raises(change, error, text):
    """Refused by the library's own checks, ahead of any launch."""
    from cleave_amd.runtime.dispatch import chain_plan

    kernel, args, _ = _split_kernel()
    kernel.manifest["launches"][0].update(change)
    plan = chain_plan([(kernel, None)])
    raised = []
    for call in (kernel._checked_call, plan):
        with pytest.raises(Exception, match=text) as e:
            call(*args)
        raised.append((type(e.value), str(e.value), getattr(e.value, "status", None)))
    assert raised[0] == raised[1] and raised[0][0].__name__ == error
