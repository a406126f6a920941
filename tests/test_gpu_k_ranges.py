"""GPU parity of products whose contraction is dealt out to ranges inside an unsplit operator: ranges of whole steps, ranges that end
on a partly filled or an empty step, ragged rows and columns, both weight layouts, batches, SwiGLU; row lengths that are no whole
pieces of a store."""

import numpy as np
import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.pipeline.direct import kernel_for, source_for, stage_graph
from cleave_amd.runtime.compile import _compile, _load_main_kernel_from_code
from cleave_amd.schedule import search_tiling
from cleave_amd.schedule.policy import k_range
from oracle import program_oracle

pytestmark = pytest.mark.gpu

TILES = [(128, 256, 2, 4), (256, 256, 2, 4), (128, 128, 2, 4), (64, 128, 2, 2)]     # two-group kernel, its quad form, lock-step


def check(fn, dtype, shapes, tile, ranges, extra=()):
    prog = fn.trace(getattr(cl, dtype), **shapes)
    tiling = dict(zip(("BM", "BN", "WM", "WN"), tile), BK=64, KS=ranges, **dict(extra), **({"DMA": 1} if shapes["K"] % 64 else {}))
    args = prog.random_inputs(seed=13)
    print(f"k ranges {prog.name} {dtype} {shapes} {tiling}", flush=True)
    out = kernel_for(prog, template="gemm" if shapes["K"] % 64 else "gemm_dma", tiling=tiling)(*args)
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, list(args))[0]
    got = out.float().cpu().numpy()
    # sums in 32 bits in another order, then one rounding of the result
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < (2.0 ** -7 if dtype == "bf16" else 2.0 ** -10)
    np.testing.assert_allclose(got, want, rtol=2e-2, atol=2e-2 * np.abs(want).max())


@pytest.mark.parametrize("tile", TILES, ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("K,ranges", [(256, 2), (512, 4), (320, 3), (448, 2), (1000, 2), (3000, 4), (600, 3), (136, 2)])
def test_ranges(tile, K, ranges):
    assert k_range(K, ranges)
    check(C.matmul, "f16", dict(M=300, N=520, K=K), tile, ranges)
    check(C.matmul_nt, "bf16", dict(M=77, N=264, K=K), tile, ranges)


@pytest.mark.parametrize("K,ranges", [(512, 2), (448, 2), (1152, 4)])
def test_swiglu_ranges(K, ranges):
    for tile in TILES[:3]:
        check(C.swiglu, "f16", dict(M=150, N=384, K=K), tile, ranges, extra=(("SWIGLU", 1),))


def test_batched_ranges():
    prog = C.batched_matmul.trace(cl.f16, BX=2, BW=2, M=100, N=128, K=1024)
    args = prog.random_inputs(seed=4)
    out = kernel_for(prog, template="gemm_dma", tiling=dict(BM=128, BN=128, BK=64, WM=2, WN=4, KS=4))(*args)
    want = program_oracle.evaluate(prog, list(args))[0]
    assert np.linalg.norm(out.float().cpu().numpy() - want) / np.linalg.norm(want) < 2.0 ** -10


FORMS = [("gemm", dict(BM=64, BN=64, BK=64, WM=2, WN=2), None), ("gemm", dict(BM=32, BN=32, BK=64, WM=1, WN=1), 2),
         ("gemm_dma", dict(BM=64, BN=128, BK=64, WM=2, WN=2), None), ("gemm_dma", dict(BM=256, BN=256, BK=64, WM=2, WN=2), None),
         ("gemm_dma", dict(BM=128, BN=128, BK=64, WM=2, WN=4), 2), ("gemm_dma", dict(BM=128, BN=256, BK=64, WM=2, WN=4, KS=2), None)]


@pytest.mark.parametrize("N", [1, 2, 7, 261, 262, 263, 264])
@pytest.mark.parametrize("template,tiling,split", FORMS)
def test_columns_that_are_no_whole_pieces(template, tiling, split, N):
    """A (N, K) weight leaves N free: no store of a row's last columns reaches the next row, which is another workgroup's where a
    row ends on a tile's edge, or the memory behind the last one."""
    prog = C.matmul_nt.trace(cl.f16, M=70, N=N, K=512)
    args = prog.random_inputs(seed=13)
    print(f"columns {template} {tiling} split {split} N {N}", flush=True)
    loaded = _load_main_kernel_from_code(source_for(prog, template=template, tiling=tiling, split=split))
    room = torch.full((70 * N + 64,), 7.0, device="cuda", dtype=torch.float16)
    _compile(loaded, None)(*args, room[:70 * N].view(70, N))
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, list(args))[0]
    got = room.float().cpu().numpy()
    assert (got[70 * N:] == 7.0).all()
    np.testing.assert_allclose(got[:70 * N].reshape(70, N), want, rtol=2e-3, atol=2e-3 * np.abs(want).max())


def test_search_proposes_them_where_tiles_are_few():
    def ranges(fn, topk=8, **shapes):
        return [c.tiling["KS"] for c in search_tiling(stage_graph(fn.trace(cl.f16, **shapes)), topk=topk) if "KS" in c.tiling]

    assert ranges(C.matmul, M=655, N=3264, K=6912) == [3, 3] and ranges(C.matmul, topk=4, M=655, N=3264, K=6912) == []
    assert ranges(C.swiglu, M=156, N=3968, K=8064) == [3, 3]
    assert ranges(C.matmul, M=4096, N=4096, K=4096) == [] and ranges(C.matmul, M=906, N=1152, K=1024) == []
