"""GPU parity of the 256 x 256 matmul whose two wave groups alternate between memory and matrix work, against
the numpy oracle at the sizes where its walk can go wrong: two to five K steps (the loop, the two steps without
loads behind it, both stage parities), whole halves of a tile past the edge, edges of one row and of one
8-column piece, all operand layouts, split ranges, batches, half-height tail tiles and the SwiGLU form.
Tolerance 1e-2 / 1e-2 as for every f16 / bf16 kernel here (outputs are of order one or below, and one
rounding to bf16 is 2^-9)."""

import numpy as np
import pytest
import torch

import cleave_amd
import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.pipeline.direct import kernel_for
from oracle import program_oracle

pytestmark = pytest.mark.gpu


@cleave_amd.jit
def matmul_tn(x: cl.Tensor["K", "M"], w: cl.Tensor["K", "N"]):
    return x.mT @ w


def _check(fn, dtype, shapes, grid=(2, 4), split=None, **knobs):
    prog = fn.trace(dtype, **shapes)
    x, *weights = prog.random_inputs(seed=7)
    args = [x] + [(w.float() / shapes["K"] ** 0.5).to(w.dtype) for w in weights]
    tiling = dict(BM=256, BN=256, BK=64, WM=grid[0], WN=grid[1], **knobs)
    print(f"case {prog.name} {dtype} {shapes} {tiling} split={split}", flush=True)
    kernel = kernel_for(prog, template="gemm_dma", tiling=tiling, split=split)
    assert "gp_barrier" in kernel.get_kernel_source()
    got = kernel(*args)
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, [t.cpu() for t in args])[0]
    np.testing.assert_allclose(got.float().cpu().numpy().reshape(want.shape), want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("grid", [(2, 4), (4, 2)], ids=["2x4", "4x2"])
@pytest.mark.parametrize("m,n,k", [(256, 256, 128), (257, 264, 192), (100, 72, 256), (600, 776, 320), (129, 392, 448)])
@pytest.mark.parametrize("fn,dtype", [(C.matmul, cl.f16), (C.matmul_nt, cl.bf16), (matmul_tn, cl.f16)], ids=["nn", "nt", "tn"])
def test_layouts_edges_and_step_counts(fn, dtype, m, n, k, grid):
    if fn is matmul_tn:
        m = -(-m // 8) * 8                      # its A rows are read as 16-byte pieces along M
    _check(fn, dtype, dict(M=m, N=n, K=k), grid)


@pytest.mark.parametrize("tail", [1, 4, 8])
def test_half_height_tail_tiles(tail):
    _check(C.matmul, cl.f16, dict(M=512, N=1032, K=320), TAIL=tail)
    _check(C.matmul_nt, cl.bf16, dict(M=512, N=1032, K=256), grid=(4, 2), TAIL=tail)


def test_split_ranges_and_batches():
    _check(C.matmul, cl.f16, dict(M=300, N=264, K=768), split=3)
    _check(C.batched_matmul, cl.bf16, dict(BX=4, BW=2, M=264, N=136, K=192))


@pytest.mark.parametrize("m,n,k", [(256, 128, 128), (300, 384, 320)])
def test_swiglu(m, n, k):
    _check(C.swiglu, cl.f16, dict(M=m, N=n, K=k), SWIGLU=1)
    _check(C.swiglu, cl.bf16, dict(M=m, N=n, K=k), grid=(4, 2), SWIGLU=1)
