"""GPU parity of the matmul whose two wave groups alternate between memory and matrix work, against
the numpy oracle at the sizes where its walk can go wrong: two to seven K steps (the loop, the two steps without
loads behind it, both stage parities), a last step that K fills only partly, whole halves of a tile past the edge, edges of one row and of one
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


TILES = {"256x256_2x4": (256, 256, 2, 4), "256x256_4x2": (256, 256, 4, 2), "128x256_2x4": (128, 256, 2, 4),
         "128x256_4x2": (128, 256, 4, 2), "256x128_4x2": (256, 128, 4, 2)}


def _check(fn, dtype, shapes, tile=TILES["256x256_2x4"], split=None, **knobs):
    prog = fn.trace(dtype, **shapes)
    x, *weights = prog.random_inputs(seed=7)
    args = [x] + [(w.float() / shapes["K"] ** 0.5).to(w.dtype) for w in weights]
    tiling = dict(zip(("BM", "BN", "WM", "WN"), tile), BK=64, **knobs)
    print(f"case {prog.name} {dtype} {shapes} {tiling} split={split}", flush=True)
    kernel = kernel_for(prog, template="gemm_dma", tiling=tiling, split=split)
    phased = tile in TILES.values() and shapes["K"] // (split or 1) > 64
    assert phased == ("gp_barrier" in kernel.get_kernel_source())
    got = kernel(*args)
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, [t.cpu() for t in args])[0]
    np.testing.assert_allclose(got.float().cpu().numpy().reshape(want.shape), want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("tile", TILES.values(), ids=TILES)
@pytest.mark.parametrize("m,n,k", [(256, 256, 128), (257, 264, 192), (100, 72, 256), (600, 776, 320), (129, 392, 448)])
@pytest.mark.parametrize("fn,dtype", [(C.matmul, cl.f16), (C.matmul_nt, cl.bf16), (matmul_tn, cl.f16)], ids=["nn", "nt", "tn"])
def test_layouts_edges_and_step_counts(fn, dtype, m, n, k, tile):
    if fn is matmul_tn:
        m = -(-m // 8) * 8                      # its A rows are read as 16-byte pieces along M
    _check(fn, dtype, dict(M=m, N=n, K=k), tile)


@pytest.mark.parametrize("tile", [*TILES.values(), (64, 128, 2, 4), (128, 128, 2, 2)], ids=[*TILES, "64x128_lockstep", "128x128_lockstep"])
@pytest.mark.parametrize("k", [72, 136, 184, 248, 328, 440])
def test_partly_filled_last_step(tile, k):
    """Chunks past K come as zeros for both operands (every layout; batches, whose rows continue past K in memory), in the
    lock-step kernel too."""
    for fn, dtype in ((C.matmul, cl.f16), (C.matmul_nt, cl.bf16), (matmul_tn, cl.f16)):
        _check(fn, dtype, dict(M=304, N=264, K=k), tile)
    _check(C.batched_matmul, cl.f16, dict(BX=2, BW=2, M=130, N=136, K=k), tile)


@pytest.mark.parametrize("k", [8, 40, 136, 200, 328])
def test_partly_filled_last_step_of_three_stages_and_small_tiles(k):
    for tile, knobs in (((64, 64, 2, 2), dict(STAGES=3)), ((16, 32, 1, 2), {}), ((16, 64, 1, 4), {})):
        _check(C.matmul, cl.f16, dict(M=100, N=136, K=k), tile, **knobs)
        _check(C.matmul_nt, cl.bf16, dict(M=100, N=136, K=k), tile, **knobs)


@pytest.mark.parametrize("tail", [1, 4, 8])
def test_half_height_tail_tiles(tail):
    _check(C.matmul, cl.f16, dict(M=512, N=1032, K=320), TAIL=tail)
    _check(C.matmul_nt, cl.bf16, dict(M=512, N=1032, K=256), tile=TILES["256x256_4x2"], TAIL=tail)


@pytest.mark.parametrize("tail", [1, 4])
@pytest.mark.parametrize("k", [136, 200, 328, 392])
def test_half_height_tail_tiles_with_a_partly_filled_last_step(tail, k):
    """The phased and the lock-step kernel, whole tiles and halves (two to seven steps, both stage parities)."""
    _check(C.matmul, cl.f16, dict(M=512, N=1032, K=k), TAIL=tail)
    _check(C.matmul_nt, cl.bf16, dict(M=512, N=1032, K=k), tile=TILES["256x256_4x2"], TAIL=tail)
    _check(C.matmul, cl.f16, dict(M=256, N=264, K=k), tile=(128, 128, 2, 2), TAIL=tail)


@pytest.mark.parametrize("tile", [(128, 128, 2, 2), (256, 64, 4, 2), (64, 256, 2, 4)], ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("k", [40, 136, 200, 328])
def test_partly_filled_last_step_of_three_stages_on_larger_tiles(tile, k):
    for fn, dtype in ((C.matmul, cl.f16), (C.matmul_nt, cl.bf16), (matmul_tn, cl.f16)):
        _check(fn, dtype, dict(M=304, N=264, K=k), tile, STAGES=3)


@pytest.mark.parametrize("dtype", [cl.f16, cl.bf16], ids=["f16", "bf16"])
@pytest.mark.parametrize("fn", [C.rmsnorm_matmul_plain, C.rmsnorm_matmul_eps], ids=["plain", "eps"])
@pytest.mark.parametrize("k", [72, 200, 328])
def test_fused_norm_with_a_partly_filled_last_step(fn, dtype, k):
    """The rows' squares are summed over the images, zeros past K among them, and divided by K itself; as the search names
    such tilings (``gemm`` with DMA).  Every output is one rounding of a value of order one and the row scale's: 2e-2 as
    for whole steps in bf16 (8 bits), 1e-2 in f16."""
    for tile, m, knobs in (((16, 32, 1, 2), 100, {}), ((64, 64, 2, 2), 200, {}), ((256, 128, 4, 2), 304, {}), ((256, 256, 4, 2), 512, dict(TAIL=2))):
        shapes = dict(M=m, N=264, K=k)
        prog = fn.trace(dtype, **shapes)
        ins = [t.to(dtype.torch) for t in C.inputs_plain_norm(shapes)]
        tiling = dict(zip(("BM", "BN", "WM", "WN"), tile), BK=64, DMA=1, **knobs)
        print(f"case {prog.name} {dtype} {shapes} {tiling}", flush=True)
        kernel = kernel_for(prog, template="gemm", tiling=tiling)
        assert "gd_sumsq" in kernel.get_kernel_source()
        got = kernel(*[t.cuda() for t in ins])
        torch.cuda.synchronize()
        want = program_oracle.evaluate(prog, ins)[0]
        tol = 2e-2 if dtype is cl.bf16 else 1e-2
        np.testing.assert_allclose(got.float().cpu().numpy(), want, rtol=tol, atol=tol)


@pytest.mark.parametrize("tile,kw", [((16, 16), 8), ((16, 32), 4), ((32, 16), 2), ((32, 32), 8), ((32, 64), 4), ((64, 64), 4), ((16, 16), 16)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else f"kw{v}")
@pytest.mark.parametrize("k", [8, 64, 200, 512, 1096])
def test_waves_that_share_the_contraction(tile, kw, k):
    """Fewer steps than waves (some own none), one to many steps per wave, a partly filled last step, ragged edges."""
    for fn, dtype in ((C.matmul, cl.f16), (C.matmul_nt, cl.bf16), (matmul_tn, cl.f16)):
        _check(fn, dtype, dict(M=72, N=104, K=k), (*tile, 1, 1), KW=kw)
    _check(C.batched_matmul, cl.f16, dict(BX=4, BW=2, M=50, N=72, K=k), (*tile, 1, 1), KW=kw)


def test_split_ranges_and_batches():
    for tile in (TILES["256x256_2x4"], TILES["128x256_2x4"]):
        _check(C.matmul, cl.f16, dict(M=300, N=264, K=768), tile, split=3)
        _check(C.batched_matmul, cl.bf16, dict(BX=4, BW=2, M=264, N=136, K=192), tile)


@pytest.mark.parametrize("m,n,k", [(256, 128, 128), (300, 384, 320)])
def test_swiglu(m, n, k):
    _check(C.swiglu, cl.f16, dict(M=m, N=n, K=k), tile=TILES["128x256_2x4"], SWIGLU=1)
    _check(C.swiglu, cl.f16, dict(M=m, N=n, K=k), tile=TILES["256x128_4x2"], SWIGLU=1)
    _check(C.swiglu, cl.f16, dict(M=m, N=n, K=k), SWIGLU=1)
    _check(C.swiglu, cl.bf16, dict(M=m, N=n, K=k), tile=TILES["256x256_4x2"], SWIGLU=1)


@pytest.mark.parametrize("m,n,k", [(192, 256, 128), (193, 264, 192), (320, 72, 256), (130, 520, 136), (700, 392, 200), (385, 264, 328), (64, 256, 448)])
def test_tiles_whose_halves_are_128_and_64_rows(m, n, k):
    """Two to seven steps, a partly filled last one, edges within either half and whole halves past the edge; batches, ranges and SwiGLU."""
    tiling = dict(BM=192, BN=256, BK=64, WM=2, WN=4)
    for fn, dtype, shapes, knobs in ((C.matmul, cl.f16, {}, {}), (C.matmul_nt, cl.bf16, {}, {}), (C.batched_matmul, cl.bf16, dict(BX=4, BW=2), {}),
                                     *([(C.matmul, cl.f16, {}, dict(KS=2))] if k >= 256 else []), *([(C.swiglu, cl.f16, {}, dict(SWIGLU=1))] if k % 64 == 0 else [])):
        shapes = dict(shapes, M=m, N=n, K=k) if fn is not C.swiglu else dict(M=m, N=-(-n // 128) * 128, K=k)
        prog = fn.trace(dtype, **shapes)
        x, *weights = prog.random_inputs(seed=7)
        args = [x] + [(w.float() / k ** 0.5).to(w.dtype) for w in weights]
        print(f"case {prog.name} {dtype} {shapes} {knobs}", flush=True)
        kernel = kernel_for(prog, template="gemm_dma" if k % 64 == 0 else "gemm", tiling=dict(tiling, **knobs, **({} if k % 64 == 0 else dict(DMA=1))))
        assert "#define GP_UNEVEN" in kernel.get_kernel_source()
        got = kernel(*args)
        torch.cuda.synchronize()
        want = program_oracle.evaluate(prog, [t.cpu() for t in args])[0]
        np.testing.assert_allclose(got.float().cpu().numpy().reshape(want.shape), want, rtol=1e-2, atol=1e-2)
