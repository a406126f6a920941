"""GPU parity of the many-row attention kernels where a turn of their loops, a row block or a key range ends: step counts
around the rotation of the LDS images, workgroups of one row, partly filled and empty key ranges, scores that raise every
row's reference point on the way."""

import numpy as np
import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.pipeline.direct import kernel_for
from oracle import program_oracle

pytestmark = pytest.mark.gpu

LOCKSTEP, PHASED = dict(SHARED=1), dict(SHARED=1, PHASED=1)
# outputs are averages of unit-variance values, below 4 in magnitude: a rounding of the result is 2^-9 (f16) or 2^-6 (bf16) of that
# scale at most; the weights' own roundings average out below it
ATOL = {"f16": 4e-3, "bf16": 2.5e-2}


def check(fn, dtype, shapes, tiling, args=None, seed=11):
    prog = fn.trace(getattr(cl, dtype), **shapes)
    args = prog.random_inputs(seed=seed) if args is None else args(prog)
    print(f"attention form {prog.name} {dtype} {shapes} {tiling}", flush=True)
    out = kernel_for(prog, template="attn_prefill", tiling=tiling)(*args)
    torch.cuda.synchronize()
    want = program_oracle.evaluate(prog, list(args))[0]
    np.testing.assert_allclose(out.float().cpu().numpy(), want, rtol=1e-2, atol=ATOL[dtype])


@pytest.mark.parametrize("tiling", [LOCKSTEP, PHASED], ids=["lockstep", "phased"])
@pytest.mark.parametrize("keys", [1, 31, 32, 33, 64, 65, 97, 128, 160, 193, 256, 257, 321, 449])
def test_key_counts_around_the_rotation_of_the_images(tiling, keys):
    check(C.gqa_decode_exact, "f16", dict(HQ=2, HKV=1, SQ=70, SKV=keys, D=128), tiling)
    check(C.gqa_decode_exact, "bf16", dict(HQ=2, HKV=2, SQ=33, SKV=keys, D=64), tiling)


@pytest.mark.parametrize("tiling", [LOCKSTEP, PHASED, dict(SHARED=1, KEYS=3)], ids=["lockstep", "phased", "ranges"])
def test_every_row_of_a_chip_full_of_workgroups(tiling):
    """All outputs against float64 on the card: 2^-11 of the output for its rounding and as much for the weights'."""
    shapes = dict(HQ=16, HKV=8, SQ=2048, SKV=1100, D=128)
    q, k, v = C.gqa_decode_exact.trace(cl.f16, **shapes).random_inputs(seed=3)
    out = kernel_for(C.gqa_decode_exact.trace(cl.f16, **shapes), template="attn_prefill", tiling=tiling)(q, k, v)
    for h in range(16):
        w = torch.softmax((q[h].double() @ k[h // 2].double().T) * 128 ** -0.5, dim=-1)
        want = w @ v[h // 2].double()
        assert ((out[h].double() - want).norm() / want.norm()).item() < 2.0 ** -10


@pytest.mark.parametrize("rows", [1, 16, 127, 128, 129, 255, 256, 257, 513])
def test_row_counts_around_a_workgroup(rows):
    for tiling in (LOCKSTEP, PHASED):
        check(C.gqa_decode_exact, "f16", dict(HQ=3, HKV=3, SQ=rows, SKV=100, D=128), tiling)


@pytest.mark.parametrize("widths", [(64, 128), (128, 64), (192, 128), (192, 64)])
def test_phased_widths(widths):
    check(C.mla_prefill, "f16", dict(H=2, SQ=300, SKV=200, DK=widths[0], DV=widths[1]), PHASED)


def test_phased_with_normalised_queries_and_keys_and_without_a_softmax():
    check(C.qknorm, "f16", dict(HQ=8, HKV=2, SQ=100, SKV=300, D=128), dict(PHASED, KPRE=1))
    scaled = lambda prog: [(t.float() / 8).to(t.dtype) if i == 0 else t for i, t in enumerate(prog.random_inputs(seed=29))]  # noqa: E731
    prog = C.matmul_matmul.trace(cl.f16, H=2, SQ=300, SKV=130, D=64)
    args = scaled(prog)
    want = program_oracle.evaluate(prog, list(args))[0]
    for tiling in (PHASED, dict(SHARED=1, KEYS=3)):
        out = kernel_for(prog, template="attn_prefill", tiling=tiling)(*args)
        # weights are raw scores here, rounded to 11 bits, and their sums cancel
        np.testing.assert_allclose(out.float().cpu().numpy(), want, rtol=1e-2, atol=1e-2 + np.abs(want).max() * 2.0 ** -9)


@pytest.mark.parametrize("keys,ranges", [(256, 2), (257, 2), (300, 4), (290, 8), (1000, 5)])
def test_key_ranges_inside_an_operator(keys, ranges):
    """Ranges of whole 32-key steps: equal, with a partly filled last step, shorter and empty last ones."""
    check(C.gqa_decode_exact, "f16", dict(HQ=4, HKV=2, SQ=75, SKV=keys, D=128), dict(SHARED=1, KEYS=ranges))
    check(C.gqa_decode_exact, "bf16", dict(HQ=2, HKV=2, SQ=130, SKV=keys, D=64), dict(SHARED=1, KEYS=ranges))


@pytest.mark.parametrize("tiling", [LOCKSTEP, PHASED, dict(SHARED=1, KEYS=3)], ids=["lockstep", "phased", "ranges"])
def test_scores_that_rise_along_the_keys(tiling):
    """Every row's reference point is raised several times on the way (weights taken again, sums and accumulators moved)."""
    def rising(prog):
        q, k, v = prog.random_inputs(seed=5)
        q[..., 0] = 4.0
        k[..., 0] = torch.linspace(0.0, 35.0 * 128 ** 0.5 / (4 * 1.4427), k.shape[1], device=k.device).to(k.dtype)
        return q, k, v

    check(C.gqa_decode_exact, "f16", dict(HQ=4, HKV=2, SQ=150, SKV=600, D=128), tiling, args=rising)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tiling", [LOCKSTEP, PHASED, dict(SHARED=1, KEYS=3)], ids=["lockstep", "phased", "ranges"])
def test_a_value_that_is_the_same_for_every_key_comes_back_exactly(tiling, dtype):
    """64-wide heads add the weights up as they multiply them, rounded: what is left of a constant value's error is that of two
    sums of 600 positive terms in 32 bits, far below the 2^-12 and 2^-9 that would reach the next 16-bit number."""
    prog = C.gqa_decode_exact.trace(getattr(cl, dtype), HQ=4, HKV=2, SQ=150, SKV=600, D=64)
    q, k, v = prog.random_inputs(seed=21)
    v[:] = (1.9 - torch.arange(64, device=v.device) / 128).to(v.dtype)
    out = kernel_for(prog, template="attn_prefill", tiling=tiling)((q.float() * 4).to(q.dtype), k, v)
    assert torch.equal(out, v[:1, :1].expand_as(out))


@pytest.mark.parametrize("d,tiling", [(d, t) for t in (LOCKSTEP, PHASED, dict(SHARED=1, KEYS=3)) for d in (64, 128, 256)
                                      if d < 256 or "PHASED" not in t])
def test_a_row_does_not_depend_on_the_rows_beside_it(d, tiling):
    """Every other row's scores rise along the keys, so that its reference point is raised on the way; the rows between them keep
    their bits whether that happens beside them or not."""
    prog = C.gqa_decode_exact.trace(cl.f16, HQ=2, HKV=2, SQ=290, SKV=700, D=d)
    q, k, v = prog.random_inputs(seed=8)
    q = (q.float() * 2).to(q.dtype)
    q[..., 0] = 0.0
    k[..., 0] = torch.linspace(0.0, 40.0 * d ** 0.5 / (4 * 1.4427), k.shape[1], device=k.device).to(k.dtype)
    kernel = kernel_for(prog, template="attn_prefill", tiling=tiling)
    calm = kernel(q, k, v)
    q[:, 1::2, 0] = 4.0
    beside = kernel(q, k, v)
    assert torch.equal(calm[:, ::2], beside[:, ::2]) and not torch.equal(calm[:, 1::2], beside[:, 1::2])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("d", [64, 128])
def test_both_kernels_round_the_weights_at_the_same_places(d, dtype):
    """Where no row outgrows its first reference point (logits of standard deviation 1), the two kernels' weights are the same
    numbers; what is left is the order of sums in 32 bits, which moves a 16-bit result in less than one case of a hundred."""
    prog = C.gqa_decode_exact.trace(getattr(cl, dtype), HQ=4, HKV=2, SQ=200, SKV=1000, D=d)
    args = prog.random_inputs(seed=17)
    a, b = (kernel_for(prog, template="attn_prefill", tiling=t)(*args) for t in (LOCKSTEP, PHASED))
    assert (a != b).float().mean().item() < 0.01


@pytest.mark.parametrize("place", [0, 40, 130, 261])
@pytest.mark.parametrize("d,tiling", [(d, t) for t in (LOCKSTEP, PHASED, dict(SHARED=1, KEYS=3)) for d in (64, 128, 256)
                                      if d < 256 or "PHASED" not in t])
def test_infinite_and_undefined_scores(d, tiling, place):
    """A key with an infinite feature, in the first step, the second, a middle one and the last: rows that see it at +inf or as a NaN
    are NaN, rows that see it at -inf give it no weight, and a NaN in a query row stays in that row."""
    prog = C.gqa_decode_exact.trace(cl.f16, HQ=2, HKV=2, SQ=150, SKV=262, D=d)
    q, k, v = prog.random_inputs(seed=9)
    q[0, :, 0] = torch.where(torch.arange(150, device=q.device) % 3 == 0, 1.0, -1.0).to(q.dtype)
    q[0, 7, 0] = 0.0
    q[1, 5, 3] = float("nan")
    k[0, place, 0] = float("inf")
    out = kernel_for(prog, template="attn_prefill", tiling=tiling)(q, k, v).double().cpu()
    want = torch.softmax((q.double().cpu() @ k.double().cpu().transpose(1, 2).contiguous()) * d ** -0.5, dim=-1) @ v.double().cpu()
    assert torch.isnan(want[0, ::3]).all() and torch.isnan(want[0, 7]).all() and torch.isnan(want[1, 5]).all()
    assert torch.equal(torch.isnan(out), torch.isnan(want)) and torch.isnan(want).any(dim=-1).sum() == 52
    np.testing.assert_allclose(out.nan_to_num(0).numpy(), want.nan_to_num(0).numpy(), rtol=1e-2, atol=ATOL["f16"])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("widths", [(192, 192), (128, 256), (192, 256), (256, 256)], ids=lambda w: f"{w[0]}_{w[1]}")
def test_widths_with_a_compute_unit_to_themselves(widths, dtype):
    """Key counts around a turn of four (192 / 256: three) images, and scores that rise along the keys, so that the accumulators are
    moved out of the matrix half of the registers and back."""
    def rising(prog):
        q, k, v = prog.random_inputs(seed=5)
        q[..., 0] = 4.0
        k[..., 0] = torch.linspace(0.0, 35.0 * widths[0] ** 0.5 / (4 * 1.4427), k.shape[1], device=k.device).to(k.dtype)
        return q, k, v

    for keys in (1, 33, 97, 128, 129, 300):
        check(C.mla_prefill, dtype, dict(H=2, SQ=140, SKV=keys, DK=widths[0], DV=widths[1]), LOCKSTEP)
    check(C.mla_prefill, dtype, dict(H=2, SQ=140, SKV=600, DK=widths[0], DV=widths[1]), LOCKSTEP, args=rising)


def test_search_proposes_them_behind_the_first_four():
    from cleave_amd.pipeline.direct import stage_graph
    from cleave_amd.schedule import search_tiling

    def forms(topk, **shapes):
        return [c.tiling for c in search_tiling(stage_graph(C.gqa_decode_exact.trace(cl.f16, **shapes)), topk=topk)]

    many = dict(HQ=32, HKV=8, SQ=4096, SKV=4096, D=128)
    assert PHASED in forms(8, **many) and LOCKSTEP not in forms(8, **many)
    assert PHASED not in forms(4, **many) and not any("KEYS" in t for t in forms(8, **many))
    shorter = dict(many, SKV=1024)
    assert PHASED in forms(8, **shorter) and LOCKSTEP in forms(8, **shorter)
    few = forms(8, HQ=32, HKV=8, SQ=193, SKV=3897, D=128)
    assert dict(SHARED=1, KEYS=4) in few
