"""Infinite and undefined elements through the kernels that cut an attention's keys into ranges or items and fold them: an infinite value
stays infinite wherever its key has a weight, and elsewhere nothing of it shows; a key that a row sees at +inf makes that row
undefined, one that it sees at -inf has no weight."""

import numpy as np
import pytest
import torch

import cleave_amd.lang as cl
from cleave_amd import examples as C
from cleave_amd.pipeline.direct import kernel_for
from cleave_amd.schedule.policy import combine_groups
from oracle import paged_oracle
from tests.test_gpu_chunk_tokens import token_table
from tests.test_gpu_mla_prefill_stay import inputs as prefill_inputs, kernel as prefill_kernel
from tests.test_gpu_paged import paged_kernel, run

pytestmark = pytest.mark.gpu
INF = float("inf")


def same(out, want, rtol=1e-2, atol=1e-2):
    """Infinite and undefined elements at the same places, the others equal to the roundings of weights and results."""
    out, want = np.asarray(out, np.float64), np.asarray(want, np.float64)
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.array_equal(np.isinf(out), np.isinf(want))
    live = np.isfinite(want)
    assert np.array_equal(np.sign(out[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    np.testing.assert_allclose(out[live], want[live], rtol=rtol, atol=atol)


@pytest.mark.parametrize("keys,ranges,d", [(4032, 21, 128), (3264, 17, 128), (3264, 17, 64), (1600, 25, 64), (2048, 32, 128), (1280, 8, 128)])
@pytest.mark.parametrize("where", [0, 1])
def test_an_infinite_value_of_a_key_range(keys, ranges, d, where):
    """In the first and the last range; the combine by groups of 8 and 16 threads with and without slots past the last range, and the
    one that adds a row's ranges up in one thread."""
    assert combine_groups(4 * 128, d, ranges) == (1 if ranges <= 16 else 1024 // d)
    prog = C.gqa_decode_exact.trace(cl.f16, HQ=4, HKV=4, SQ=128, SKV=keys, D=d)
    q, k, v = prog.random_inputs(seed=21)
    v[1, where * (keys - 20) + 5, 3], v[2, where * (keys - 20) + 6, d - 1] = INF, -INF
    print(f"infinite value keys={keys} ranges={ranges} d={d} where={where}", flush=True)
    out = kernel_for(prog, template="attn_prefill", tiling=dict(SHARED=1, KEYS=ranges))(q, k, v).double().cpu()
    scores = q.double().cpu() @ k.double().cpu().transpose(1, 2).contiguous() * d ** -0.5
    want = torch.softmax(scores, dim=-1) @ v.double().cpu()
    assert torch.isinf(want[1, :, 3]).all() and torch.isinf(want[2, :, d - 1]).all() and torch.isinf(want).sum() == 256
    same(out, want, atol=4e-3)


@pytest.mark.parametrize("page,requests", [(1, 3), (64, 3), (1, 90), (64, 90)])
def test_an_infinite_value_of_an_item(page, requests):
    """In the first, a middle and the last item of requests; few requests of five to nine items, which are added up by groups of threads,
    and many of one to five, where one thread takes a row's."""
    unit = 32 if page == 1 else 64
    lens = [unit * (9 - 2 * i if requests == 3 else 1 + i % 3) for i in range(requests - 1)] + [5 * unit]
    places = {0: 3, requests // 2: lens[requests // 2] // 2, requests - 1: 5 * unit - 9}
    args = token_table(lens, sum(lens) + 8) if page == 1 else C.paged_workload(lens, page_size=64, num_pages=sum(lens) // 64 + 2)
    indptr, table = args[3].tolist(), args[4].tolist()
    for b, at in places.items():
        args[2][table[indptr[b] + at // page], at % page, 2, 7] = INF
    print(f"infinite value page={page} requests={requests}", flush=True)
    kernel = paged_kernel(page_size=page, split=8, waves=8, chunk_pages=32 if page == 1 else 1, lockstep=True)
    out, lse = run(kernel, args)
    want, want_lse = paged_oracle.decode(*args[:5], lens, page, args[-1], out_dtype="float16")
    assert np.isinf(want).sum() == 3 * 4                      # (a kv head's four query heads)
    same(out, want)
    np.testing.assert_allclose(lse, want_lse, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("place", [5, 40, 150])
def test_infinite_scores_of_a_token_table(place):
    """As the single kernel has them, up to the order of sums."""
    lens = [160, 64, 33]
    args = token_table(lens, 300)
    args[0][0, :, 0] = torch.where(torch.arange(32) % 3 == 0, 1.0, -1.0).to(args[0].dtype)
    args[1][args[4][place], 0, :, 0] = INF
    print(f"infinite score place={place}", flush=True)
    want, _ = run(paged_kernel(page_size=1, waves=8), args)
    out, _ = run(paged_kernel(page_size=1, split=8, waves=8, chunk_pages=32, lockstep=True), args)
    assert np.isnan(want[0, ::3]).all() and np.isnan(want).any(axis=-1).sum() == 11
    same(out, want)


@pytest.mark.parametrize("heads,tiling,ranges", [(16, dict(WAVES=1, STAGES=2), 17), (16, dict(WAVES=1, STAGES=2), 5), (64, dict(DUO=1), 20)])
@pytest.mark.parametrize("place", [3, 300, 630])
def test_infinite_and_undefined_scores_of_latent_key_ranges(heads, tiling, ranges, place):
    prog = C.mla_decode.trace(cl.bf16, B=2, H=heads, D=512, PE=64, SKV=640)
    q, kv, qpe, kpe = prog.random_inputs(seed=4)
    qpe[0, :, 0] = torch.where(torch.arange(heads, device=q.device) % 3 == 0, 1.0, -1.0).to(q.dtype)
    q[1, 2, 9] = float("nan")
    kpe[0, place, 0] = INF
    print(f"infinite score heads={heads} {tiling} ranges={ranges} place={place}", flush=True)
    one, cut = (kernel_for(prog, template="mla_decode", tiling=t)(q, kv, qpe, kpe).float().cpu() for t in (tiling, dict(tiling, KEYS=ranges)))
    nan = torch.isnan(one)
    assert nan[0, ::3].all() and nan[1, 2].all() and nan.any(dim=-1).sum() == -(-heads // 3) + 1
    # (both forms round the weights to 8 bits and the result once)
    same(cut.numpy(), one.numpy(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("place", [2, 37, 95])
def test_undefined_scores_of_workgroups_that_stay(place):
    """Bit for bit as one workgroup an item has them: an infinite rope feature, an undefined query row."""
    lens = [40, 7, 96, 4, 33]
    args = [a.cuda() if isinstance(a, torch.Tensor) else a for a in prefill_inputs(lens, [n + 10 for n in lens], 16, 512, "bfloat16", 0.05)]
    args[3][args[6][67 + place]] = INF                        # a key of the third request
    args[0][3, 5, 11] = float("nan")
    print(f"undefined score place={place}", flush=True)
    want, stay = (prefill_kernel(16, 512, "bfloat16", few)(*args) for few in (1 << 30, 0))
    assert torch.isnan(want[0][3, 5]).all() and torch.isnan(want[0]).any(dim=-1).sum() > 100
    for a, b in zip(stay, want):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a.nan_to_num(0), b.nan_to_num(0))
