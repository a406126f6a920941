"""Paged decode cut into items of a token table (page size 1): item sizes around the 32-token step, the most that an item holds, one
chosen at launch; requests that end on, before and after an item's edge and span many items, empty ones, table entries outside the
pool; other head counts and widths.  Its combine, like that of items of larger pages, over requests of more items than one
round of its thread groups takes."""

import numpy as np
import pytest
import torch

from cleave_amd import examples as C
from cleave_amd.codegen import HipCodeGen, parse_manifest
from cleave_amd.dynamic.paging import PAGED_DECODE_SLAB, DenseAttention, PagingSpec, build_split_decode, CombineTiling
from cleave_amd.dynamic.paging.apply import MAX_CHUNK_TOKENS, UnsupportedTiling, chunk_pages_expr, max_chunk_pages
from cleave_amd.runtime.compile import eval_extent
from tests.test_gpu_paged import check, paged_kernel, run


def token_table(lens, num_pages, **kw):
    """Arguments of an operator of page size 1, which reads no last-page lengths."""
    args = C.paged_workload(lens, page_size=1, num_pages=num_pages, **kw)
    return [*args[:5], args[-1]]


LENS = [1, 31, 32, 33, 64, 0, 65, 700, 0, 1500, 96, 5]


@pytest.mark.gpu
@pytest.mark.parametrize("chunk", [1, 7, 32, 45, 64, MAX_CHUNK_TOKENS, -1])
@pytest.mark.parametrize("prefetch,lockstep", [(1, False), (2, False), (1, True)])
def test_items_of_a_token_table(chunk, prefetch, lockstep):
    args = token_table(LENS, 3000)
    check(args, LENS, 1, split=8, waves=8, chunk_pages=chunk, prefetch=prefetch, lockstep=lockstep)


@pytest.mark.gpu
def test_requests_longer_than_an_item_holds():
    lens = [4100, 2048, 2049, 0, 100]
    args = token_table(lens, 9000)
    check(args, lens, 1, split=8, waves=8, chunk_pages=MAX_CHUNK_TOKENS, lockstep=True)


@pytest.mark.gpu
def test_other_heads_and_widths():
    for hq, hkv, d in ((16, 4, 128), (32, 8, 64), (16, 2, 256)):
        args = token_table(LENS, 3000, hq=hq, hkv=hkv, d=d)
        check(args, LENS, 1, split=4, hq=hq, hkv=hkv, d=d, waves=hkv, chunk_pages=64, lockstep=True)


@pytest.mark.gpu
def test_table_entries_outside_the_pool_are_clamped():
    args = token_table([70, 40], 200)
    table = args[4]
    low, high = table.clone(), table.clone()
    low[3], high[100] = -7, 10 ** 6
    kernel = paged_kernel(page_size=1, split=8, waves=8, chunk_pages=32, lockstep=True)
    for hostile, at, row in ((low, 3, 0), (high, 100, 199)):
        tame = table.clone()
        tame[at] = row
        got = run(kernel, [*args[:4], hostile, *args[5:]])
        want = run(kernel, [*args[:4], tame, *args[5:]])
        assert all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("page", [1, 16])
@pytest.mark.parametrize("d", [64, 128])
def test_more_items_than_one_round_of_the_combine(page, d):
    """Groups of 8 (16 at 64 wide) take four items each a round: 31, 32, 33, 65 and 130 items."""
    unit = 32 if page == 1 else 16
    lens = [31 * unit, 32 * unit, 33 * unit, 0, 65 * unit - 3, 130 * unit]
    args = token_table(lens, 12000, d=d) if page == 1 else C.paged_workload(lens, page_size=page, num_pages=400, d=d)
    check(args, lens, page, d=d, split=8, waves=8, chunk_pages=32 if page == 1 else 1, lockstep=True)


def test_item_sizes():
    spec = PagingSpec(num_qo_heads=32, num_kv_heads=8, kind="paged_decode", page_size=1)
    sizes = [eval_extent(chunk_pages_expr(spec, -1), {spec.index_dim: n, spec.batch_dim: b}) for n, b in ((1, 1), (9000, 6), (68237, 64), (10 ** 7, 40), (5000, 300))]
    assert sizes == [32, 64, 384, MAX_CHUNK_TOKENS, MAX_CHUNK_TOKENS] and chunk_pages_expr(spec, 9999) == str(MAX_CHUNK_TOKENS)
    assert max_chunk_pages(spec) == MAX_CHUNK_TOKENS
    dense = DenseAttention(16, 32, 128, 512, "float16", "float16", waves=8, chunk_pages=MAX_CHUNK_TOKENS + 1, lockstep=True)
    with pytest.raises(UnsupportedTiling, match="chunk_pages in 1..2048"):
        build_split_decode(spec, dense, 8, CombineTiling(split=8))


@pytest.mark.gpu
@pytest.mark.parametrize("page", [1, 16])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_one_thread_for_the_items_of_many_rows(page, d):
    """Six items a round: 6, 7, 12, 13 and 19 items among short requests, and an empty one."""
    unit = 32
    lens = [6 * unit, 7 * unit, 1, 12 * unit - 5, 0, 13 * unit, 19 * unit] + [1 + i % 9 for i in range(200)]
    args = token_table(lens, 3200, d=d) if page == 1 else C.paged_workload(lens, page_size=page, num_pages=400, d=d)
    assert -(-args[4].numel() // (32 // page)) + len(lens) <= len(lens) * 32 * d // 1024       # (as many items as workgroups, or fewer)
    check(args, lens, page, d=d, split=8, waves=8, chunk_pages=32 // page, lockstep=True)


@pytest.mark.parametrize("page,d", [(1, 128), (64, 64), (64, 256)])
def test_who_adds_the_items_up(page, d):
    """Groups of threads where one thread per four columns would be fewer workgroups than there are items."""
    spec = PagingSpec(num_qo_heads=32, num_kv_heads=8, kind="paged_decode" if page == 1 else PAGED_DECODE_SLAB, page_size=page)
    dense = DenseAttention(16, 32, d, 512, "float16", "float16", waves=8, chunk_pages=32, lockstep=True)
    launches = parse_manifest(HipCodeGen().gen(build_split_decode(spec, dense, 8, CombineTiling(split=8, cols=min(128, d)))))["launches"]

    def grid(batch, table):
        return eval_extent(launches[1]["grid"][0], {spec.batch_dim: batch, spec.index_dim: table, "chunk_pages": 32})

    one = 10 * 32 * d // 1024                               # ten requests, one thread per four columns
    assert grid(10, 32 * (one - 10)) == one and grid(10, 32 * (one - 10) + 1) == 10 * 32 * max(1, d // 128)
    assert grid(0, 64) == 0
