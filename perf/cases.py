"""What the compiled operators are measured on: the work a model server or a user's program hands them.

Every case names an operator of ``cleave_amd.examples`` (a ``@jit`` program), its sizes and its element type.  ``prepare``
compiles the operator once per size, as a program does at start-up (``cleave_amd.compile`` with a short search; a paged
operator is compiled once for all its sizes), and makes the tensors of one call on the GPU.  ``run`` is the call.

Cases: linear layers from a skinny latency-bound product to the largest square one, with odd and ragged sizes; the fused
RMSNorm -> linear of a decode step and the SwiGLU of a prompt; decode attention over dense and paged caches, grouped-query
and latent (MLA); prompt attention, dense and causal over ragged batches.
"""

from __future__ import annotations

import contextlib
import io
import math
import random

import torch

import cleave_amd
import cleave_amd.lang as cl
from cleave_amd import examples
from cleave_amd.dynamic import OPERATORS
from cleave_amd.pipeline import EvalConfig, ScheduleConfig

DTYPES = {"f16": (cl.f16, torch.float16), "bf16": (cl.bf16, torch.bfloat16)}
RAGGED_PREFILL = "gqa_ragged_prefill_causal_h32_kv8_d128"
MLA_PREFILL = "mla_paged_prefill_causal_h16_ckv512_kpe64_ps1"
TOKEN_DECODE = "gqa_paged_decode_h32_kv8_d128_ps1"
MLA_SCALE = 192 ** -0.5


def listed():
    return [
        # the smallest call: a narrow projection with a long contraction, a few microseconds of work
        dict(name="linear_small", op="matmul", dtype="f16", M=128, N=128, K=4096),
        # the normalised up-projection of one decode step of sixteen sequences: one pass over the weight
        dict(name="decode_norm_linear", op="rmsnorm_matmul", dtype="f16", M=16, N=11008, K=4096),
        # one decode step of eight sequences with 8192 cached keys (their 8 kv heads are 64 units, 256 query heads)
        dict(name="decode_gqa", op="gqa_decode_exact", dtype="f16", HQ=256, HKV=64, SQ=1, SKV=8192, D=128),
        # one latent-attention decode step of sixteen sequences
        dict(name="decode_mla", op="mla_decode", dtype="bf16", B=16, H=128, D=512, PE=64, SKV=4096),
        # a serving batch: 32 requests of 256 to 16384 tokens, pages of 64 in random order
        dict(name="paged_decode", op="paged_decode", dtype="f16", page=64, batch=32, shortest=256, longest=16384, lengths=5),
        # a young batch over a token table: 16 short requests, where latency is all there is
        dict(name="paged_decode_short", op="paged_decode", dtype="bf16", page=1, batch=16, shortest=8, longest=128, lengths=1),
        # prompts of ten requests packed into one call
        dict(name="prefill_ragged", op="ragged_prefill", dtype="bf16", batch=10, shortest=64, longest=2500, prefix=0, lengths=2),
        # chunked prompts over cached prefixes, latent attention through a token table
        dict(name="prefill_mla_paged", op="mla_prefill", dtype="bf16", batch=24, shortest=16, longest=350, prefix=200, lengths=3),
        # prompt attention over dense tensors
        dict(name="attention_dense", op="gqa_decode_exact", dtype="f16", HQ=32, HKV=8, SQ=4096, SKV=4096, D=128),
        # gated feed-forward of a 4096-token prompt
        dict(name="swiglu_prompt", op="swiglu", dtype="f16", M=4096, N=14336, K=4096),
        # an ordinary linear layer whose rows and columns are no multiple of any tile
        dict(name="linear_ragged", op="matmul", dtype="f16", M=3000, N=5000, K=2048),
        # the largest: a square product, weight stored (N, K) as linear layers store it
        dict(name="linear_large", op="matmul_nt", dtype="bf16", M=8192, N=8192, K=8192),
    ]


# ------------------------------------------------------------------------------- drawn cases
def _spread(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], uniform over the logarithm."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step), min(hi // step, round(n / step))) * step


def _width(rng, lo, hi):
    """A feature width: usually a multiple of 64, sometimes only of 8 (what a row of 16-byte pieces needs)."""
    return _spread(rng, lo, hi, 64 if rng.random() < 0.7 else 8)


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "matmul_nt", "rmsnorm_matmul", "gqa_decode", "mla_decode", "paged_decode",
                       "token_decode", "ragged_prefill", "mla_prefill", "attention", "swiglu"])
    dtype = rng.choice(["f16", "bf16"])
    if kind in ("matmul", "matmul_nt"):
        return dict(op=kind, dtype=dtype, M=_spread(rng, 65, 6000), N=_width(rng, 128, 8192), K=_width(rng, 256, 8192))
    if kind == "rmsnorm_matmul":
        return dict(op=kind, dtype=dtype, M=_spread(rng, 1, 64), N=_width(rng, 1024, 16384), K=_spread(rng, 1024, 8192, 256))
    if kind == "gqa_decode":
        units = _spread(rng, 4, 128)
        return dict(op="gqa_decode_exact", dtype=dtype, HQ=units * rng.choice([1, 4, 8]), HKV=units, SQ=1,
                    SKV=_spread(rng, 256, 16384), D=rng.choice([64, 128]))
    if kind == "mla_decode":
        return dict(op=kind, dtype="bf16", B=_spread(rng, 1, 32), H=rng.choice([16, 64, 128]), D=512, PE=64,
                    SKV=_spread(rng, 256, 8192))
    if kind == "paged_decode":
        longest = _spread(rng, 512, 16384)
        return dict(op=kind, dtype="f16", page=64, batch=_spread(rng, 1, 64), shortest=longest // 64, longest=longest,
                    lengths=rng.randrange(1 << 20))
    if kind == "token_decode":
        longest = _spread(rng, 16, 4096)
        return dict(op="paged_decode", dtype="bf16", page=1, batch=_spread(rng, 1, 64), shortest=max(1, longest // 16),
                    longest=longest, lengths=rng.randrange(1 << 20))
    if kind == "ragged_prefill":
        longest = _spread(rng, 16, 4096)
        return dict(op=kind, dtype="bf16", batch=_spread(rng, 1, 16), shortest=max(1, longest // 32), longest=longest, prefix=0,
                    lengths=rng.randrange(1 << 20))
    if kind == "mla_prefill":
        longest = _spread(rng, 1, 512)
        return dict(op=kind, dtype="bf16", batch=_spread(rng, 1, 32), shortest=max(1, longest // 16), longest=longest,
                    prefix=rng.choice([0, 32, 200]), lengths=rng.randrange(1 << 20))
    if kind == "attention":
        hkv = rng.choice([4, 8])
        return dict(op="gqa_decode_exact", dtype=dtype, HQ=hkv * rng.choice([1, 4, 8]), HKV=hkv, SQ=_spread(rng, 128, 4096),
                    SKV=_spread(rng, 128, 4096), D=rng.choice([64, 128]))
    return dict(op="swiglu", dtype=dtype, M=_spread(rng, 65, 4096), N=_spread(rng, 512, 14336, 128), K=_spread(rng, 512, 8192, 64))


# ------------------------------------------------------------------------------- compiled operators
_KERNELS: dict = {}          # a program compiles an operator once and keeps it

# contraction (or key) ranges worth trying where a product or a cache has too few tiles to fill the chip
SPLITS = {"matmul": cl.Split("K", (4, 8)), "rmsnorm_matmul": cl.Split("K", (4, 8)), "mla_decode": cl.Split("SKV", (4, 8)),
          "decode": cl.Split("SKV", (8, 16))}


def _split_for(case):
    if case["op"] == "matmul" and case["M"] * case["N"] <= 1 << 20:
        return SPLITS["matmul"]
    if case["op"] == "gqa_decode_exact":
        return SPLITS["decode"] if case["SQ"] == 1 else False
    return SPLITS.get(case["op"], False) if case["op"] != "matmul" else False


def _compile_dense(case):
    split = _split_for(case)
    fn = getattr(examples, case["op"])
    shapes = {k: v for k, v in case.items() if isinstance(v, int) and k.isupper()}
    return cleave_amd.compile(fn, shapes=shapes, dtype=DTYPES[case["dtype"]][0], preset="fast", split=split, cache_kernels=False,
                              schedule=ScheduleConfig(topk=8, split_k=getattr(split, "factors", ())),
                              eval=EvalConfig(warmup=3, iters=30, max_parallel=0))


def _captured(name, *picks):
    """Some of a shipped operator's captured workloads, for its search."""
    from cleave_amd.dynamic import workloads
    from cleave_amd.runtime.autotune import workload_key

    op = OPERATORS[name]

    def generate():
        for i in picks:
            axes = op.workloads[i]
            yield (workload_key(axes), *workloads.case(name, axes, op.dims, op.page_size, op.scale, dtype=torch.bfloat16))

    return generate


def _compile_paged(case):
    dtype = DTYPES[case["dtype"]][0]
    config = dict(schedule=ScheduleConfig(topk=1), max_workloads=3)
    if case["op"] == "paged_decode" and case["page"] == 1:
        fn = examples.paged_decode_op(32, 8, 128, 1, dtype=dtype, name=TOKEN_DECODE)
        return cleave_amd.compile(fn, split=cl.Split("kv_len", (8,)), workloads=_captured(TOKEN_DECODE, 0, 1, 3), **config)
    if case["op"] == "paged_decode":
        fn = examples.paged_decode_op(32, 8, 128, case["page"], dtype=dtype)
        mix = cl.workloads.paged_decode(batch=(1, 32), kv_len=(512, 12288), samples=2)
        return cleave_amd.compile(fn, split=cl.Split("kv_len", (8,)), workloads=mix, **config)
    if case["op"] == "ragged_prefill":
        fn = examples.prefill_op(32, 8, 128, ragged=True, dtype=dtype, name=RAGGED_PREFILL)
        return cleave_amd.compile(fn, workloads=_captured(RAGGED_PREFILL, 0, 1, 3), **config)
    fn = examples.mla_paged_prefill_op(16, 512, 64, dtype=dtype, name=MLA_PREFILL)
    return cleave_amd.compile(fn, workloads=_captured(MLA_PREFILL, 0, 2, 3), **config)


PAGED = ("paged_decode", "ragged_prefill", "mla_prefill")


def _kernel(case):
    if case["op"] in PAGED:
        key = (case["op"], case["dtype"], case.get("page"))
    else:
        key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _KERNELS:
        with contextlib.redirect_stdout(io.StringIO()):
            _KERNELS[key] = _compile_paged(case) if case["op"] in PAGED else _compile_dense(case)
    return _KERNELS[key]


# ------------------------------------------------------------------------------- inputs
def _lengths(case):
    """``(query tokens, keys)`` of every request: part of the case, not of the seed."""
    rng = random.Random(case["lengths"])
    new = [rng.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]
    return new, [n + (rng.randint(0, case["prefix"]) if case.get("prefix") else 0) for n in new]


def _indptr(counts):
    out = [0]
    for n in counts:
        out.append(out[-1] + n)
    return torch.tensor(out, dtype=torch.int32, device="cuda")


def _dense_inputs(case, normal, uniform):
    op, at = case["op"], case.get
    if op in ("matmul", "matmul_nt"):
        r = at("K") ** -0.5
        return [uniform(r, at("M"), at("K")), uniform(r, at("K"), at("N")) if op == "matmul" else uniform(r, at("N"), at("K"))]
    if op == "rmsnorm_matmul":
        return [normal(1.0, at("M"), at("K")), 1 + normal(0.1, 1, at("K")), normal(at("K") ** -0.5, at("K"), at("N"))]
    if op == "swiglu":
        r = at("K") ** -0.5
        return [normal(1.0, at("M"), at("K")), normal(r, at("K"), at("N")), normal(r, at("K"), at("N"))]
    if op == "mla_decode":
        return [normal(0.5, at("B"), at("H"), at("D")), normal(0.5, at("B"), at("SKV"), at("D")),
                normal(0.5, at("B"), at("H"), at("PE")), normal(0.5, at("B"), at("SKV"), at("PE"))]
    return [normal(1.0, at("HQ"), at("SQ"), at("D")), normal(1.0, at("HKV"), at("SKV"), at("D")),
            normal(1.0, at("HKV"), at("SKV"), at("D"))]


def _paged_inputs(case, gen, normal):
    """The call's arguments and, for decode, the longest request in page-table units (a serving loop knows it)."""
    new, keys = _lengths(case)
    if case["op"] == "ragged_prefill":
        return [normal(1.0, sum(new), 32, 128), normal(1.0, sum(keys), 8, 128), normal(1.0, sum(keys), 8, 128), _indptr(new),
                _indptr(keys), 128 ** -0.5], {}
    if case["op"] == "mla_prefill":
        pool = sum(keys) + sum(keys) // 4 + 16
        table = torch.randperm(pool, generator=gen, device="cuda")[:sum(keys)].to(torch.int32)
        return [normal(1.0, sum(new), 16, 512), normal(1.0, sum(new), 16, 64), normal(1.0, pool, 1, 512), normal(1.0, pool, 1, 64),
                _indptr(new), _indptr(keys), table, MLA_SCALE], {}
    page = case["page"]
    pages = [-(-n // page) for n in keys]
    pool = sum(pages) + sum(pages) // 4 + 16
    table = torch.randperm(pool, generator=gen, device="cuda")[:sum(pages)].to(torch.int32)
    args = [normal(1.0, case["batch"], 32, 128), normal(1.0, pool, page, 8, 128), normal(1.0, pool, page, 8, 128), _indptr(pages), table]
    if page > 1:
        args.append(torch.tensor([n - (p - 1) * page for n, p in zip(keys, pages)], dtype=torch.int32, device="cuda"))
    return [*args, 128 ** -0.5], {"longest": max(pages)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]][1]

    def normal(scale, *shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=dtype).mul_(scale)

    def uniform(scale, *shape):
        return torch.rand(*shape, generator=gen, device="cuda", dtype=dtype).mul_(2).sub_(1).mul_(scale)

    kernel = _kernel(case)
    if case["op"] in PAGED:
        args, named = _paged_inputs(case, gen, normal)
    else:
        args, named = _dense_inputs(case, normal, uniform), {}
    return {"kernel": kernel, "args": args, "options": named}


def run(state):
    return state["kernel"](*state["args"], **state["options"])


# ------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    at = case.get
    op = case["op"]
    if op in ("matmul", "matmul_nt", "rmsnorm_matmul"):
        M, N, K = at("M"), at("N"), at("K")
        return {"bytes": 2 * (M * K + K * N + M * N + (K if op == "rmsnorm_matmul" else 0)), "flops": 2 * M * N * K}
    if op == "swiglu":
        M, N, K = at("M"), at("N"), at("K")
        return {"bytes": 2 * (M * K + 2 * K * N + M * N), "flops": 4 * M * N * K}
    if op == "mla_decode":
        rows, keys, width = at("B") * at("H"), at("B") * at("SKV"), at("D") + at("PE")
        return {"bytes": 2 * (rows * (width + at("D")) + keys * width), "flops": 2 * rows * at("SKV") * (width + at("D"))}
    if op == "gqa_decode_exact":
        rows, keys, d = at("HQ") * at("SQ"), at("HKV") * at("SKV"), at("D")
        return {"bytes": 2 * (2 * rows * d + 2 * keys * d), "flops": 4 * rows * at("SKV") * d}
    new, keys = _lengths(case)
    if op == "paged_decode":
        pages = sum(-(-n // at("page")) for n in keys)
        return {"bytes": sum(keys) * 4096 + 4 * pages + at("batch") * (2 * 32 * 128 * 2 + 32 * 4 + 8), "flops": 4 * sum(keys) * 32 * 128}
    seen = sum(q * (k - q) + q * (q + 1) // 2 for q, k in zip(new, keys))     # (query, key) pairs under the causal limit
    if op == "ragged_prefill":
        return {"bytes": sum(new) * 32 * (2 * 128 * 2 + 4) + sum(keys) * 4096 + 8 * at("batch"), "flops": 4 * seen * 32 * 128}
    return {"bytes": sum(new) * 16 * (2 * (576 + 512) + 4) + sum(keys) * (576 * 2 + 4) + 8 * at("batch"),
            "flops": 2 * seen * 16 * (576 + 512)}


def tolerance(case):
    """About four times what the listed cases differ by from the same path in float64: 2.1e-4 to 3.0e-4 in f16 (largest single
    difference 1.7e-3 of the outputs' scale), 1.7e-3 to 2.4e-3 in bf16 (2.8e-2): the rounding of the outputs and, in attention,
    of the softmax weights."""
    return {"rel": 9e-3, "max": 0.11} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 7e-3}
