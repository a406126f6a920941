"""``cleave_amd.compile`` for paged operators.

The stages, in order (those of ``python/cleave/pipeline/dynamic.py:423-504``): trace the operator
and read its attention off the program; tile the dense body one block computes; wrap every tiling
in the operator's access layer (and, for decode layers, derive split-KV pairs from the single
kernels); check every candidate on every workload; time the correct ones; calibrate when a call
should run the split pair; hand back a ``PagedKernel``.  ``_Search`` carries the state from stage
to stage and keeps each stage's wall time.

A saved ``PagedKernel`` holds its program as JSON (``program.json``), never as a pickle: loading
a kernel directory executes nothing from it.
"""

from __future__ import annotations

import contextlib
import dataclasses
import json
import math
import time
from collections import Counter
from dataclasses import dataclass, field
from typing import Callable, Optional

from ..core.errors import CleaveError, SpecError
from .compile import resolve_configs
from .kernel import Kernel, Stage
from .plans import Plan, PlanSet, Refusal
from .superopt import superoptimize

PROGRAM_FILE = "program.json"
DISPATCH_FILE = "dispatch.json"


@dataclass(eq=False)
class PagedPlan(Plan):
    """A plan whose kernel text already exists (paging is applied while scheduling)."""

    source: str = field(default="", repr=False)
    dense: object = None          # what the access layer read off the dense tiling
    origin: str = "searched"      # or "derived split-K"


# ================================================================================ scheduling
def _emit(plan_or_pair) -> str:
    from ..codegen import HipCodeGen

    return HipCodeGen().gen(plan_or_pair)


def _layer_variants(spec):
    """``tiled plan -> [paged plans]`` for the spec's access layer: the causal prefill layers and
    the MLA prefill layer have several kernels per tiling and all of them go to the measurement."""
    from ..dynamic.paging import CAUSAL_KINDS, MLA_PAGED_PREFILL_CAUSAL, apply_paging
    from ..dynamic.paging import MLASpec
    from ..dynamic.paging.apply import mla_decode_variants, mla_prefill_variants, prefill_variants

    if spec.kind in CAUSAL_KINDS:
        return lambda tiled: prefill_variants(tiled, spec)
    if spec.kind == MLA_PAGED_PREFILL_CAUSAL:
        return lambda tiled: mla_prefill_variants(tiled, spec)
    if isinstance(spec, MLASpec):
        return lambda tiled: mla_decode_variants(tiled, spec)
    return lambda tiled: [apply_paging(tiled, spec)]


def schedule_paged(graphs, spec, config, *, split_graphs=(), filter_before_topk=False) -> PlanSet:
    """Plans for ``spec``: every dense graph is tiled, every tiling paged, and kernels whose text
    is already in the set are dropped.  With ``config.split_k`` (decode layers only) each single
    kernel also gives one split-KV pair per factor."""
    from ..dynamic.paging import SPLIT_KINDS, CombineTiling, build_split_decode, paging_accept, read_dense
    from ..lower import to_ir
    from ..schedule import apply_tiling, search_tiling

    started = time.perf_counter()
    plans, refusals, texts = [], [], set()

    def keep(graph, variant, tile, dense, source, rank, label, factor=None, origin="searched"):
        if source not in texts:
            texts.add(source)
            plans.append(PagedPlan(graph.index, variant, "main", tile, f"g{graph.index} {variant} {label}", rank,
                                   factor, graph, source=source, dense=dense, origin=origin))

    paged_forms = _layer_variants(spec)
    accept = paging_accept(spec) if filter_before_topk else None
    for graph in graphs:
        body = graph.program
        ir = to_ir(graph.structure, graph.symbol_map, graph.dtype, graph.dtype, [s.name for s in body.inputs], body.name)
        for rank, tile in enumerate(search_tiling(ir, topk=config.topk, accept=accept)):
            try:
                tiled = apply_tiling(tile)
                dense = read_dense(tiled, spec)
                emitted = [(form, _emit(form)) for form in paged_forms(tiled)]
            except Exception as problem:  # noqa: BLE001  (a refusal is one of the search's results)
                refusals.append(Refusal(graph.index, "solo", "main", problem))
                continue
            for form, source in emitted:
                keep(graph, "solo", tile, dense, source, rank, form.label)

    factors = tuple(config.split_k) if spec.kind in SPLIT_KINDS else ()
    for single in [p for p in plans if p.split_factor is None]:
        for factor in factors:
            combine = CombineTiling(split=factor, split_step=1, cols=min(128, single.dense.head_dim), n_threads=256)
            variant = f"split-kv={factor}"
            # the equal cut, and (where the kernel has it: a text of its own) the cut that spreads a request's
            # splits over the XCDs and skews the ranges between even and odd ones
            forms = [single.dense]
            if hasattr(single.dense, "skew") and not single.dense.skew and not single.dense.chunk_pages:
                forms.append(dataclasses.replace(single.dense, skew=30))
                # pages of many tokens: work items of a few pages each (one wave per kv head, the waves in step),
                # sized at launch so that one item lands on each compute unit -- requests of unlike lengths then
                # cost items in proportion, where a fixed split gives every request the same number of parts
                # (a token table has them too, of up to 2048 tokens.  us, bf16, 32 / 8 heads, the better of single kernel and fixed
                # split / these: 64 requests, 68237 tokens 66 / 41.6, 40 of up to 4000 91 / 66, 23 of 2682 40 / 28.8, 18 of 1056 16.2 / 14.9;
                # behind the fixed split for four requests and fewer, 3 of 2882 11.5 / 12.9, which keep it by the calibrated rule, and the single
                # kernel for short ones, 63 of 50 8.1 / 10.5)
                if (getattr(spec, "page_size", 1) == 1 or spec.page_size >= 16) and single.dense.query_rows <= 16 and factor == max(factors):
                    forms.append(dataclasses.replace(single.dense, chunk_pages=-1, lockstep=True, waves=spec.num_kv_heads,
                                                     n_threads=spec.num_kv_heads * 64))
            for d in forms:
                try:
                    source = _emit(build_split_decode(spec, d, factor, combine))
                except Exception as problem:  # noqa: BLE001
                    refusals.append(Refusal(single.graph_index, variant, "main", problem))
                    continue
                label = (f"S={factor} kv={d.kv_tile} q={d.query_rows} thr={d.n_threads} "
                         f"comb={combine.split_step}x{combine.cols}@{combine.n_threads}" + (f" skew={d.skew}" if getattr(d, "skew", 0) else "")
                         + (" chunked items" if getattr(d, "chunk_pages", 0) else ""))
                keep(single.graph, variant, single.tile, d, source, single.rank, label, factor, "derived split-K")
    return PlanSet(plans, graphs, config, refusals, seconds=time.perf_counter() - started)


# ================================================================================ workloads
def resolve_workloads(attention, workloads=None, tolerance=None):
    """``(factory, tolerance)`` where ``factory(keep)`` gives a generator function over ``keep``
    workloads (0: all), each ``(key, inputs, expected outputs)``.

    ``workloads`` may be: nothing -- a shipped operator then gets its captured axes from the
    registry, any other decode operator ``cl.workloads.paged_decode()``, and a prefill or MLA
    operator is an error; an object with ``factory(attention, keep=)`` (a ``cl.workloads`` spec);
    or a ready generator function, used as it is."""
    from ..dynamic import GATHER_TOLERANCE, OPERATORS
    from ..frontend.paged import PagedDecodeWorkloads

    tolerance = tolerance or GATHER_TOLERANCE
    program = attention.program
    if workloads is None:
        shipped = OPERATORS.get(program.name)
        if shipped is not None and shipped.matches(attention):
            return (lambda keep=0: shipped.keyed_workloads(keep=keep, dtype=program.dtype.torch)), tolerance
        if attention.is_mla or attention.is_prefill:
            raise SpecError(f"{program.name}: no captured {attention.kind} workloads; pass workloads=")
        workloads = PagedDecodeWorkloads()
    if hasattr(workloads, "factory"):
        return (lambda keep=0: workloads.factory(attention, keep=keep)), tolerance
    if callable(workloads):
        return (lambda keep=0: workloads), tolerance
    raise TypeError(f"workloads must be a cl.workloads spec or a factory, got {workloads!r}")


def crossing(low: int, low_ratio: float, high: int, high_ratio: float) -> int:
    """The first tile count in (``low``, ``high``] at which the split pair is the faster one, with its time over the
    single kernel's given at both ends and taken as a power of the tile count between them.  (Workloads of 16
    and 384 tiles used to put the threshold at 384: seven requests of up to 96 tiles ran the single kernel in
    31 us where the pair takes 17.)"""
    if low_ratio <= 1.0 or high_ratio >= 1.0:          # no change of sides between them: the middle
        at = math.sqrt(low * high)
    else:
        at = low * (high / low) ** (math.log(low_ratio) / (math.log(low_ratio) - math.log(high_ratio)))
    return min(high, max(low + 1, math.ceil(at)))


def split_threshold(tiles: dict, split_us: dict, single_us: dict) -> int:
    """The tile count from which the split pair runs, with the smallest geometric-mean time over the workloads
    timed (the lower one on a tie).  All thresholds between two neighbouring workloads share that mean; the one
    taken is where the two kernels' times cross between them."""
    from ..runtime.autotune import geomean

    keys = [k for k in tiles if k in split_us and k in single_us]
    seen = sorted({tiles[k] for k in keys})

    def cost(threshold):
        return geomean([(split_us if tiles[k] >= threshold else single_us)[k] for k in keys])

    def ratio(at):
        return geomean([split_us[k] / single_us[k] for k in keys if tiles[k] == at])

    best = min(sorted({*seen, 1, max(seen) + 1}), key=lambda t: (cost(t), t))
    if best in seen[1:]:
        below = seen[seen.index(best) - 1]
        best = crossing(below, ratio(below), best, ratio(best))
    return int(best)


def lone_request(kernel, inputs, expected, indptr_at):
    """A workload cut down to its longest request.  What an input's leading extent is called in the kernel's parameters
    says how: the batch (the outputs' leading extent), its row pointers, or, of the other vectors, the page table's
    length; caches stay whole, also where their pages are as many as the requests."""
    bounds = inputs[indptr_at].tolist()
    b = max(range(len(bounds) - 1), key=lambda r: bounds[r + 1] - bounds[r])
    declared = [p for p in kernel.params if p.role in ("input", "scalar")]
    batch = next(p for p in kernel.params if p.role == "output").shape[0]
    cut = []
    for i, (p, value) in enumerate(zip(declared, inputs)):
        if i == indptr_at:
            cut.append(value[b:b + 2] - value[b])
        elif p.role == "input" and p.shape[0] == batch:
            cut.append(value[b:b + 1].contiguous())
        elif p.role == "input" and len(p.shape) == 1:
            cut.append(value[bounds[b]:bounds[b + 1]].contiguous())
        else:
            cut.append(value)
    return cut, [t[b:b + 1].contiguous() for t in expected]


def few_requests(spec, compute_units: int) -> int:
    """The number of requests from which the single kernel has workgroups for a quarter of the compute units: one per
    request and kv head, or, for latent attention, per request and 16 query heads."""
    per_request = int(spec.num_kv_heads) if hasattr(spec, "num_kv_heads") else -(-int(spec.num_qo_heads) // 16)
    return compute_units // (4 * per_request) + 1


def calibrate_dispatch(pair, solo, factory, spec, fixed=None) -> dict:
    """When should a call run the split pair rather than the single kernel?

    Both are timed on every workload.  A workload is described by the kv tiles of its longest request
    (``indptr`` units x page size / kv tile, rounded up), and the rule is "split from ``min_tiles`` tiles on".
    What a split is worth also depends on whether the single kernel's workgroups fill the chip: for batches of
    fewer than ``few_requests`` requests (workgroups for less than a quarter of the compute units) the threshold is ``lone_tiles``,
    calibrated on each workload's longest request alone.  (With one threshold, taken from batches of 64 requests,
    three requests of up to 2882 tokens ran the single kernel in 26 us where the pair takes 11.)

    ``fixed``: the pair that gives every request the same number of parts, where ``pair`` cuts the table into items.  Batches so small
    that its parts are no more workgroups than compute units run it for requests of ``from_tiles`` tiles on and below ``until_tiles``
    a request (three at most): an item's ids pass through LDS and its partials are found through the row pointers, which costs such a
    call more than the even cut saves.  us, fixed / items, bf16, 32 / 8 heads: 1 x 500 tokens 6.4 / 8.2, 1 x 3000 10.1 / 9.8, 1 x 9000 18.5 / 14.5,
    2 x 3000 10.4 / 11.0, 2 x 9000 19.8 / 18.3, 3 x 3000 11.5 / 13.1, 4 x 6000 21.3 / 22.0, 4 x 9000 33.1 / 32.7; 5 x 500 9.8 / 8.8, 5 x 3000 19.5 / 16.6."""
    import dataclasses

    from ..core.target import current_target
    from ..runtime.autotune import benchmark_over_workloads, geomean, param_index

    pair, solo = dataclasses.replace(pair, latency_us={}), dataclasses.replace(solo, latency_us={})
    indptr_at = param_index(solo.kernel, f"PlaceHolder_{spec.indptr_input}")
    tokens_per_unit, kv_tile = int(getattr(spec, "page_size", 1)), int(pair.tiling.kv_tile)
    longest, requests = {}, {}

    def observed():
        for key, inputs, expected in factory(0)():
            bounds = inputs[indptr_at].tolist()
            units = max(hi - lo for lo, hi in zip(bounds, bounds[1:]))
            longest[key], requests[key] = math.ceil(units * tokens_per_unit / kv_tile), len(bounds) - 1
            yield key, inputs, expected

    def alone():
        for key, inputs, expected in factory(0)():
            yield (key, *lone_request(solo.kernel, inputs, expected, indptr_at))

    benchmark_over_workloads([pair, solo], observed, ramp_seconds=0.2)
    min_tiles = split_threshold(longest, pair.latency_us, solo.latency_us)
    units = current_target().arch.compute_units
    few = few_requests(spec, units)
    lone_pair, lone_solo, lone_fixed = (c and dataclasses.replace(c, latency_us={}) for c in (pair, solo, fixed))
    benchmark_over_workloads([c for c in (lone_pair, lone_solo, lone_fixed) if c], alone, ramp_seconds=0.0)
    lone_tiles = split_threshold(longest, lone_pair.latency_us, lone_solo.latency_us)
    keys = [k for k in longest if k in pair.latency_us and k in solo.latency_us]

    few_parts = {}
    if fixed and units >= fixed.split * int(spec.num_kv_heads):
        few_parts = {"requests": units // (fixed.split * int(spec.num_kv_heads)),
                     "until_tiles": split_threshold(longest, lone_pair.latency_us, lone_fixed.latency_us), "label": fixed.label}

    def splits(key):
        return longest[key] >= (lone_tiles if requests[key] < few else min_tiles)

    per_workload = {k: (pair if splits(k) else solo).latency_us[k] for k in keys}
    return {
        "rule": "run the split pair when the longest request has at least min_tiles KV tiles (lone_tiles for batches of fewer "
                "than few_requests requests; indptr units x page_size tokens / kv_tile), else the single kernel",
        "min_tiles": min_tiles, "lone_tiles": lone_tiles, "few_requests": few, "kv_tile": kv_tile,
        "page_size": tokens_per_unit, "indptr_index": indptr_at,
        "split_label": pair.label, "single_label": solo.label,
        "n_workloads": len(keys), "split_runs": sum(map(splits, keys)),
        "geomean_us": {"hybrid": geomean(list(per_workload.values())), "split": geomean([pair.latency_us[k] for k in keys]),
                       "single": geomean([solo.latency_us[k] for k in keys])},
        "per_workload_us": per_workload, **({"fixed": few_parts} if few_parts else {}),
    }


def pick_token_threshold(winner_us: dict, other_us: dict, tokens: dict):
    """``(threshold, geomean)`` of the rule "the other kernel when a call has at most ``threshold``
    query tokens, else the winner" with the smallest geometric-mean time over the workloads both
    were timed on; ``threshold`` is one of the workloads' token counts, or None when the winner
    alone is at least as good."""
    from ..runtime.autotune import geomean

    keys = [k for k in winner_us if k in other_us and k in tokens]
    if not keys:
        return None, float("inf")

    def cost(threshold):
        return geomean([other_us[k] if threshold is not None and tokens[k] <= threshold else winner_us[k] for k in keys])

    best = min([None] + sorted({tokens[k] for k in keys}), key=lambda t: (cost(t), -1 if t is None else t))
    return best, cost(best)


def calibrate_token_dispatch(winner, others, factory, query_at, *, gain: float = 0.01):
    """Prefill layers: should a call with few query tokens run another kernel than the winner?

    Every candidate was timed on every workload.  A workload is described by its packed query
    tokens (the leading extent of Q, known on the host without a look at the row pointers); the
    rule is "the other kernel up to ``max_tokens`` tokens", with the kernel and the threshold that
    give the smallest geometric-mean time -- kept only when that beats the winner alone by more
    than ``gain``: a kernel built for 128-row items pays for them on a call of a few rows."""
    from ..runtime.autotune import geomean

    tokens = {key: int(inputs[query_at].shape[0]) for key, inputs, _ in factory(0)()}
    alone = geomean([winner.latency_us[k] for k in winner.latency_us if k in tokens])
    chosen = None
    for other in others:
        threshold, us = pick_token_threshold(winner.latency_us, other.latency_us, tokens)
        if threshold is not None and us < (1.0 - gain) * alone and (chosen is None or us < chosen[2]):
            chosen = (other, threshold, us)
    if chosen is None:
        return None, None
    other, threshold, us = chosen
    keys = [k for k in winner.latency_us if k in other.latency_us and k in tokens]
    return {
        "rule": "run the few-token kernel when the call has at most max_tokens packed query tokens, else the winner",
        "by": "query_tokens", "max_tokens": int(threshold), "few_label": other.label, "many_label": winner.label,
        "n_workloads": len(keys), "few_runs": sum(tokens[k] <= threshold for k in keys),
        "geomean_us": {"hybrid": us, "many": alone, "few": geomean([other.latency_us[k] for k in keys])},
        "per_workload_us": {k: (other if tokens[k] <= threshold else winner).latency_us[k] for k in keys},
    }, other


# ================================================================================ the report
class DynamicReport:
    """What the search over a paged operator found: its plans, one ``WorkloadCandidate`` per plan
    with what was checked and measured, the errors met, stage times, and the dispatch
    calibration when one was made."""

    def __init__(self, plans, candidates, errors, *, workloads: int, timings: dict, expected=None, tuned=None,
                 dispatch=None):
        self.plans, self.candidates, self.errors = plans, list(candidates), list(errors)
        self.n_workloads, self.timings = workloads, dict(timings)
        self.expected, self.tuned, self.dispatch = expected, tuned, dispatch

    correct = property(lambda self: [c for c in self.candidates if c.correct])
    failures = property(lambda self: [c for c in self.candidates if not c.correct])
    timed = property(lambda self: [c for c in self.candidates if c.correct and c.latency_us])

    def best(self, split: Optional[bool] = None):
        """The fastest eligible candidate; ``split=True`` / ``False`` restricts the choice to the
        split pairs / the single kernels."""
        from ..runtime.autotune import pick_best, rank

        field_ = [c for c in self.timed if c.eligible and (split is None or bool(c.split) == bool(split))]
        return pick_best(rank(field_)) if field_ else None

    def histogram(self) -> dict:
        """Error headline -> how many candidates met it, most frequent first."""
        def headline(error):
            first = (str(error).strip().splitlines() or [""])[0]
            return f"{type(error).__name__}: {first[:100]}"

        return dict(Counter(headline(error) for _, error in self.errors).most_common())

    def summary(self) -> str:
        took = self.timings.get
        lines = [("superoptimize", f"{len(self.plans.graphs)} dense graph(s)", took("superoptimize")),
                 ("schedule", self.plans.summary().replace("\n  ", "  "), took("schedule")),
                 ("validate", f"{len(self.correct)} of {len(self.candidates)} correct over {self.n_workloads} workloads",
                  took("validate"))]
        lines += [("", f"  {count}x {what}", None) for what, count in self.histogram().items()]
        winner = self.best()
        if winner is not None:
            lines.append(("benchmark", f"best {winner.geomean_us:.2f} us geomean  {winner.label}", took("benchmark")))
        if self.dispatch and self.dispatch.get("by") == "query_tokens":
            d, us = self.dispatch, self.dispatch["geomean_us"]
            lines.append(("dispatch", f"{d['few_label']} up to {d['max_tokens']} query tokens: hybrid {us['hybrid']:.2f} us "
                          f"vs {us['many']:.2f} alone over {d['n_workloads']} workloads", took("dispatch")))
        elif self.dispatch:
            d, us = self.dispatch, self.dispatch["geomean_us"]
            lines.append(("dispatch", f"split when >= {d['min_tiles']} KV tiles of {d['kv_tile']}: hybrid {us['hybrid']:.2f} us "
                          f"vs split {us['split']:.2f} vs single {us['single']:.2f} over {d['n_workloads']} workloads",
                          took("dispatch")))
        return "\n".join(f"{stage:<14}{text}" + (f"  {seconds:.2f} s" if seconds is not None else "")
                         for stage, text, seconds in lines)

    __str__ = summary

    def table(self, top: int = 10) -> str:
        from ..runtime.autotune import format_ranking

        return format_ranking(self.timed, self.failures)

    def to_dict(self) -> dict:
        return {"candidates": len(self.candidates), "correct": len(self.correct), "refused": len(self.plans.refused),
                "failures": self.histogram(), "timings_s": self.timings,
                "latency_us": {c.label: c.geomean_us for c in self.timed}, "dispatch": self.dispatch}


# ================================================================================ the kernel
class PagedKernel(Kernel):
    """``kernel(*inputs)`` in the traced signature's order gives ``out`` or ``(out, lse)``.

    Outputs are allocated per call; split partials belong to the compiled kernel.  ``dispatch`` is
    the split / single calibration (threshold and times), kept and saved with both kernels'
    sources beside the main one.  A plain call runs the kernel the search ranked best (what a call
    of the reference's object does).  A caller that knows its longest request on the host -- a
    serving loop does -- can pass ``longest=<its length in page-table units>``: the call then runs
    the split pair or the single kernel by the calibrated rule, without reading anything back from
    the device."""

    def __init__(self, attention, spec, source: str, compiled=None, *, dispatch=None, dispatch_sources=None, **kernel_kw):
        self.attention, self.spec = attention, spec
        self.dispatch, self.dispatch_sources = dispatch, dict(dispatch_sources or {})
        stage = Stage("main", source, [], [], kernel_kw.get("label", ""), kernel_kw.get("latency_us"))
        super().__init__([stage], name=attention.program.name, input_names=[p.name for p in attention.inputs],
                         input_shapes=[], **kernel_kw)
        self._compiled, self._argument_order = compiled, None
        self._by_role = {}               # "split" / "single" -> (compiled kernel, argument order), built on first use
        self._plans = {}                 # role (None: the main kernel) -> native call plan, or False
        kept = attention.inputs
        self._n_kept, self._query_at = len(kept), next(i for i, p in enumerate(kept) if p.name == attention.query.name)

    # ---- persistence
    def save(self, path):
        folder = super().save(path)
        document = json.loads((folder / "kernel.json").read_text())
        (folder / PROGRAM_FILE).write_text(json.dumps(self.attention.program.to_doc(), indent=1))
        document["paged"] = PROGRAM_FILE
        if self.dispatch:
            files = {role: f"dispatch.{role}.hip" for role in self.dispatch_sources}
            for role, name in files.items():
                (folder / name).write_text(self.dispatch_sources[role], encoding="utf-8")
            (folder / DISPATCH_FILE).write_text(json.dumps({**self.dispatch, "files": files}, indent=1))
            document["dispatch"] = DISPATCH_FILE
        (folder / "kernel.json").write_text(json.dumps(document, indent=1, default=str))
        return folder

    @classmethod
    def _load(cls, folder, document) -> "PagedKernel":
        from ..frontend.paged import PagedProgram

        program_file = folder / document["paged"]
        if program_file.suffix != ".json":
            raise ValueError(f"{folder}: the paged program is stored as {program_file.name!r}; only the JSON form "
                             "is read (a pickle would run code from the directory)")
        attention = PagedProgram.from_doc(json.loads(program_file.read_text())).attention()
        dispatch, sources = None, {}
        if document.get("dispatch"):
            dispatch = json.loads((folder / document["dispatch"]).read_text())
            sources = {role: (folder / name).read_text() for role, name in dispatch.pop("files", {}).items()}
        return cls(attention, attention.paging_spec(), (folder / document["stages"][0]["file"]).read_text(),
                   label=document["label"], variant=document["variant"], latency_us=document["latency_us"],
                   dispatch=dispatch, dispatch_sources=sources,
                   meta={**(document.get("meta") or {}), "loaded_from": str(folder)})

    # ---- running
    def compile(self) -> "PagedKernel":
        if self._compiled is None:
            from ..runtime.autotune import _compiled

            self._compiled = _compiled(self.source)
        return self

    def _order_for(self, compiled) -> list:
        """The traced arguments in the order ``compiled`` takes them: tensors where their
        ``PlaceHolder_<NAME>`` sits, scalars in the slots left over, in signature order."""
        from ..runtime.autotune import param_index

        kept = self.attention.inputs
        order = [None] * len(kept)
        for p in kept:
            if not p.is_scalar:
                order[param_index(compiled, f"PlaceHolder_{p.kernel_name}")] = p
        scalars = (p for p in kept if p.is_scalar)
        return [p if p is not None else next(scalars) for p in order]

    def _order(self) -> list:
        if self._argument_order is None:
            self._argument_order = self._order_for(self._compiled)
        return self._argument_order

    def dispatch_role(self, longest: int, requests: int | None = None) -> str:
        """``"split"`` or ``"single"`` for a batch of ``requests`` requests whose longest spans ``longest``
        page-table units, by the calibrated rule (kv tiles of the longest request against ``min_tiles``, or
        ``lone_tiles`` where the requests are too few to fill the chip); ``"fixed"`` where the split pair cuts the table into
        items and a pair of equal parts was kept beside it for batches as small as this one."""
        rule, sources = self.dispatch, self.dispatch_sources
        if not rule or "split" not in sources or "single" not in sources:
            raise CleaveError(f"{self.name}: no split / single calibration was made (or saved) for this operator")
        few = requests is not None and requests < rule.get("few_requests", 0)
        # (tiles of the longest request, rounded up, against a whole number of them)
        tokens, kv_tile = int(longest) * rule["page_size"], rule["kv_tile"]
        if tokens <= (rule["lone_tiles" if few else "min_tiles"] - 1) * kv_tile:
            return "single"
        if requests is not None and "fixed" in sources and "fixed" in rule:
            parts = rule["fixed"]
            if requests <= parts["requests"] and tokens <= (parts["until_tiles"] * min(requests, max(1, parts["requests"] - 1)) - 1) * kv_tile:
                return "fixed"
        return "split"

    def token_role(self, tokens: int):
        """``"few"`` or ``"many"`` for a call with ``tokens`` packed query tokens, by the rule
        calibrated for a prefill layer; None when no such rule was made (or saved)."""
        rule, sources = self.dispatch, self.dispatch_sources
        if not rule or rule.get("by") != "query_tokens" or "few" not in sources or "many" not in sources:
            return None
        return "few" if int(tokens) <= rule["max_tokens"] else "many"

    def _dispatched(self, longest: int, role=None):
        role = role or self.dispatch_role(longest)
        if role not in self._by_role:
            from ..runtime.autotune import _compiled

            compiled = _compiled(self.dispatch_sources[role])
            self._by_role[role] = (compiled, self._order_for(compiled))
        return self._by_role[role]

    def _bind(self, positional, named) -> dict:
        """name -> value for every parameter of the traced signature.  Positional calls may give
        the full signature or only the inputs the kernel reads."""
        signature, kept = self.attention.program.params, self.attention.inputs
        listing = ", ".join(p.name for p in signature)
        if positional and named:
            raise TypeError("pass inputs either positionally or by name, not both")
        if named:
            unknown = sorted(set(named) - {p.name for p in signature})
            if unknown:
                raise TypeError(f"{self.name}: unexpected inputs {unknown}")
            bound = {p.name: named.get(p.name) for p in signature}
        else:
            matching = [ps for ps in (signature, kept) if len(ps) == len(positional)]
            if not matching:
                raise TypeError(f"{self.name}: expected inputs ({listing})")
            bound = {p.name: None for p in signature}
            bound.update(zip((p.name for p in matching[0]), positional))
        for p in signature:
            given = bound[p.name] is not None
            if p in kept and not given:
                raise TypeError(f"{self.name}: missing input {p.name!r}")
            if p not in kept and given:
                raise ValueError(f"{self.name}: page_size=1 reads no {p.name}; pass None")
        return bound

    def _native_plan(self, role):
        """The native call plan of the kernel that ``role`` names: arguments in the order of the inputs it reads."""
        from ..runtime.dispatch import chain_plan

        if role is None:
            self.compile()
            compiled, order = self._compiled, self._order()
        else:
            compiled, order = self._dispatched(0, role=role)
        kept = list(self.attention.inputs)
        declared = [p for p in compiled.params if p.role in ("input", "scalar")]
        if compiled.out_idx is not None or len(declared) != len(order):
            return False
        position = {id(p): i for i, p in enumerate(kept)}
        sources = {d.name: ("arg", position[id(p)]) for d, p in zip(declared, order)}
        by_position = {position[id(p)]: d for d, p in zip(declared, order)}
        return chain_plan([(compiled, sources)], arguments=[(by_position[i], None) for i in range(len(kept))], as_tuple=True) or False

    def __call__(self, *positional, longest=None, **named):
        role, plan = None, False
        if not named and len(positional) == self._n_kept and positional[self._query_at] is not None:
            # (a token rule, where one was made, decides before `longest` does)
            role = self.token_role(positional[self._query_at].shape[0])
            if role is None and longest is not None:
                role = self.dispatch_role(longest, positional[self._query_at].shape[0])
            plan = self._plans.get(role)
            if plan:
                done = plan(*positional)
                if done is not NotImplemented:
                    return done
        done = self._checked_call(positional, longest, named)
        if plan is None:                 # a first call of this kernel went through: later ones take the native plan
            from ..runtime.dispatch import plan_or_false

            self._plans[role] = plan_or_false(lambda: self._native_plan(role))
        return done

    def _checked_call(self, positional, longest, named):
        import torch

        bound = self._bind(positional, named)
        by_tokens = self.token_role(bound[self.attention.query.name].shape[0])
        if by_tokens is not None:
            compiled, order = self._dispatched(0, role=by_tokens)
        elif longest is None:
            self.compile()
            compiled, order = self._compiled, self._order()
        else:
            compiled, order = self._dispatched(longest, role=self.dispatch_role(longest, bound[self.attention.query.name].shape[0]))
        sizes = {}
        for p in self.attention.inputs:
            if not p.is_scalar:
                for d, n in zip(p.spec.dims, bound[p.name].shape):
                    if hasattr(d, "name"):
                        sizes.setdefault(d.name, int(n))
        device = bound[self.attention.query.name].device
        outputs = [torch.empty([sizes[d.name] if hasattr(d, "name") else int(d) for d in dims], dtype=dtype.torch,
                               device=device)
                   for dims, dtype in zip(self.attention.output_dims(), self.attention.output_dtypes())]
        compiled(*[bound[p.name] for p in order], *outputs)
        return outputs[0] if len(outputs) == 1 else tuple(outputs)


# ================================================================================ the search
class _Search:
    def __init__(self, note):
        self.note = note
        self.seconds = {}

    @contextlib.contextmanager
    def stage(self, name):
        started = time.perf_counter()
        try:
            yield
        finally:
            self.seconds[name] = time.perf_counter() - started


def compile_dynamic(fn, *, dtype=None, preset="default", superopt=None, schedule=None, eval=None,  # noqa: A002
                    split=None, hints=None, workloads=None, tolerance=None, max_workloads: int = 6,
                    filter_before_topk: bool = False, reference: bool = True, dispatch: bool = True,
                    progress: Optional[Callable] = None, **others) -> PagedKernel:
    """Search, check and time a paged operator; see the module text for the stages.

    ``split``: the kv dimension to also build split-KV pairs over, e.g. ``cl.Split("kv_len", (4, 8))``
    (decode layers only; elsewhere it is noted and dropped).  Every candidate is checked on every
    workload and timed on ``max_workloads`` of them.  ``dispatch``: when both a split pair and a
    single kernel are correct, calibrate which one a workload should run.  ``progress(stage,
    value)`` is called after each stage."""
    from ..dynamic.paging import SPLIT_KINDS
    from ..frontend.paged import trace_paged
    from ..runtime.autotune import WorkloadCandidate, benchmark_over_workloads, compile_and_validate_over_workloads, pick_best, rank

    others.pop("cache_kernels", None)
    if others:
        raise TypeError(f"compile(): unexpected options for a paged program: {sorted(others)}")
    search = _Search(progress or (lambda stage, value: None))
    program = trace_paged(fn, dtype, hints=hints)
    attention = program.attention()
    spec = attention.paging_spec()
    search.note("spec", spec)
    body = attention.dense_body()

    split = (program.split or None) if split is None else split
    if split and spec.kind not in SPLIT_KINDS:
        search.note("split", f"split-KV is not built for the {spec.kind!r} layer; searching without it")
        split = False
    so, sc, ev = resolve_configs(body, preset=preset, superopt=superopt, schedule=schedule, eval=eval, split=split)
    if split is False:
        sc = sc.replace(split_k=())

    with search.stage("superoptimize"):
        graphs = superoptimize(body, so.replace(split=()))
    search.note("superoptimize", graphs)
    with search.stage("schedule"):
        plans = schedule_paged(graphs, spec, sc, filter_before_topk=filter_before_topk)
    search.note("schedule", plans)
    if not plans:
        raise CleaveError(f"{program.name}: the access layer refused every tiling\n{plans.summary()}")

    factory, tolerance = resolve_workloads(attention, workloads, tolerance or ev.tolerance)
    plan_of = {}
    for plan in plans:
        candidate = WorkloadCandidate(label=plan.label, source=plan.source, origin=plan.origin, tiling=plan.dense,
                                      split=plan.split_factor)
        plan_of[id(candidate)] = (candidate, plan)
    candidates = [c for c, _ in plan_of.values()]
    passed, errors = [], []
    with search.stage("validate"):
        compile_and_validate_over_workloads(candidates, factory(0), passed, errors, tolerance=tolerance)
    with search.stage("benchmark"):
        if any(c.eligible for c in passed):
            benchmark_over_workloads(passed, factory(max_workloads), ramp_seconds=0.3)
    report = DynamicReport(plans, candidates, errors, workloads=max((c.checked for c in candidates), default=0),
                           timings=search.seconds)
    winner = report.best()
    if winner is None:
        search.note("evaluate", report)
        failure = CleaveError(f"{program.name}: no searched candidate is correct over its workloads")
        failure.report = report
        raise failure

    pair, single = report.best(split=True), report.best(split=False)
    both = {}
    if dispatch and pair is not None and single is not None:
        with search.stage("dispatch"):
            # (pages of many tokens go by the pair and the single kernel alone: an item of them has its ids in registers)
            equal = [c for c in report.timed if c.eligible and c.split and not getattr(c.tiling, "chunk_pages", 0)]
            items = getattr(pair.tiling, "chunk_pages", 0) and getattr(spec, "page_size", 1) == 1 and hasattr(spec, "num_kv_heads")
            fixed = pick_best(rank(equal)) if items and equal else None
            report.dispatch = calibrate_dispatch(pair, single, factory, spec, fixed)
        report.timings["dispatch"] = search.seconds["dispatch"]
        both = {"split": pair.source, "single": single.source, **({"fixed": fixed.source} if "fixed" in report.dispatch else {})}
    elif dispatch and attention.is_prefill:
        from ..runtime.autotune import param_index

        others = [c for c in report.timed if c.eligible and c is not winner]
        if others:
            with search.stage("dispatch"):
                query_name = spec.query_inputs[0] if hasattr(spec, "query_inputs") else spec.query_input
                query_at = param_index(winner.kernel, f"PlaceHolder_{query_name}")
                report.dispatch, few = calibrate_token_dispatch(winner, others, factory, query_at)
            report.timings["dispatch"] = search.seconds["dispatch"]
            if report.dispatch:
                both = {"few": few.source, "many": winner.source}
    search.note("evaluate", report)
    for c in candidates:
        if c is not winner:
            c.kernel = None                   # only the winner keeps its module loaded
    plan = plan_of[id(winner)][1]
    return PagedKernel(attention, spec, winner.source, winner.kernel, label=winner.label, variant=plan.variant,
                       latency_us=winner.geomean_us, report=report, plans=[plan], meta={}, dispatch=report.dispatch,
                       dispatch_sources=both)
