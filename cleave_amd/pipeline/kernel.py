"""What ``compile`` returns: a ``Kernel`` that is called like the traced function.

A kernel is a short chain of *stages*.  A solo variant has one; a split variant has the partial
stage followed by its combine, the partial's outputs feeding the combine's placeholders.  Each
stage carries its HIP source and the wiring of its placeholders, which is all that is needed to
run it again later: ``save`` writes ``kernel.json`` (format 1), one source file per stage
(``kernel.hip``, or ``kernel_<i>_<role>.hip``) and, when the kernel came out of a search, the
search's ``report.json``; ``load`` reads them back and recompiles on first use without searching.
The directory layout and the format number are the reference's
(``python/cleave/pipeline/kernel.py:113-157``); the sources are HIP instead of TileLang.
"""

from __future__ import annotations

import json
import math
from dataclasses import dataclass, field
from pathlib import Path
from typing import Any

FORMAT = 1
SOURCE_SUFFIX = ".hip"
FROM_PROGRAM, FROM_STAGE = "input", "stage"


@dataclass
class Param:
    """A stage placeholder and where its tensor comes from: the program's input number ``index``
    (``source == "input"``) or output number ``index`` of the stage before (``"stage"``)."""
    name: str
    source: str
    index: int
    shape: tuple

    def to_json(self) -> dict:
        return {"name": self.name, "source": self.source, "index": self.index, "shape": list(self.shape)}

    @classmethod
    def from_json(cls, doc: dict) -> "Param":
        return cls(doc["name"], doc["source"], int(doc["index"]), tuple(doc["shape"]))


@dataclass
class Stage:
    role: str                                  # "main", "partial" or "combine"
    source: str = field(repr=False)
    out_idx: list = field(default_factory=list)
    params: list = field(default_factory=list)
    label: str = ""
    latency_us: float | None = None
    built: Any = field(default=None, repr=False, compare=False)   # pipeline.build.BuiltKernel, when known

    def file_name(self, position: int, alone: bool) -> str:
        return ("kernel" if alone else f"kernel_{position}_{self.role}") + SOURCE_SUFFIX

    def to_json(self, file_name: str) -> dict:
        doc = {"role": self.role, "file": file_name, "label": self.label, "latency_us": self.latency_us,
               "out_idx": list(self.out_idx), "params": [p.to_json() for p in self.params]}
        if self.built is not None:
            doc["kernel"] = self.built.to_dict()
        return doc

    @classmethod
    def from_json(cls, doc: dict, folder: Path) -> "Stage":
        from .build import BuiltKernel

        text = (folder / doc["file"]).read_text()
        built = BuiltKernel.from_dict(doc["kernel"], text) if "kernel" in doc else None
        return cls(doc["role"], text, list(doc["out_idx"]), [Param.from_json(p) for p in doc["params"]],
                   doc.get("label", ""), doc.get("latency_us"), built)


def _as_shape(tensor, shape):
    """``tensor`` viewed as ``shape`` when the element counts agree (unit and batch axes are laid
    out differently between a program and its stages); otherwise ``tensor`` itself."""
    shape = tuple(shape)
    if tuple(tensor.shape) != shape and math.prod(tensor.shape) == math.prod(shape):
        return tensor.reshape(shape)
    return tensor


class Kernel:
    """Callable result of a compile.  ``unrunnable`` holds the reason when the stages could not be
    wired to the program's inputs (the sources and timings are still there to inspect)."""

    def __init__(self, stages, *, name: str, input_names, input_shapes, output_shapes=None, variant: str = "solo",
                 label: str = "", latency_us=None, report=None, plans=(), unrunnable=None, meta=None):
        self.name, self.variant, self.label = name, variant, label
        self.stages = list(stages)
        self.plans = list(plans)
        self.input_names = list(input_names)
        self.input_shapes = [tuple(shape) for shape in input_shapes]
        self.output_shapes = [tuple(shape) for shape in output_shapes] if output_shapes is not None else None
        self.latency_us = latency_us
        self.report = report
        self.unrunnable = unrunnable
        self.meta = dict(meta or {})
        self._callables = None
        self._plan = None                # the native call plan over all stages, made on the first call

    def __repr__(self):
        timing = f"{self.latency_us:.2f} us" if self.latency_us is not None else "?"
        return f"Kernel({self.name!r}, {self.variant}, {timing}, {self.label!r})"

    @property
    def source(self) -> str:
        """The one stage's source, or all of them under ``// ---- stage i: role ----`` headers."""
        if len(self.stages) == 1:
            return self.stages[0].source
        return "\n\n".join(f"// ---- stage {n}: {stage.role} ----\n{stage.source}" for n, stage in enumerate(self.stages))

    @property
    def plan(self):
        return self.plans[0] if len(self.plans) == 1 else tuple(self.plans)

    @property
    def kernels(self) -> list:
        return [stage.built for stage in self.stages]

    # -- running ---------------------------------------------------------------------------------
    def compile(self) -> "Kernel":
        """Compile every stage's source with hiprtc (no search).  ``__call__`` does it on demand."""
        if self.unrunnable:
            raise NotImplementedError(self.unrunnable)
        if self._callables is None:
            from ..runtime.compile import _compile, _load_main_kernel_from_code

            self._callables = [_compile(_load_main_kernel_from_code(stage.source), stage.out_idx)
                               for stage in self.stages]
        return self

    def _arguments(self, positional, named) -> list:
        if positional and named:
            raise TypeError("pass inputs either positionally or by name, not both")
        if named:
            wanted = set(self.input_names)
            absent = [n for n in self.input_names if n not in named]
            surplus = sorted(set(named) - wanted)
            if absent or surplus:
                raise TypeError(f"{self.name}: missing inputs {absent}, unexpected {surplus}")
            positional = tuple(named[n] for n in self.input_names)
        if len(positional) != len(self.input_names):
            raise TypeError(f"{self.name}: expected {len(self.input_names)} inputs ({', '.join(self.input_names)}), "
                            f"got {len(positional)}")
        for name, shape, tensor in zip(self.input_names, self.input_shapes, positional):
            if tuple(tensor.shape) != shape:
                raise ValueError(f"{self.name}: input {name!r} has shape {tuple(tensor.shape)}, expected {shape}")
        return list(positional)

    def _native_plan(self):
        """One native plan for the whole chain (the partials between stages are scratch of a call), or
        False where a stage's shapes are not all known or do not line up."""
        from types import SimpleNamespace

        from ..runtime.dispatch import chain_plan

        self.compile()
        dtype_of: dict = {}
        stages = []
        for stage, kernel in zip(self.stages, self._callables):
            shape_of = {p.name: tuple(p.shape) for p in kernel.params}
            sources = {}
            for p in stage.params:
                declared, origin_shape = shape_of.get(p.name), None
                if declared is None or not all(isinstance(e, int) for e in declared):
                    return False
                if p.source == FROM_PROGRAM:
                    if not 0 <= p.index < len(self.input_shapes):
                        return False
                    origin_shape = self.input_shapes[p.index]
                    dtype_of.setdefault(p.index, next(q.dtype for q in kernel.params if q.name == p.name))
                elif not stages or p.index >= sum(q.role == "output" for q in stages[-1][0].params):
                    return False
                if origin_shape is not None and math.prod(origin_shape) != math.prod(declared):
                    return False
                sources[p.name] = ("arg" if p.source == FROM_PROGRAM else "stage", p.index)
            if kernel.dyn_dims or any(p.role in ("input", "scalar") and p.name not in sources for p in kernel.params):
                return False
            stages.append((kernel, sources))
        if set(dtype_of) != set(range(len(self.input_shapes))):
            return False
        arguments = [(SimpleNamespace(role="input", dtype=dtype_of[i]), shape) for i, shape in enumerate(self.input_shapes)]
        return chain_plan(stages, arguments=arguments, output_shapes=self.output_shapes, as_tuple=True) or False

    def __call__(self, *positional, **named):
        if self._plan and not named:
            done = self._plan(*positional)
            if done is not NotImplemented:
                return done
        done = self._checked_call(positional, named)
        if self._plan is None:           # a first call went through: later ones take the native plan
            from ..runtime.dispatch import plan_or_false

            self._plan = plan_or_false(self._native_plan)
        return done

    def _checked_call(self, positional, named):
        from ..runtime.reference import order_inputs_for_kernel

        program_inputs = self._arguments(positional, named)
        self.compile()
        carried: list = []                   # outputs of the stage before
        for stage, run in zip(self.stages, self._callables):
            by_placeholder = {}
            for p in stage.params:
                origin = program_inputs if p.source == FROM_PROGRAM else carried
                by_placeholder[p.name] = _as_shape(origin[p.index], p.shape)
            produced = run(*order_inputs_for_kernel(by_placeholder, run))
            carried = list(produced) if isinstance(produced, (tuple, list)) else [produced]
        if self.output_shapes is not None:
            carried = [_as_shape(t, shape) for t, shape in zip(carried, self.output_shapes)]
        return carried[0] if len(carried) == 1 else tuple(carried)

    # -- persistence ---------------------------------------------------------------------------
    def save(self, path) -> Path:
        folder = Path(path).expanduser()
        folder.mkdir(parents=True, exist_ok=True)
        alone = len(self.stages) == 1
        stage_docs = []
        for position, stage in enumerate(self.stages):
            file_name = stage.file_name(position, alone)
            (folder / file_name).write_text(stage.source)
            stage_docs.append(stage.to_json(file_name))
        document = {"format": FORMAT, "name": self.name, "variant": self.variant, "label": self.label,
                    "latency_us": self.latency_us, "unrunnable": self.unrunnable,
                    "input_names": self.input_names, "input_shapes": self.input_shapes,
                    "output_shapes": self.output_shapes, "meta": self.meta, "stages": stage_docs}
        (folder / "kernel.json").write_text(json.dumps(document, indent=1, default=str))
        if hasattr(self.report, "to_dict"):
            (folder / "report.json").write_text(json.dumps(self.report.to_dict(), indent=1, default=str))
        return folder


def load(path) -> Kernel:
    """The kernel saved under ``path`` (a paged operator's directory gives a ``PagedKernel``)."""
    folder = Path(path).expanduser()
    document = json.loads((folder / "kernel.json").read_text())
    if document.get("format") != FORMAT:
        raise ValueError(f"{folder}: unsupported kernel format {document.get('format')!r}")
    if document.get("paged"):
        from .dynamic import PagedKernel

        return PagedKernel._load(folder, document)
    meta = dict(document.get("meta") or {})
    meta["loaded_from"] = str(folder)
    return Kernel([Stage.from_json(doc, folder) for doc in document["stages"]], name=document["name"],
                  input_names=document["input_names"], input_shapes=document["input_shapes"],
                  output_shapes=document.get("output_shapes"), variant=document["variant"], label=document["label"],
                  latency_us=document["latency_us"], unrunnable=document.get("unrunnable"), meta=meta)


# --------------------------------------------------------------------------- wiring stages
def _extent(node) -> tuple:
    return tuple(map(int, node.get_shape(0)))


def stages_for(plans_and_results, program):
    """``(stages, problem)`` from ``[(plan, run result[, BuiltKernel])]`` in execution order.

    Wiring: a main or partial stage reads the program's inputs through the plan's input binding.
    A combine stage reads the outputs of the stage before it, placeholder i from output i; a
    placeholder beyond those that carries the name of a program input reads that input (the LoRA
    combine reads the up factor).  ``problem`` is the first reason the chain cannot be run."""
    from ..runtime.reference import graph_out_indices, output_order, placeholder_order

    stages = []
    problems = []
    input_slot: dict = {}          # placeholder name -> program input number, from the last main / partial stage
    upstream: list = []            # output shapes of the stage before
    for plan, result, *extra in plans_and_results:
        built = extra[0] if extra else None
        graph = plan.tile.flat_graph
        wiring = []
        if plan.role == "combine":
            for position, holder in enumerate(placeholder_order(graph)):
                shape = _extent(holder)
                if position < len(upstream):
                    if math.prod(upstream[position]) != math.prod(shape):
                        problems.append(f"{plan.label}: combine inputs do not line up with the partial kernel's outputs")
                    wiring.append(Param(holder.name, FROM_STAGE, position, shape))
                elif holder.name in input_slot:
                    wiring.append(Param(holder.name, FROM_PROGRAM, input_slot[holder.name], shape))
                else:
                    problems.append(f"{plan.label}: combine inputs do not line up with the partial kernel's outputs")
                    wiring.append(Param(holder.name, FROM_STAGE, position, shape))
        else:
            if plan.inputs is None:
                problems.append(f"{plan.label}: could not bind kernel placeholders to the Program inputs")
                input_slot = {}
            else:
                input_slot = {name: number for number, name in enumerate(plan.inputs)}
            wiring = [Param(h.name, FROM_PROGRAM, input_slot.get(h.name, -1), _extent(h)) for h in placeholder_order(graph)]
        upstream = [_extent(out) for out in output_order(graph)]
        latency_us = result.latency_ms * 1e3 if result is not None and result.latency_ms is not None else None
        text = built.source if built is not None else (result.code if result is not None else "")
        stages.append(Stage(plan.role, text, graph_out_indices(graph), wiring, plan.label, latency_us, built))
    return stages, (problems[0] if problems else None)
