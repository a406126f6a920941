"""Native call plans: what ``csrc/dispatch.cpp`` needs to know to run a compiled operator in one step.

``chain_plan`` turns compiled kernels (one, or the stages of a split operator in order) into a callable
that checks its arguments, allocates outputs and scratch and launches everything on the current
stream.  The callable returns ``NotImplemented`` for arguments it does not take (wrong type, extent,
layout, device); its owner then goes through the checked Python path, which says what is wrong.
"""

from __future__ import annotations

import ast
import ctypes
import importlib.util
import math
import sys
import threading
import warnings

from ..core.errors import BackendUnavailable, CompileError
from . import shim

MODULE_NAME = "_dispatch.so"
TENSOR, F32, I32 = range(3)
V_ARG, V_OUT, V_TEMP, V_DIM = range(4)
# postfix operators of csrc/dispatch.cpp, in its order
CONST, DIM, ADD, SUB, MUL, FLOORDIV, MOD, NEG, CEILDIV, MIN, MAX = range(11)
_BINARY = {ast.Add: ADD, ast.Sub: SUB, ast.Mult: MUL, ast.FloorDiv: FLOORDIV, ast.Mod: MOD}
_CALLS = {"ceildiv": CEILDIV, "min": MIN, "max": MAX}
BYTES = {"float16": 2, "bfloat16": 2, "float32": 4, "int32": 4}

_lock = threading.Lock()
_native = None


def native():
    """The extension module (cached).  Raises ``BackendUnavailable`` when it has not been built."""
    global _native
    with _lock:
        if _native is None:
            import torch  # noqa: F401  (its libraries must be mapped first)

            path = shim.CSRC_DIR / MODULE_NAME
            if not path.is_file():
                raise BackendUnavailable(f"{path} is missing: build it with `python -c 'import __graft_entry__ as g; "
                                         "g.build()'` or `make -C cleave_amd/csrc`; until then calls go step by step in Python")
            name = "cleave_amd.csrc._dispatch"
            spec = importlib.util.spec_from_file_location(name, path)
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
            sys.modules[name] = _native = module
    return _native


def postfix(expr, dims: dict) -> list:
    """``expr`` (an integer or an expression over named dims) as a postfix program; ``dims``: name -> index."""
    if isinstance(expr, int):
        return [CONST, int(expr)]

    def walk(node):
        if isinstance(node, ast.Constant) and isinstance(node.value, int):
            return [CONST, node.value]
        if isinstance(node, ast.Name):
            if node.id not in dims:
                raise CompileError(f"extent {expr!r} names an unknown dim {node.id!r}")
            return [DIM, dims[node.id]]
        if isinstance(node, ast.UnaryOp) and isinstance(node.op, ast.USub):
            return walk(node.operand) + [NEG]
        if isinstance(node, ast.BinOp) and type(node.op) in _BINARY:
            return walk(node.left) + walk(node.right) + [_BINARY[type(node.op)]]
        if isinstance(node, ast.Call) and isinstance(node.func, ast.Name) and node.func.id in _CALLS and node.args:
            code = walk(node.args[0])
            for arg in node.args[1:]:
                code += walk(arg) + [_CALLS[node.func.id]]
            return code
        raise CompileError(f"extent {expr!r} uses {type(node).__name__}")

    return walk(ast.parse(str(expr), mode="eval").body)


def _argument(p, dims: dict, shape=None, align=1):
    """``(kind, dtype, dims, alignment)`` of one argument; plain names found on the way get an index in ``dims``."""
    if p.role == "scalar":
        return (F32 if p.dtype.startswith("float") else I32, "", (), 1)
    axes = []
    for extent in p.shape if shape is None else shape:
        if isinstance(extent, int):
            axes.append(extent)
        elif str(extent).isidentifier():
            axes.append(-1 - dims.setdefault(str(extent), len(dims)))
        else:
            axes.append(str(extent))          # resolved once every plain name is known
    return (TENSOR, p.dtype, axes, align)


def plan_or_false(make):
    """``make()``, a native call plan; False where there is none, and calls stay on the checked Python path: the extension
    module is not built or does not load (said once), or the kernels are beyond what a plan holds (its numbers of
    dims, arguments, scratch buffers, output axes and launches, and its operators in extents)."""
    try:
        native()
    except (BackendUnavailable, ImportError, OSError) as e:
        warnings.warn(f"calls of compiled kernels go step by step in Python: {e}", RuntimeWarning, stacklevel=3)
        return False
    try:
        return make() or False
    except (CompileError, ValueError, OverflowError):
        return False


def chain_plan(stages, *, arguments=None, output_shapes=None, as_tuple=False):
    """A native call plan, or None where a kernel has a run-time extent that no argument names.  Kernels beyond the
    limits of a plan raise ``ValueError`` or ``CompileError`` (``plan_or_false`` answers False for them).

    ``stages``: ``[(compiled kernel, sources)]`` in order; ``sources[name]`` is ``("arg", i)`` or
    ``("stage", j)`` (output j of the stage before) for every input and scalar of the kernel, or
    ``sources`` is None for a single kernel whose arguments come in its own parameter order.
    ``arguments``: the plan's own argument list as ``[(ParamSpec-like, shape or None)]`` (None: the single
    kernel's caller parameters).  ``output_shapes``: shapes the last stage's outputs are given to the caller in."""
    module = native()
    import torch

    dims: dict = {}
    last = stages[-1][0]
    if arguments is None:
        caller = [p for p in last.params if p.role != "scratch" and (p.role != "output" or last.out_idx is None)]
        arguments = [(p, None) for p in caller]
        stages = [(last, {p.name: ("arg", i) for i, p in enumerate(caller)})]
    aligned = {sources[name] for kernel, sources in stages for name in kernel.aligned_inputs}
    args = [_argument(p, dims, shape, 16 if ("arg", i) in aligned else 1) for i, (p, shape) in enumerate(arguments)]
    n_dims = len(dims)
    derived = []
    for kernel, _ in stages:
        for name, expr in kernel.manifest.get("derived_dims", ()):
            program = postfix(expr, dims)
            if name not in dims:
                dims[name] = len(dims)
                derived.append(program)
    if any(d not in dims for kernel, _ in stages for d in kernel.dyn_dims):
        return None
    args = [(kind, dtype, [a if isinstance(a, int) else postfix(a, dims) for a in axes], al) for kind, dtype, axes, al in args]

    outs, temps, launches, before = [], [], [], []
    for kernel, sources in stages:
        place = {}

        def temp(p):
            size = [CONST, BYTES[p.dtype]]
            for extent in p.shape:
                size += postfix(extent, dims) + [MUL]
            temps.append(size)
            return V_TEMP, len(temps) - 1

        produced = []
        for p in kernel.params:
            if p.role == "scratch":
                owner = p.alias or p.name
                if owner not in place:
                    place[owner] = temp(p)
                place[p.name] = place[owner]
            elif p.role == "output":
                if kernel is not last:
                    place[p.name] = temp(p)
                elif kernel.out_idx is None and p.name in sources:
                    place[p.name] = (V_ARG, sources[p.name][1])
                else:
                    shape = p.shape
                    if output_shapes is not None and len(output_shapes) > len(outs) and all(isinstance(e, int) for e in p.shape) \
                            and math.prod(output_shapes[len(outs)]) == math.prod(p.shape):
                        shape = output_shapes[len(outs)]
                    place[p.name] = (V_OUT, len(outs))
                    outs.append((p.dtype, [postfix(e, dims) for e in shape]))
                produced.append(place[p.name])
            else:
                where, index = sources[p.name]
                place[p.name] = (V_ARG, index) if where == "arg" else before[index]
        for launch in kernel.manifest["launches"]:
            values = [place[name] if name in place else (V_DIM, dims[name]) for name in launch["args"]]
            block = list(launch["block"]) + [1] * (3 - len(launch["block"]))
            grid = list(launch["grid"]) + [1] * (3 - len(launch["grid"]))
            launches.append((kernel.module.function(launch["entry"]), [postfix(_number(g), dims) for g in grid],
                             tuple(int(b) for b in block), int(launch["lds"]), values, int(bool(launch.get("optional")))))
        before = produced
    lib = shim.load()
    return module.make_plan(args, n_dims, derived, outs, temps, launches, 2 if as_tuple else 1 if outs else 0,
                            tuple(kernel.module for kernel, _ in stages), torch._C._cuda_getCurrentRawStream,
                            _launch_failed, ctypes.cast(lib.chip_launch, ctypes.c_void_p).value)


def _launch_failed(status):
    """What a failed launch raises: the errors of the checked path (its text is the calling thread's own)."""
    shim._check(status, "chip_launch_seq")


def _number(text):
    try:
        return int(text)
    except (TypeError, ValueError):
        return text
