"""Runs a module function operation by operation on the gfx950 kernel library.

The reference lowers ANY module made of `linalg` / `sparse_tensor` / `scf` / `arith` operations to loops and
emits a kernel per loop nest (python/lapis/KokkosBackend.py:83-127, Pipelines/KokkosPipelines.cpp:42-153).
The prebuilt module has whole functions for the computations of the reference's examples; this file covers
every other function written in the same vocabulary: it walks the function's statements and hands each one
to the entry point of `include/lapis_hip.h` that computes it, with all tensors resident on the device
between operations.

    linalg.matvec / linalg.matmul with a CSR operand     lapis_hip_spmv_csr_* / lapis_hip_spmm_csr_*
    linalg.dot                                            lapis_hip_dot_*_host (the scalar comes back to the host, as
                                                          the reference's parallel_reduce does, TranslateToKokkosCpp.cpp:1696-1705)
    linalg.fill / copy / add / sub / mul / div, and parallel linalg.generic bodies that are a*x + b*y, a*x,
    x*y, x or a constant (lapis_amd/elementwise.py)       lapis_hip_fill / copy / axpby / mult / div
    tensor.empty / splat / dim / extract, memref.alloc / dim / load / store / copy, scalar arith.* and math.sqrt,
    scf.while / for / if, func.call
    scf.parallel nests that lapis_amd/loop_mapping.py recognises: the CSR SpMV nest, the CSR x dense SpMM nest,
    depth-1 reductions (dot) and depth-1 elementwise loops

Anything else is refused when the module is compiled (`check`), with the operation named, as the reference
refuses what its pipeline cannot lower.

Tensor values are immutable in MLIR; an operation's `outs` operand is overwritten in place only when it is a
temporary this region made itself (tensor.empty, tensor.splat or the result of an earlier linalg operation)
and no name that may stand for its buffer (its own, or that of a call's, a loop's or a branch's result that
may have passed it through) is mentioned afterwards, otherwise the result gets a buffer of its own.  Memref
operands are buffers and are always updated in place.
"""
import math
import re

import numpy

from . import elementwise as _ew
from . import loop_mapping as _lm
from . import mlir_text as _mt
from . import schedule as _sched


class Refused(Exception):
    """The function uses something outside the vocabulary; the message names it."""


_NAME = r"%[\w.$-]+(?:#\d+)?"
def _ieee(fn, quick=None):
    """Host scalars follow IEEE 754 as the emitted C++ does: x/0 is an infinity or a NaN, not an exception,
    and the maximum of a NaN and a number is a NaN."""
    def apply(a, b):
        if quick is not None and type(a) is float and type(b) is float and b:
            return quick(a, b)
        f32 = isinstance(a, numpy.float32) and isinstance(b, numpy.float32)
        with numpy.errstate(all="ignore"):
            r = fn(numpy.float32(a) if f32 else numpy.float64(a), numpy.float32(b) if f32 else numpy.float64(b))
        return numpy.float32(r) if f32 else float(r)
    return apply


_FLOAT_BIN = {"arith.addf": lambda a, b: a + b, "arith.subf": lambda a, b: a - b, "arith.mulf": lambda a, b: a * b,
              "arith.divf": _ieee(numpy.divide, lambda a, b: a / b), "arith.maximumf": _ieee(numpy.maximum),
              "arith.minimumf": _ieee(numpy.minimum)}
_INT_BIN = {"arith.addi": lambda a, b: a + b, "arith.subi": lambda a, b: a - b, "arith.muli": lambda a, b: a * b,
            "arith.divui": lambda a, b: a // b, "arith.divsi": lambda a, b: int(a / b) if b else 0,
            "arith.remui": lambda a, b: a % b, "arith.remsi": lambda a, b: a - b * int(a / b),
            "arith.andi": lambda a, b: a & b, "arith.ori": lambda a, b: a | b, "arith.xori": lambda a, b: a ^ b,
            "arith.maxsi": max, "arith.minsi": min, "arith.maxui": max, "arith.minui": min}
_CMPI = {"eq": lambda a, b: a == b, "ne": lambda a, b: a != b, "slt": lambda a, b: a < b, "sle": lambda a, b: a <= b,
         "sgt": lambda a, b: a > b, "sge": lambda a, b: a >= b, "ult": lambda a, b: a < b, "ule": lambda a, b: a <= b,
         "ugt": lambda a, b: a > b, "uge": lambda a, b: a >= b}
_CMPF = {"oeq": lambda a, b: a == b, "one": lambda a, b: a != b and a == a and b == b, "olt": lambda a, b: a < b,
         "ole": lambda a, b: a <= b, "ogt": lambda a, b: a > b, "oge": lambda a, b: a >= b,
         "ueq": lambda a, b: a == b or a != a or b != b, "une": lambda a, b: a != b,
         "ult": lambda a, b: not (a >= b), "ule": lambda a, b: not (a > b), "ugt": lambda a, b: not (a <= b),
         "uge": lambda a, b: not (a < b)}
_CASTS = ("arith.index_cast", "arith.index_castui", "arith.extui", "arith.extsi", "arith.trunci", "arith.sitofp",
          "arith.uitofp", "arith.fptosi", "arith.fptoui", "arith.extf", "arith.truncf")
_SCALAR_OPS = set(_FLOAT_BIN) | set(_INT_BIN) | set(_CASTS) | {
    "arith.constant", "arith.negf", "arith.cmpi", "arith.cmpf", "arith.select", "math.sqrt", "math.absf"}
_LINALG_NAMED = {"linalg.add": ("axpby", 1.0, 1.0), "linalg.sub": ("axpby", 1.0, -1.0), "linalg.mul": ("mult",),
                 "linalg.div": ("div",)}
_STRUCTURE = {"scf.while", "scf.for", "scf.if", "scf.condition", "scf.yield", "func.call", "call", "return",
              "func.return", "scf.parallel", "scf.reduce"}
_OWNING = {"tensor.empty", "tensor.splat", "memref.alloc", "memref.alloca", "bufferization.alloc_tensor", "linalg.fill",
           "linalg.copy", "linalg.matvec", "linalg.matmul", "linalg.generic"} | set(_LINALG_NAMED)  # results are buffers of this region
_NO_BUFFERS = (_SCALAR_OPS - {"arith.select"}) | {"linalg.dot", "tensor.dim", "tensor.extract", "memref.dim", "memref.load",
                                                  "lapis.dot_start", "lapis.dot_finish"}
_BUFFER_OPS = {"tensor.empty", "tensor.splat", "tensor.dim", "tensor.extract", "memref.alloc", "memref.alloca",
               "memref.dealloc", "memref.dim", "memref.load", "memref.store", "memref.copy", "linalg.fill",
               "linalg.copy", "linalg.dot", "linalg.matvec", "linalg.matmul", "linalg.generic",
               "bufferization.alloc_tensor"} | set(_LINALG_NAMED)
VOCABULARY = _SCALAR_OPS | _STRUCTURE | _BUFFER_OPS


class Csr:
    """A CSR operand on the device: the three buffers, the sizes, and the SpMV plan made at its first product."""

    def __init__(self, pos, crd, val, nrows, ncols):
        self.pos, self.crd, self.val, self.nrows, self.ncols = pos, crd, val, int(nrows), int(ncols)
        self.nnz = int(crd.shape[0])
        # the kernels index with what the buffers hold: sizes that do not agree must stop here, on the host
        if self.nrows < 0 or self.ncols < 0 or int(pos.shape[0]) != self.nrows + 1:
            raise ValueError("a %d x %d CSR operand needs %d positions, got %d" % (
                self.nrows, self.ncols, self.nrows + 1, int(pos.shape[0])))
        if int(val.shape[0]) != self.nnz:
            raise ValueError("a CSR operand with %d coordinates and %d values" % (self.nnz, int(val.shape[0])))
        self.plan = None
        self.products = 0
        self.staged = None  # makes the plan where the pass that brought the buffers to the device has counted the structure

    def release(self):
        if self.plan is not None:
            self.plan.destroy()
            self.plan = None
        self.staged = None


class Cell:
    """A zero-dimensional memref: one scalar, kept on the host."""

    def __init__(self, value=0.0):
        self.value = value


def _same_size(what, *tensors):
    """The kernels take one element count for all their operands: refuse, on the host, operands that differ."""
    sizes = [int(t.numel()) for t in tensors]
    if len(set(sizes)) > 1:
        raise ValueError("%s over operands of %s elements" % (what, ", ".join(map(str, sizes))))


def _elem(ty):
    m = re.search(r"x?(f64|f32|i64|i32|i1|index)\s*(?:,|>)", ty)
    return m.group(1) if m else ty.strip()


def _shape_spec(ty):
    """Dimensions of a tensor / memref type as a list of ints and None (dynamic), and its element type."""
    m = re.match(r"\s*(?:tensor|memref)<(.*)>\s*$", ty, re.S)
    if not m:
        raise Refused("a value of type %s" % ty.strip())
    first = _mt.split_top(m.group(1))[0].strip()
    parts = first.split("x")
    return [None if p == "?" else int(p) for p in parts[:-1]], parts[-1].strip()


def _split_colon(text):
    """`names : types` split at the first depth-0 colon."""
    depth = 0
    for i, ch in enumerate(text):
        if ch in "<([{":
            depth += 1
        elif ch in ">)]}" and not (ch == ">" and i and text[i - 1] == "-"):
            depth -= 1
        elif ch == ":" and depth == 0 and text[i:i + 2] != "::":
            return text[:i], text[i + 1:]
    return text, ""


def _rsplit_colon(text):
    """`left : type` split at the LAST depth-0 colon."""
    depth, at = 0, -1
    for i, ch in enumerate(text):
        if ch in "<([{":
            depth += 1
        elif ch in ">)]}" and not (ch == ">" and text[i - 1] == "-"):
            depth -= 1
        elif ch == ":" and depth == 0:
            at = i
    return (text[:at], text[at + 1:]) if at >= 0 else (text, "")


def _group(head, keyword):
    """(names, types) inside `keyword( ... )` of a statement head, or ([], [])."""
    m = re.search(r"\b%s\s*\(" % keyword, head)
    if not m:
        return [], []
    i = m.end() - 1
    inner = head[i + 1:_mt._match(head, i) - 1]
    names, types = _split_colon(inner)
    return re.findall(_NAME, names), [t.strip() for t in _mt.split_top(types)] if types.strip() else []


def _flat(t):
    return t if t.dim() == 1 else t.reshape(-1)


def _constant(head):
    left, ty = _split_colon(head)
    tok, ty = left.strip(), ty.strip()
    if tok in ("true", "false"):
        return tok == "true"
    if ty in ("f64", "f32"):
        return numpy.float32(tok) if ty == "f32" else float(tok)
    return int(float(tok)) if ty != "i1" else bool(int(tok))


def _sqrt(v):
    if type(v) is float and v >= 0.0:
        return math.sqrt(v)
    with numpy.errstate(all="ignore"):  # the root of a negative number is a NaN
        return numpy.sqrt(v) if isinstance(v, numpy.floating) else float(numpy.sqrt(v))


def _coefficient(expr):
    """A function (values by name, destination) that gives the number a coefficient expression stands for."""
    def general(env, d):
        return float(_ew.evaluate(expr, env.__getitem__, numpy.float32 if d.element_size() == 4 else float))
    if expr[0] == "const":
        return general if float(numpy.float32(expr[1])) != expr[1] else (lambda env, d, v=expr[1]: v)
    sign = 1.0
    while expr[0] == "neg":
        sign, expr = -sign, expr[1]
    if expr[0] != "name":
        if sign < 0.0:
            expr = ("neg", expr)
        return general
    name = expr[1]

    def value(env, d):
        v = float(env[name])
        return sign * (float(numpy.float32(v)) if d.element_size() == 4 else v)
    return value


def _raises(e):
    def step(env):
        raise e
    return step


def _giving(op, names, fn):
    """A step that stores what `fn(values)` returns (a list, or None for no results) under `names`."""
    def step(env):
        results = fn(env)
        if results is not None:
            if len(results) != len(names):
                raise RuntimeError("%s gave %d values for %d results" % (op, len(results), len(names)))
            env.update(zip(names, results))
    return step


class _Block:
    """The steps of a region, its constants, and the terminator with the names of the values it passes on."""

    def __init__(self):
        self.constants, self.steps, self.ops, self.end, self.names = {}, [], [], "end", []

    def add(self, op, step):
        self.ops.append(op)
        self.steps.append(step)

    def run(self, env):
        env.update(self.constants)
        at = 0
        try:
            for step in self.steps:
                step(env)
                at += 1
            return self.end, [env[n] for n in self.names]
        except KeyError as e:
            name = e.args[0] if e.args else None
            if isinstance(name, str) and name.startswith("%"):
                raise RuntimeError("value %s is used before it is defined" % name)
            self._wrong_type(at, e)
        except ZeroDivisionError:
            raise RuntimeError("%s: integer division by zero" % self.ops[at])
        except (AttributeError, TypeError, IndexError) as e:
            self._wrong_type(at, e)

    def _wrong_type(self, at, e):
        # an operand that is not what the operation's types say (a scalar where a tensor is named, ...):
        # text MLIR's own verifier would not have let through
        raise RuntimeError("%s: an operand does not have the type the operation declares (%s: %s)" % (
            self.ops[at] if at < len(self.ops) else self.end, type(e).__name__, e))


class Executor:
    def __init__(self, canonicalizer, torch_module=None, hip_module=None, device="cuda"):
        # `hip_module` / `device`: the tests of the host logic pass a stand-in for lapis_amd.hip that works on
        # CPU tensors; the product never does (KokkosBackend constructs Executor(canonicalizer))
        self.device = device
        self.c = canonicalizer
        self.aliases = canonicalizer.aliases
        self._parsed = {}
        self._programs = {}
        self._torch = torch_module
        self._hip = hip_module

    # ---- lazily imported plumbing -----------------------------------------------------------------
    @property
    def torch(self):
        if self._torch is None:
            import torch
            self._torch = torch
        return self._torch

    @property
    def hip(self):
        if self._hip is None:
            from . import hip
            hip.init()
            self._hip = hip
        return self._hip

    def _function(self, name):
        if name not in self.c.functions:
            raise Refused("a call of @%s, which the module does not define" % name)
        f = self.c.functions[name]
        if f.body is None:
            raise Refused("a call of @%s, which is declared without a body" % name)
        if name not in self._parsed:
            stmts, _ = _mt.read_region(f.body)
            nests = {}
            if "scf.parallel" in f.body:
                for n in _lm.map_statements(stmts, hip_kernels=True):
                    nests[id(n.stmt)] = n
            self._parsed[name] = (stmts, nests)
        return f, self._parsed[name][0], self._parsed[name][1]

    # ---- what can be told without running -----------------------------------------------------------
    def check(self, name, _seen=None):
        """Raises Refused naming the first thing in @name (or a function it calls) that the library cannot run."""
        seen = _seen if _seen is not None else set()
        if name in seen:
            return
        seen.add(name)
        f, stmts, nests = self._function(name)
        for _, ty in f.args:
            self._check_type(ty)
        self._check_region(stmts, nests, seen, {nm: ty for nm, ty in f.args})

    def _check_type(self, ty):
        ty = ty.strip()
        if ty in ("f64", "f32", "index", "i64", "i32", "i1"):
            return
        kind = _mt.type_kind(ty, self.aliases) if ty.startswith("tensor<") else None
        if kind:
            if kind.startswith("sparse(") or kind.startswith("csrv"):
                raise Refused("an operand stored as %s; CSR with 32-bit positions and coordinates is what the kernel "
                              "library multiplies with" % kind)
            if kind.split(":")[1] not in ("f64", "f32"):
                raise Refused("a tensor of %s" % kind.split(":")[1])
            return
        if ty.startswith("memref<"):
            if "strided" in ty or "affine_map" in ty:
                raise Refused("a memref with a layout (%s)" % ty)
            return
        raise Refused("a value of type %s" % ty)

    def _check_region(self, stmts, nests, seen, arg_types):
        for s in stmts:
            if s.op not in VOCABULARY:
                raise Refused("the operation %s" % s.op)
            if s.op == "scf.parallel":
                n = nests.get(id(s))
                if n is None or not (n.csr_spmv or n.depth1 or n.csr_spmm):
                    raise Refused("a %s loop nest of depth %s that is none of the CSR SpMV nest, the CSR x dense SpMM "
                                  "nest, a depth-1 dot product or a depth-1 elementwise loop"
                                  % ((n.space, n.depth) if n is not None else ("nested", "?")))
                roles = n.csr_spmv or n.csr_spmm
                if roles:
                    what = "SpMV" if n.csr_spmv else "SpMM"
                    for role in ("pos", "crd"):
                        ty = arg_types.get(roles[role])
                        if ty is None or not re.match(r"memref<\?xi32>$", ty.replace(" ", "")):
                            raise Refused("the %s buffer of its %s nest is %s; the kernel library indexes with 32-bit "
                                          "positions and coordinates held in function arguments of type memref<?xi32>"
                                          % (role, what, ty or "not a function argument"))
                continue
            if s.op in ("func.call", "call"):
                m = re.search(r"@([\w$.-]+)", s.head)
                if not m:
                    raise Refused("an indirect call")
                self.check(m.group(1), seen)
            elif s.op in ("linalg.matvec", "linalg.matmul"):
                _, types = _group(s.head, "ins")
                if not types or not _mt.type_kind(types[0], self.aliases).startswith("csr:"):
                    raise Refused("%s whose first operand is not a CSR tensor with 32-bit positions and coordinates"
                                  % s.op)
                if len(types) > 1 and "#" in types[1]:
                    raise Refused("%s with a sparse second operand" % s.op)
            elif s.op == "linalg.generic":
                self._generic_plan(s)
            elif s.op == "arith.constant" and "dense" in s.head:
                raise Refused("a dense constant")
            if s.op != "linalg.generic":
                for _, sub in s.regions:
                    self._check_region(sub, nests, seen, arg_types)

    # ---- linalg.generic ------------------------------------------------------------------------------
    def _generic_plan(self, s):
        """("elementwise", call, n_ins) | ("matvec",) | ("matmul",) for a linalg.generic statement."""
        maps_m = re.search(r"indexing_maps\s*=\s*\[", s.head)
        iters = re.search(r"iterator_types\s*=\s*\[([^\]]*)\]", s.head)
        if not maps_m or not iters or len(s.regions) != 1:
            raise Refused("a linalg.generic without indexing maps, iterator types or a body")
        i = maps_m.end() - 1
        maps = []
        for a in _mt.split_top(s.head[i + 1:_mt._match(s.head, i) - 1]):
            a = a.strip()
            seen = set()
            while a in self.aliases and a not in seen:
                seen.add(a)
                a = self.aliases[a]
            m = re.search(r"\(([^)]*)\)\s*->\s*\(([^)]*)\)", a)
            if not m:
                raise Refused("an indexing map %s" % a)
            dims = [d.strip() for d in m.group(1).split(",") if d.strip()]
            maps.append(tuple(dims.index(r.strip()) if r.strip() in dims else r.strip()
                              for r in m.group(2).split(",") if r.strip()))
        kinds = re.findall(r"parallel|reduction", iters.group(1))
        ins, in_types = _group(s.head, "ins")
        outs, _ = _group(s.head, "outs")
        bargs, body = s.regions[0]
        if len(outs) != 1 or len(bargs) != len(ins) + 1 or not body or body[-1].op != "linalg.yield":
            raise Refused("a linalg.generic with %d outputs" % len(outs))
        yielded = re.findall(_NAME, body[-1].head)
        if len(yielded) != 1:
            raise Refused("a linalg.generic that yields %d values" % len(yielded))
        rank = len(kinds)
        ident = tuple(range(rank))
        if all(k == "parallel" for k in kinds) and all(m == ident for m in maps):
            for t in in_types:
                if "#" in t:
                    raise Refused("an elementwise linalg.generic over a sparse operand")
            try:
                poly = _ew.polynomial(body[:-1], lambda nm: bargs.index(nm) if nm in bargs else None, yielded[0])
                call = _ew.classify(poly)
            except _ew.Unsupported as e:
                raise Refused("a linalg.generic body the library has no kernel for: %s" % e)
            return ("elementwise", call, len(ins))
        # the two contractions, written as generics (examples/spmm_dcsr_opdsl.py:73-78 of the reference)
        if len(ins) == 2 and in_types and _mt.type_kind(in_types[0], self.aliases).startswith("csr:"):
            try:
                poly = _ew.polynomial(body[:-1], lambda nm: bargs.index(nm) if nm in bargs else None, yielded[0])
            except _ew.Unsupported as e:
                raise Refused("a contraction body the library has no kernel for: %s" % e)
            one = ("const", 1.0)
            if {k: c for k, c in poly.terms.items() if c != ("const", 0.0)} == {(0, 1): one, (2,): one}:
                if kinds == ["parallel", "reduction"] and maps == [(0, 1), (1,), (0,)]:
                    return ("matvec",)
                if kinds == ["parallel", "parallel", "reduction"] and maps == [(0, 2), (2, 1), (0, 1)]:
                    return ("matmul",)
        raise Refused("a linalg.generic that is neither elementwise over identity maps nor out += A*b with a CSR A")

    # ---- running --------------------------------------------------------------------------------------
    def run(self, name, args):
        """Results of @name for `args` (device tensors, Csr operands, host scalars), as a list."""
        names, block = self._program(name)
        kind, values = block.run(dict(zip(names, args)))
        if kind != "return":
            raise RuntimeError("@%s ended without a return" % name)
        return values

    def _program(self, name):
        """(argument names, the function's statements as steps), made when a function is first run."""
        if name not in self._programs:
            f, stmts, nests = self._function(name)
            if hasattr(self.hip, "dot_start") and not nests:
                stmts = _sched.inline(stmts, self._inlinable, {name}, [0])
            self._programs[name] = ([nm for nm, _ in f.args], self._block(stmts, nests, {}))
        return self._programs[name]

    def _inlinable(self, name):
        f, stmts, nests = self._function(name)
        return None if nests else ([nm for nm, _ in f.args], stmts)

    def _kind(self, s):
        if s.op == "linalg.matvec":
            return "product"
        if s.op in ("linalg.add", "linalg.sub"):
            return "axpby" if len(_group(s.head, "ins")[0]) == 2 else None
        if s.op == "linalg.generic":
            try:
                plan = self._generic_plan(s)
            except Refused:
                return None
            return "product" if plan == ("matvec",) else "axpby" if plan[0] == "elementwise" and plan[1][0] == "axpby" else None
        return None

    def _block(self, stmts, nests, constants):
        constants = dict(constants)
        for s in stmts:
            if s.op == "arith.constant" and len(s.results) == 1:
                try:
                    constants[s.results[0]] = _constant(s.head)
                except ValueError:
                    pass
        if hasattr(self.hip, "dot_start") and not nests:
            stmts = _sched.rewrite(stmts, self._kind, constants)
        said = [_sched.mentions(s) for s in stmts]
        scalar = lambda s: s.op in _NO_BUFFERS or (s.op == "arith.select" and not re.search(r"\b(?:tensor|memref)\s*<", s.head))
        fresh = lambda s: (s.op in _OWNING or isinstance(s, _sched.Fused)) and not scalar(s)
        buffers = _sched.buffers(zip(stmts, said), fresh, scalar)
        last = {}  # the last statement that mentions a name of the buffer
        for k, names in enumerate(said):
            for n in names:
                for nm in buffers.get(n, (n,)):
                    last[nm] = k
        block, owned, defined = _Block(), set(), set()
        for k, s in enumerate(stmts):
            op = s.op
            if op in ("return", "func.return", "scf.yield", "scf.condition"):
                block.end, block.names = op.split(".")[-1], re.findall(_NAME, _split_colon(s.head)[0])
                break
            if op == "arith.constant" and s.results[0] in constants:
                block.constants[s.results[0]] = constants[s.results[0]]
                continue
            # `reads`: operands whose elements the operation still needs when it has written others
            can_overwrite = lambda nm, *reads, k=k: nm in owned and nm in defined and last.get(nm, k) <= k and \
                not any(nm in buffers.get(other, (other,)) for other in reads)
            try:
                step = self._step(s, nests, can_overwrite, constants)
            except (AttributeError, TypeError, IndexError, KeyError, ValueError) as e:
                step = _raises(e)
            block.add(op, step)
            names = _sched.result_names(s)
            defined.update(names)
            if fresh(s):
                owned.update(names[:1])
        return block

    # Every statement becomes a step: a function of the values by name that leaves its results among them.
    def _step(self, s, nests, can_overwrite, constants):
        op, head = s.op, s.head
        names = _sched.result_names(s)
        if op in _SCALAR_OPS:
            return self._scalar_step(op, head, names[0])
        if op.startswith("lapis."):
            return self._fused_step(s, can_overwrite)
        if op == "scf.parallel":
            nest = nests[id(s)]
            return _giving(op, names, lambda env: self._nest(s, nest, env))
        if op in ("func.call", "call"):
            callee = re.search(r"@([\w$.-]+)", head).group(1)
            i = head.index("(")
            given = re.findall(_NAME, head[i:_mt._match(head, i)])
            return _giving(op, names, lambda env: self.run(callee, [env[n] for n in given]))
        if op == "scf.while":
            return _giving(op, names, self._while(s, nests, constants))
        if op == "scf.for":
            return _giving(op, names, self._for(s, nests, constants))
        if op == "scf.if":
            cond = re.findall(_NAME, head)[0]
            blocks = [self._block(sub, nests, constants) for _, sub in s.regions]

            def branch(env):
                if env[cond]:
                    values = blocks[0].run(dict(env))[1]
                elif len(blocks) > 1:
                    values = blocks[1].run(dict(env))[1]
                else:
                    return None
                return values if s.results else None
            return _giving(op, names, branch)
        return self._buffer_step(s, names, can_overwrite)

    def _scalar_step(self, op, head, r):
        left, ty = _split_colon(head)
        ty = ty.strip()
        if op == "arith.constant":
            v = _constant(head)

            def step(env):
                env[r] = v
            return step
        ops = re.findall(_NAME, left)
        if op in ("arith.cmpi", "arith.cmpf"):
            fn = (_CMPI if op == "arith.cmpi" else _CMPF)[re.match(r"\s*(\w+)", left).group(1)]
        else:
            fn = _FLOAT_BIN.get(op) or _INT_BIN.get(op)
        if fn is not None:
            a, b = ops[0], ops[1]

            def step(env):
                env[r] = fn(env[a], env[b])
            return step
        if op == "arith.select":
            c, a, b = ops[:3]

            def step(env):
                env[r] = env[a] if env[c] else env[b]
            return step
        if op == "arith.negf":
            fn = lambda v: -v
        elif op == "math.sqrt":
            fn = _sqrt
        elif op == "math.absf":
            fn = abs
        elif op in _CASTS:
            target = ty.split("to")[-1].strip()
            fn = numpy.float32 if target == "f32" else float if target == "f64" else int
        else:
            raise Refused("the operation %s" % op)
        a = ops[0]

        def step(env):
            env[r] = fn(env[a])
        return step

    # ---- structured control flow -----------------------------------------------------------------------
    def _while(self, s, nests, constants):
        head = s.head
        i = head.index("(")
        inits = [p.split("=") for p in _mt.split_top(head[i + 1:_mt._match(head, i) - 1]) if "=" in p]
        before_names = [a.strip() for a, _ in inits]
        init_names = [b.strip() for _, b in inits]
        (_, before), (after_args, after) = s.regions
        before, after = self._block(before, nests, constants), self._block(after, nests, constants)

        def loop(env):
            values = [env[n] for n in init_names]
            while True:
                e = dict(env)
                e.update(zip(before_names, values))
                kind, out = before.run(e)
                if kind != "condition":
                    raise RuntimeError("the first region of scf.while does not end in scf.condition")
                if not out[0]:
                    return out[1:]
                e = dict(env)
                e.update(zip(after_args, out[1:]))
                kind, values = after.run(e)
                if kind != "yield":
                    raise RuntimeError("the second region of scf.while does not end in scf.yield")
        return loop

    def _for(self, s, nests, constants):
        m = re.match(r"\s*(%s)\s*=\s*(%s)\s*to\s*(%s)\s*step\s*(%s)" % ((_NAME,) * 4), s.head)
        if not m:
            raise Refused("an scf.for that is not `%i = lo to hi step st`")
        iv, lo, hi, st = m.groups()
        carried, inits = [], []
        im = re.search(r"iter_args\s*\(", s.head)
        if im:
            i = im.end() - 1
            for p in _mt.split_top(s.head[i + 1:_mt._match(s.head, i) - 1]):
                a, b = p.split("=")
                carried.append(a.strip())
                inits.append(b.strip())
        body = self._block(s.regions[0][1], nests, constants)

        def loop(env):
            values = [env[n] for n in inits]
            for k in range(env[lo], env[hi], env[st]):
                e = dict(env)
                e[iv] = k
                e.update(zip(carried, values))
                kind, out = body.run(e)
                if carried:
                    values = out
            return values if s.results else None
        return loop

    # ---- tensors and memrefs ---------------------------------------------------------------------------
    def _allocation(self, ty, names):
        """A function of the values that allocates a tensor of the type, its dynamic sizes taken from `names`; None for
        zero dimensions."""
        dims, elem = _shape_spec(ty)
        if not dims:
            return None
        torch = self.torch
        dtype = torch.float64 if elem == "f64" else torch.float32 if elem == "f32" else torch.int32
        dyn = iter(names)
        dims = [d if d is not None else next(dyn) for d in dims]
        device = torch.device(self.device)
        return lambda env: torch.empty([env[d] if isinstance(d, str) else d for d in dims], dtype=dtype, device=device)

    def _csr_product(self, A, x, y, k=None, overwrite=False, dot=None):
        """y += A x, or with k columns Y += A X; overwrite: y = A x; dot: y = A x and the start of dot + x . y."""
        hip = self.hip
        if k is None:
            if x.numel() != A.ncols or y.numel() != A.nrows:
                raise ValueError("a %d x %d matrix times a vector of %d elements into one of %d" % (
                    A.nrows, A.ncols, x.numel(), y.numel()))
        elif tuple(x.shape) != (A.ncols, k) or tuple(y.shape) != (A.nrows, k):
            raise ValueError("a %d x %d matrix times a %s matrix into a %s one" % (
                A.nrows, A.ncols, "x".join(map(str, x.shape)), "x".join(map(str, y.shape))))
        if A.plan is None:
            A.plan = A.staged() if A.staged else \
                hip.CsrPlan(A.nrows, A.ncols, A.pos, A.crd, value_bytes=A.val.element_size(), nnz=A.nnz)
        A.products += 1
        if k is not None:
            hip.spmm(A.nrows, A.ncols, A.pos, A.crd, A.val, x, y, plan=A.plan)
            return y
        if A.products == 6:  # a matrix multiplied with again and again: let the library decide on its blocked copy
            A.plan.analyze(A.crd, A.val)
        if dot is not None:
            return y, hip.spmv_dot_start(A.plan, A.nrows, A.ncols, A.pos, A.crd, A.val, x, y, dot)
        (hip.spmv_overwrite if overwrite else hip.spmv)(A.plan, A.nrows, A.ncols, A.pos, A.crd, A.val, x, y)
        return y

    def _elementwise(self, call):
        """A function (operands, dst, values by name) that computes dst = call(operands) on flat device tensors."""
        hip, kind = self.hip, call[0]
        coefficient = [_coefficient(c) if isinstance(c, tuple) else None for c in call]

        def checked(fn):
            def go(operands, dst, env):
                _same_size("an elementwise operation", dst, *operands)
                fn([_flat(o) for o in operands], _flat(dst), env)
                return dst
            return go
        if kind == "fill":
            return checked(lambda o, d, env: hip.fill(d, coefficient[1](env, d)))
        if kind == "copy":
            return checked(lambda o, d, env: hip.copy(o[call[1]], d) if o[call[1]].data_ptr() != d.data_ptr() else None)
        if kind == "scale":
            return checked(lambda o, d, env: hip.axpby(coefficient[1](env, d), o[call[2]], 0.0, o[call[2]], d))
        if kind == "mult":
            return checked(lambda o, d, env: hip.mult(o[call[1]], o[call[2]], d))
        if kind == "axpby":
            return checked(lambda o, d, env: hip.axpby(coefficient[1](env, d), o[call[2]], coefficient[3](env, d), o[call[4]], d))
        raise Refused("elementwise %s" % kind)

    def _dest(self, nm, can_overwrite, *reads):
        """A function of the values that gives the buffer a tensor operation's result goes to: the `outs` operand
        itself where that is allowed, else a new one of its size.  What the operation reads of the operand it
        reads from the operand; `reads` names what must not be the same buffer."""
        if can_overwrite(nm, *reads):
            return lambda env: env[nm]
        empty_like = self.torch.empty_like
        return lambda env: empty_like(env[nm])

    def _axpby_operands(self, s):
        """(first coefficient, its operand, second coefficient, its operand, outs operand) of an a*x + b*y statement."""
        ins, outs = _group(s.head, "ins")[0], _group(s.head, "outs")[0]
        if s.op == "linalg.generic":
            call = self._generic_plan(s)[1]
            operands = ins + outs
            return _coefficient(call[1]), operands[call[2]], _coefficient(call[3]), operands[call[4]], outs[0]
        spec = _LINALG_NAMED[s.op]
        return (lambda env, d: spec[1]), ins[0], (lambda env, d: spec[2]), ins[1], outs[0]

    # what lapis_amd/schedule.py makes of several statements
    def _fused_step(self, s, can_overwrite):
        hip, op = self.hip, s.op
        if op == "lapis.alias":
            name, value = s.results[0], s.head.strip()

            def step(env):
                env[name] = env[value]
            return step
        if op == "lapis.product":
            r = s.results[0]
            A, x = _group(s.parts[0].head, "ins")[0]
            dest = self._dest(s.outs, can_overwrite, x)

            def step(env):
                env[r] = self._csr_product(env[A], env[x], dest(env), overwrite=True)
            return step
        if op == "lapis.product_dot":
            r, product = s.results[0], s.parts[0]
            A, x = _group(product.parts[0].head, "ins")[0]
            init = _group(s.parts[1].head, "outs")[0][0]
            dest = self._dest(product.outs, can_overwrite, x)

            def step(env):
                d, x_ = dest(env), env[x]
                _same_size("linalg.dot", x_, d)
                env[r], env[id(s)] = self._csr_product(env[A], x_, d, dot=float(env[init]))
            return step
        if op == "lapis.elementwise_dot":
            r, other = s.results[0], s.other
            ca, a, cb, b, out = self._axpby_operands(s.parts[0])
            init = _group(s.parts[1].head, "outs")[0][0]
            dest = self._dest(out, can_overwrite, *([] if other is None else [other]))

            def step(env):
                d, va, vb = dest(env), env[a], env[b]
                _same_size("an elementwise operation", d, va, vb)
                z = None
                if other is not None:
                    z = env[other]
                    _same_size("linalg.dot", d, z)
                    z = _flat(z)
                env[id(s)] = hip.axpby_dot_start(ca(env, d), _flat(va), cb(env, d), _flat(vb), _flat(d), z, float(env[init]))
                env[r] = d
            return step
        if op == "lapis.dot_start":
            a, b = _group(s.parts[0].head, "ins")[0]
            init = _group(s.parts[0].head, "outs")[0][0]

            def step(env):
                va, vb = env[a], env[b]
                _same_size("linalg.dot", va, vb)
                env[id(s)] = hip.dot_start(_flat(va), _flat(vb), float(env[init]))
            return step
        if op == "lapis.dot_finish":
            r, start = s.results[0], id(s.start)
            f32 = re.search(r"f32\s*>\s*$", s.start.parts[-1].head) is not None

            def step(env):
                v = hip.dot_finish(env.pop(start))
                env[r] = numpy.float32(v) if f32 else v
            return step
        raise Refused("the operation %s" % op)

    def _buffer_step(self, s, names, can_overwrite):
        op, head = s.op, s.head
        torch, hip = self.torch, self.hip
        r = names[0] if names else None
        if op in ("tensor.empty", "memref.alloc", "memref.alloca", "bufferization.alloc_tensor"):
            left, ty = _rsplit_colon(head)
            i = left.index("(")
            new = self._allocation(ty, re.findall(_NAME, left[i:_mt._match(left, i)]))
            if new is None:
                new = (lambda env: Cell(0.0)) if op.startswith("memref") else (lambda env: 0.0)

            def step(env):
                env[r] = new(env)
            return step
        if op == "memref.dealloc":
            return lambda env: None
        if op == "tensor.splat":
            left, ty = _rsplit_colon(head)
            ops = re.findall(_NAME, left)
            v, new = ops[0], self._allocation(ty, ops[1:])

            def step(env):
                if new is None:
                    env[r] = env[v]
                else:
                    t = new(env)
                    hip.fill(t.view(-1), float(env[v]))
                    env[r] = t
            return step
        ops = re.findall(_NAME, _split_colon(head)[0])
        if op in ("tensor.dim", "memref.dim"):
            def step(env):
                t, d = env[ops[0]], env[ops[1]]
                env[r] = (t.nrows, t.ncols)[d] if isinstance(t, Csr) else int(t.shape[d])
            return step
        if op in ("tensor.extract", "memref.load"):
            def step(env):
                t = env[ops[0]]
                if isinstance(t, Cell):
                    env[r] = t.value
                elif not isinstance(t, torch.Tensor):  # a zero-dimensional tensor is kept as a host scalar
                    env[r] = t
                else:
                    v = t[tuple(env[n] for n in ops[1:])].item()  # waits for the kernels that produce it
                    env[r] = numpy.float32(v) if t.dtype == torch.float32 else v
            return step
        if op == "memref.store":
            def step(env):
                v, t = env[ops[0]], env[ops[1]]
                if isinstance(t, Cell):
                    t.value = v
                else:
                    t[tuple(env[n] for n in ops[2:])] = v
            return step
        if op == "memref.copy":
            def step(env):
                src, dst = env[ops[0]], env[ops[1]]
                if isinstance(dst, Cell):
                    dst.value = src.value
                else:
                    dst.copy_(src)
            return step

        ins, _ = _group(head, "ins")
        outs, _ = _group(head, "outs")
        if len(outs) != 1:
            raise Refused("%s with %d outputs" % (op, len(outs)))
        out_nm = outs[0]
        is_tensor = lambda v: isinstance(v, torch.Tensor)  # otherwise a zero-dimensional tensor (host scalar) or a Cell
        dest = self._dest(out_nm, can_overwrite) if r else (lambda env: env[out_nm])  # memrefs are updated in place

        def giving(compute):
            """`compute(values, destination)` for an operation on tensors"""
            def step(env):
                d = dest(env)
                compute(env, d)
                if r:
                    env[r] = d
            return step

        if op == "linalg.fill":
            def fill(env, d):
                hip.fill(_flat(d), float(env[ins[0]]))
            on_tensors = giving(fill)

            def step(env):
                out = env[out_nm]
                if is_tensor(out):
                    on_tensors(env)
                elif isinstance(out, Cell):
                    out.value = env[ins[0]]
                else:
                    env[r] = env[ins[0]]
            return step
        if op == "linalg.copy":
            def copy(env, d):
                v = env[ins[0]]
                if d.data_ptr() != v.data_ptr():
                    _same_size("linalg.copy", v, d)
                    hip.copy(_flat(v), _flat(d))
            on_tensors = giving(copy)

            def step(env):
                if is_tensor(env[out_nm]):
                    on_tensors(env)
                else:
                    env[r] = env[ins[0]]
            return step
        if op == "linalg.dot":
            a, b = ins[0], ins[1]

            def step(env):
                out, va, vb = env[out_nm], env[a], env[b]
                _same_size("linalg.dot", va, vb)
                v = hip.dot_host(_flat(va), _flat(vb), float(out.value if isinstance(out, Cell) else out))
                v = numpy.float32(v) if va.element_size() == 4 else v
                if isinstance(out, Cell):
                    out.value = v
                else:
                    env[r] = v
            return step
        plan = self._generic_plan(s) if op == "linalg.generic" else None
        if op in ("linalg.matvec", "linalg.matmul") or plan in (("matvec",), ("matmul",)):
            wide = op == "linalg.matmul" or plan == ("matmul",)
            in_place = r is None or can_overwrite(out_nm, ins[1])

            def step(env):
                out, x = env[out_nm], env[ins[1]]
                d = out if in_place else out.clone()
                self._csr_product(env[ins[0]], x, d, k=int(x.shape[1]) if wide else None)
                if r:
                    env[r] = d
            return step
        if op in _LINALG_NAMED:
            spec = _LINALG_NAMED[op]

            def named(env, d):
                a, b = _flat(env[ins[0]]), _flat(env[ins[1]])
                _same_size(op, a, b, d)
                if spec[0] == "axpby":
                    hip.axpby(spec[1], a, spec[2], b, _flat(d))
                elif spec[0] == "mult":
                    hip.mult(a, b, _flat(d))
                else:
                    hip.div(a, b, _flat(d))
            return giving(named)
        if op == "linalg.generic":
            _, call, n_ins = plan
            apply = self._elementwise(call)
            used = {c for c in call[1:] if isinstance(c, int)}

            def generic(env, d):
                operands = [env[n] for n in ins]
                operands.append(env[out_nm] if n_ins in used else d)
                apply(operands, d, env)
            on_tensors = giving(generic)

            def step(env):
                if not is_tensor(env[out_nm]):
                    raise Refused("an elementwise linalg.generic over zero-dimensional tensors")
                on_tensors(env)
            return step
        raise Refused("the operation %s" % op)

    # ---- loop nests the library has kernels for ----------------------------------------------------------
    def _nest(self, s, n, env):
        hip = self.hip
        if n.csr_spmv:
            r = n.csr_spmv
            y, pos, crd, val, x = (env[r[k]] for k in ("y", "pos", "crd", "val", "x"))
            A = self._csr_for(pos, crd, val, int(y.shape[0]), int(x.shape[0]))
            self._csr_product(A, x, y)
            return None
        if n.csr_spmm:
            r = n.csr_spmm
            C, pos, crd, val, B = (env[r[k]] for k in ("C", "pos", "crd", "val", "B"))
            A = self._csr_for(pos, crd, val, int(C.shape[0]), int(B.shape[0]))
            self._csr_product(A, B, C, k=int(B.shape[1]))
            return None
        d = n.depth1
        count = env[d["n"]] if d["n"] in env else int(d["n"])
        if count < 0 or any(int(env[a].shape[0]) < count
                            for a in ([d["x"], d["y"]] if d["kind"] == "dot" else list(d["arrays"]) + [d["dst"]])):
            raise ValueError("a loop over %d elements of a shorter buffer" % count)
        if d["kind"] == "dot":
            x, y = env[d["x"]][:count], env[d["y"]][:count]
            r = hip.dot_host(x, y, float(env[d["init"]]))
            return [numpy.float32(r) if x.element_size() == 4 else r]
        arrays = [env[a][:count] for a in d["arrays"]]
        self._elementwise(d["call"])(arrays, env[d["dst"]][:count], env)
        return None

    def _csr_for(self, pos, crd, val, nrows, ncols):
        """The Csr (and its plan) of a matrix given as three memrefs; kept while the same buffers come back."""
        key = (pos.data_ptr(), crd.data_ptr(), val.data_ptr(), nrows, ncols, int(crd.shape[0]))
        cache = self.__dict__.setdefault("_csr_cache", {})
        if key not in cache:
            for old in cache.values():
                old.release()
            cache.clear()
            cache[key] = Csr(pos, crd, val, nrows, ncols)
        return cache[key]

    def release(self):
        for A in self.__dict__.get("_csr_cache", {}).values():
            A.release()
        self.__dict__.get("_csr_cache", {}).clear()
