"""Rewrites a function's statements before the executor turns them into steps, for fewer launches and waits.

A statement costs a launch (about 4 us of the host's time, as much of the GPU's on small vectors), and a `linalg.dot`
stops the host until the GPU has caught up.  On tensors, which no operation changes in place as far as the text can
tell, these rewrites give the same values:

* calls of the module's own functions are inlined, so that the rest sees a call's `linalg.dot`;
* a product into a zero-filled tensor becomes one that does not read its output (no fill);
* a product or an elementwise operation followed by a dot product with its result becomes one launch that computes
  both (`lapis.product_dot`, `lapis.elementwise_dot`);
* a dot product is split into its launch (`lapis.dot_start` or one of the two above) and the wait for its value
  (`lapis.dot_finish`), and elementwise operations whose results nothing needs before the wait are launched between.

Statements that work on memrefs stay in order, and so does everything around them.
"""
import re

from . import mlir_text as _mt

NAME = re.compile(r"%[\w.$-]+(?:#\d+)?")
_BASE = re.compile(r"%[\w.$-]+")
_HOST_ONLY = re.compile(r"arith\.|math\.|lapis\.alias$|tensor\.(?:empty|dim|splat|extract)$")
_ELEMENTWISE_NAMED = ("linalg.add", "linalg.sub")


class Fused:
    """A statement made of statements: `op` names what it does, `parts` are the originals."""

    def __init__(self, op, results, parts, **more):
        self.op, self.results, self.parts = op, results, parts
        self.head, self.regions = "", []
        self.__dict__.update(more)


def mentions(s, out=None):
    """Names a statement mentions, in its operands or in its regions."""
    out = set() if out is None else out
    if isinstance(s, Fused):
        for p in s.parts:
            mentions(p, out)
        out.update(getattr(s, "uses", ()))
        return out
    out.update(NAME.findall(s.head))
    for _, sub in s.regions:
        for t in sub:
            mentions(t, out)
    return out


def result_names(s):
    names = []
    for r in s.results:
        base, _, count = r.partition(":")
        names += ["%s#%d" % (base, j) for j in range(int(count))] if count else [base]
    return names


def buffers(stmts, fresh, scalar):
    """For every name that `stmts`, (statement, names it mentions) in order, define: the names whose buffers it may be.
    `fresh(statement)`: its results are buffers of their own; `scalar(statement)`: its results hold no buffer.  What any
    other statement gives (a call, a loop or branch that may pass an operand through, another name for a value) may be any
    buffer it mentions."""
    of = {}
    for s, said in stmts:
        shared = set() if fresh(s) or scalar(s) else set().union(*(of.get(n, (n,)) for n in said))
        for n in result_names(s):
            of[n] = shared | {n}
    return of


# ---- inlining ----------------------------------------------------------------------------------------------

def _renamed(stmts, rename):
    sub = lambda text: _BASE.sub(lambda m: rename(m.group(0)), text)
    return [_mt.Statement([sub(r) for r in s.results], s.op, sub(s.head),
                          [([sub(a) for a in bargs], _renamed(inner, rename)) for bargs, inner in s.regions]) for s in stmts]


def inline(stmts, function_of, inside, counter):
    """The statements with calls replaced by the callees' statements.  `function_of(name)` gives (argument names,
    statements), or None for a function that is to be called as it is; `inside` names the functions under way."""
    out = []
    for s in stmts:
        m = re.search(r"@([\w$.-]+)", s.head) if s.op in ("func.call", "call") else None
        callee = function_of(m.group(1)) if m and m.group(1) not in inside else None
        if callee is not None:
            args, body = callee
            i = s.head.index("(")
            given = NAME.findall(s.head[i:_mt._match(s.head, i)])
            last = body[-1] if body else None
            if len(given) == len(args) and last is not None and last.op in ("return", "func.return") and \
                    not any("#" in g for g in given):
                counter[0] += 1
                to, prefix = dict(zip(args, given)), "%%%s.%d." % (m.group(1), counter[0])
                copy = _renamed(body, lambda nm: to.get(nm) or prefix + nm[1:])
                out += inline(copy[:-1], function_of, inside | {m.group(1)}, counter)
                returned = NAME.findall(copy[-1].head.split(":")[0])
                for name, value in zip(result_names(s), returned):
                    out.append(_mt.Statement([name], "lapis.alias", value, []))
                continue
        if s.regions:
            s = _mt.Statement(s.results, s.op, s.head, [(b, inline(sub, function_of, inside, counter)) for b, sub in s.regions])
        out.append(s)
    return out


# ---- fusing and moving -------------------------------------------------------------------------------------

def _host_only(s):
    """Does the statement leave the GPU alone (and yield results)?"""
    if isinstance(s, Fused) or not s.results or s.regions or not _HOST_ONLY.match(s.op):
        return False
    return s.op not in ("tensor.splat", "tensor.extract") or _zero_dimensional(s)


def _zero_dimensional(s):
    return re.search(r"tensor<(?:f64|f32)>\s*$", s.head) is not None


def _ins(s):
    m = re.search(r"\bins\s*\(", s.head)
    if not m:
        return []
    i = m.end() - 1
    return NAME.findall(s.head[i + 1:_mt._match(s.head, i) - 1].split(":")[0])


def _outs(s):
    m = re.search(r"\bouts\s*\(", s.head)
    if not m:
        return []
    i = m.end() - 1
    return NAME.findall(s.head[i + 1:_mt._match(s.head, i) - 1].split(":")[0])


def rewrite(stmts, kind_of, constants):
    """`kind_of(statement)`: "product" (CSR matrix times vector), "axpby" (elementwise a*x + b*y, a*x or a copy) or None.
    `constants`: values of the `arith.constant`s in sight."""
    kinds = {id(s): kind_of(s) for s in stmts if s.results}
    kind = lambda s: kinds.get(id(s)) if not isinstance(s, Fused) else None
    pure = lambda s: _host_only(s) or kind(s) is not None or (s.op in ("linalg.dot", "linalg.fill", "linalg.copy") and s.results) \
        or isinstance(s, Fused)
    stmts = _products_without_fill(stmts, kind, constants)
    stmts = _pair_with_dots(stmts, kind, pure)
    return _launch_before_waits(stmts, kind, pure)


def _products_without_fill(stmts, kind, constants):
    seen = {}
    for s in stmts:
        for n in mentions(s):
            seen[n] = seen.get(n, 0) + 1
    by_name, drop, out = {}, set(), []
    for s in stmts:
        if s.op == "linalg.fill" and s.results:
            by_name[s.results[0]] = s
        fill = by_name.get(_outs(s)[0]) if kind(s) == "product" and len(_outs(s)) == 1 else None
        if fill is not None and seen[fill.results[0]] == 1 and len(_ins(fill)) == 1 and \
                constants.get(_ins(fill)[0]) == 0.0 and _outs(fill)[0] not in _ins(s):
            drop.add(id(fill))
            out.append(Fused("lapis.product", s.results, [s], outs=_outs(fill)[0], uses={_outs(fill)[0]}))
        else:
            out.append(s)
    return [s for s in out if id(s) not in drop]


def _pair_with_dots(stmts, kind, pure):
    stmts = list(stmts)
    k = 0
    while k < len(stmts):
        s = stmts[k]
        product = isinstance(s, Fused) and s.op == "lapis.product"
        if product or kind(s) == "axpby":
            result = s.results[0]
            for j in range(k + 1, len(stmts)):
                t = stmts[j]
                if t.op == "linalg.dot" and t.results and _zero_dimensional(t):
                    if len(_ins(t)) != 2:
                        break
                    a, b = _ins(t)
                    x = _ins(s.parts[0])[1] if product else None
                    if (product and sorted([a, b]) == sorted([x, result])) or (not product and result in (a, b)):
                        other = None if a == b else (b if a == result else a)
                        stmts[j] = Fused("lapis.product_dot" if product else "lapis.elementwise_dot", s.results, [s, t], other=other)
                        del stmts[k]
                        k -= 1
                    break
                if result in mentions(t) or not pure(t):
                    break
        k += 1
    return stmts


def _launch_before_waits(stmts, kind, pure):
    out = []
    for s in stmts:
        if isinstance(s, Fused) and s.op.endswith("_dot"):
            out += [s, Fused("lapis.dot_finish", s.parts[1].results, [], start=s)]
        elif s.op == "linalg.dot" and s.results and _zero_dimensional(s):
            start = Fused("lapis.dot_start", [], [s])
            out += [start, Fused("lapis.dot_finish", s.results, [], start=start)]
        else:
            out.append(s)
    # from the back: an elementwise operation goes between the next launch of a dot product and its wait
    for k in range(len(out) - 1, -1, -1):
        s = out[k]
        if kind(s) != "axpby":
            continue
        result, j = s.results[0], k + 1
        while j < len(out) and pure(out[j]) and result not in mentions(out[j]):
            if out[j].op == "lapis.dot_finish":
                out.insert(j, s)
                del out[k]
                break
            j += 1
    return out
