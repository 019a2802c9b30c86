"""What lapis_amd/schedule.py makes of a function gives the values the statements give one by one: the same modules run with
and without the entry points it fuses statements into (stand-ins on CPU tensors)."""
import types

import numpy as np
import pytest

import fake_hip
import modules_mlir as M
from test_executor_host_logic import csr, make, spd, vec
from lapis_amd import executor as ex
from lapis_amd import mlir_text as mt

import torch

_N = fake_hip._np


def _fused_hip():
    h = types.SimpleNamespace(**{k: getattr(fake_hip, k) for k in dir(fake_hip) if not k.startswith("__")})

    def overwrite(plan, nrows, ncols, pos, crd, val, x, y, stream=None):
        fake_hip.calls.append("spmv_overwrite")
        _N(y)[:] = fake_hip._matrix(nrows, ncols, pos, crd, val) @ _N(x)
        return y

    def dot_start(x, y, init=0.0, stream=None):
        fake_hip.calls.append("dot_start")
        return float(init + np.dot(_N(x).astype(np.float64), _N(y).astype(np.float64)))

    def axpby_dot_start(a, x, b, y, dst, z, init=0.0, stream=None):
        fake_hip.calls.append("axpby_dot_start")
        _N(dst)[:] = _N(x) * _N(x).dtype.type(a) + _N(y) * _N(y).dtype.type(b)
        return float(init + np.dot(_N(dst).astype(np.float64), _N(dst if z is None else z).astype(np.float64)))

    def spmv_dot_start(plan, nrows, ncols, pos, crd, val, x, y, init=0.0, stream=None):
        fake_hip.calls.append("spmv_dot_start")
        _N(y)[:] = fake_hip._matrix(nrows, ncols, pos, crd, val) @ _N(x)
        return float(init + np.dot(_N(x).astype(np.float64), _N(y).astype(np.float64)))

    def dot_finish(started):
        fake_hip.calls.append("dot_finish")
        return started
    h.__dict__.update(spmv_overwrite=overwrite, dot_start=dot_start, axpby_dot_start=axpby_dot_start,
                      spmv_dot_start=spmv_dot_start, dot_finish=dot_finish)
    return h


def _run(text, name, args, hip):
    e = ex.Executor(mt.Canonicalizer(text), torch_module=torch, hip_module=hip, device="cpu")
    fake_hip.calls.clear()
    return e.run(name, args()), list(fake_hip.calls)


A = spd(70, 8)
_rng = np.random.default_rng(8)
_x, _z, _d = _rng.standard_normal(70), _rng.standard_normal(70), 1.0 / A.diagonal()
CASES = {
    "residual": (M.SPMV_THEN_AXPBY, "residual", lambda: [csr(A), vec(_x), vec(_z), 0.75, -2.5]),
    "twice": (M.TWO_PRODUCTS, "twice_plus", lambda: [csr(A), vec(_x)]),
    "cg": (M.CG_FUSED_UPDATE, "cg", lambda: [csr(A), vec(_x), 1e-10, 40]),
    "richardson": (M.RICHARDSON, "richardson", lambda: [csr(A), vec(_x), vec(_z), 0.01, 5]),
    "pcg": (M.PCG, "pcg", lambda: [csr(A), vec(_x), vec(_d), 1e-10, 40]),
    "pcg_f32": (M.PCG_F32, "pcg", lambda: [csr(A, np.float32), vec(_x, np.float32), vec(_d, np.float32), np.float32(1e-4), 40]),
}


@pytest.mark.parametrize("name", CASES)
def test_same_values(name):
    text, fn, args = CASES[name]
    want, plain = _run(text, fn, args, fake_hip)
    got, fused = _run(text, fn, args, _fused_hip())
    assert len(got) == len(want)
    for g, w in zip(got, want):
        g, w = (np.asarray(t.numpy() if isinstance(t, torch.Tensor) else t) for t in (g, w))
        assert g.dtype == w.dtype and np.allclose(g, w, rtol=1e-6 if g.dtype == np.float32 else 1e-12, atol=1e-12)
    assert fused.count("dot_finish") == plain.count("dot") and len(fused) <= len(plain) + plain.count("dot")


def test_an_iteration_of_cg():
    text = M.CG_FUSED_UPDATE
    _, calls = _run(text, "cg", lambda: [csr(A), vec(_x), 0.0, 8], _fused_hip())
    at = [k for k, c in enumerate(calls) if c == "spmv_dot_start"]
    one = calls[at[3]:at[4]]
    # the product with its dot product; the new residual with its own, x while that is on its way; p
    assert sorted(one) == sorted(["spmv_dot_start", "dot_finish", "axpby_dot_start", "axpby", "dot_finish", "axpby"])
    assert one[2:5] == ["axpby_dot_start", "axpby", "dot_finish"]


def test_operands_that_a_delayed_operation_reads_are_kept():
    text = """
    #id = affine_map<(d0) -> (d0)>
    module {
      func.func @f(%a: tensor<?xf64>, %b: tensor<?xf64>) -> (tensor<?xf64>, f64, tensor<?xf64>) {
        %c0 = arith.constant 0 : index
        %z = arith.constant 0.0 : f64
        %n = tensor.dim %a, %c0 : tensor<?xf64>
        %e = tensor.empty(%n) : tensor<?xf64>
        %s = linalg.add ins(%a, %b : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %e2 = tensor.empty(%n) : tensor<?xf64>
        %t = linalg.sub ins(%s, %b : tensor<?xf64>, tensor<?xf64>) outs(%e2 : tensor<?xf64>) -> tensor<?xf64>
        %u = linalg.add ins(%s, %a : tensor<?xf64>, tensor<?xf64>) outs(%s : tensor<?xf64>) -> tensor<?xf64>
        %acc = tensor.splat %z[] : tensor<f64>
        %d = linalg.dot ins(%u, %u : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
        %v = tensor.extract %d[] : tensor<f64>
        return %t, %v, %u : tensor<?xf64>, f64, tensor<?xf64>
      }
    }"""
    for hip in (fake_hip, _fused_hip()):
        (t, v, u), _ = _run(text, "f", lambda: [vec(_x), vec(_z)], hip)
        assert np.allclose(t.numpy(), _x) and np.allclose(u.numpy(), 2 * _x + _z) and np.isclose(v, np.sum((2 * _x + _z) ** 2))


# Two names for one buffer: %a is a buffer of the function's own, %b another name for it that is read after an operation
# whose `outs` is %a.  Each text computes 2x as %a and 3x as %c, and returns %b + %c.
_SHARED = """
    module {
      func.func private @same(%%v: tensor<?xf64>) -> tensor<?xf64> {
        return %%v : tensor<?xf64>
      }
      func.func private @plus(%%u: tensor<?xf64>, %%v: tensor<?xf64>) -> tensor<?xf64> {
        %%s = linalg.add ins(%%u, %%v : tensor<?xf64>, tensor<?xf64>) outs(%%v : tensor<?xf64>) -> tensor<?xf64>
        return %%s : tensor<?xf64>
      }
      func.func @f(%%x: tensor<?xf64>, %%n: index, %%yes: i1) -> tensor<?xf64> {
        %%c0 = arith.constant 0 : index
        %%c1 = arith.constant 1 : index
        %%no = arith.constant false
        %%m = tensor.dim %%x, %%c0 : tensor<?xf64>
        %%e = tensor.empty(%%m) : tensor<?xf64>
        %%a = linalg.add ins(%%x, %%x : tensor<?xf64>, tensor<?xf64>) outs(%%e : tensor<?xf64>) -> tensor<?xf64>
        %(name)s
        %(plus)s
        %%g = tensor.empty(%%m) : tensor<?xf64>
        %%d = linalg.add ins(%%b, %%c : tensor<?xf64>, tensor<?xf64>) outs(%%g : tensor<?xf64>) -> tensor<?xf64>
        return %%d : tensor<?xf64>
      }
    }"""
_ANOTHER_NAME = {
    "call": "%b = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>",
    "calls of calls": """%b0 = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>
        %b = func.call @same(%b0) : (tensor<?xf64>) -> tensor<?xf64>""",
    "for without trips": """%b = scf.for %i = %c0 to %n step %c1 iter_args(%w = %a) -> (tensor<?xf64>) {
          %h = tensor.empty(%m) : tensor<?xf64>
          %k = linalg.add ins(%w, %x : tensor<?xf64>, tensor<?xf64>) outs(%h : tensor<?xf64>) -> tensor<?xf64>
          scf.yield %k : tensor<?xf64>
        }""",
    "for that yields its argument": """%b = scf.for %i = %c0 to %c1 step %c1 iter_args(%w = %a) -> (tensor<?xf64>) {
          scf.yield %w : tensor<?xf64>
        }""",
    "if": """%b = scf.if %yes -> (tensor<?xf64>) {
          scf.yield %a : tensor<?xf64>
        } else {
          scf.yield %x : tensor<?xf64>
        }""",
    "while": """%b = scf.while (%w = %a) : (tensor<?xf64>) -> (tensor<?xf64>) {
          %go = arith.andi %no, %yes : i1
          scf.condition(%go) %w : tensor<?xf64>
        } do {
        ^bb0(%w: tensor<?xf64>):
          scf.yield %w : tensor<?xf64>
        }""",
    "select": "%b = arith.select %yes, %a, %x : tensor<?xf64>",
}
_PLUS = {
    "direct": "%c = linalg.add ins(%x, %a : tensor<?xf64>, tensor<?xf64>) outs(%a : tensor<?xf64>) -> tensor<?xf64>",
    "in a call": "%c = func.call @plus(%x, %a) : (tensor<?xf64>, tensor<?xf64>) -> tensor<?xf64>",
}


@pytest.mark.parametrize("plus", _PLUS)
@pytest.mark.parametrize("name", _ANOTHER_NAME)
def test_a_buffer_with_two_names_is_not_overwritten_while_one_is_read(name, plus):
    text = _SHARED % {"name": _ANOTHER_NAME[name], "plus": _PLUS[plus]}
    for hip in (fake_hip, _fused_hip()):
        (d,), _ = _run(text, "f", lambda: [vec(_x), 0, True], hip)
        assert np.array_equal(d.numpy(), 2 * _x + (_x + 2 * _x))


def test_an_operation_moved_past_another_name_of_its_operand():
    # %c = x + %a, into %a's buffer, is launched between the dot product's start and its end, behind the call that names
    # %a once more
    text = """
    module {
      func.func private @same(%v: tensor<?xf64>) -> tensor<?xf64> {
        return %v : tensor<?xf64>
      }
      func.func @f(%x: tensor<?xf64>) -> (tensor<?xf64>, f64, tensor<?xf64>) {
        %c0 = arith.constant 0 : index
        %z = arith.constant 0.0 : f64
        %m = tensor.dim %x, %c0 : tensor<?xf64>
        %e = tensor.empty(%m) : tensor<?xf64>
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %c = linalg.add ins(%x, %a : tensor<?xf64>, tensor<?xf64>) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        %b = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>
        %acc = tensor.splat %z[] : tensor<f64>
        %d = linalg.dot ins(%b, %x : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
        %v = tensor.extract %d[] : tensor<f64>
        return %c, %v, %b : tensor<?xf64>, f64, tensor<?xf64>
      }
    }"""
    for hip in (fake_hip, _fused_hip()):
        (c, v, b), calls = _run(text, "f", lambda: [vec(_x)], hip)
        assert np.array_equal(c.numpy(), _x + 2 * _x) and np.array_equal(b.numpy(), 2 * _x) and np.isclose(v, 2 * np.sum(_x * _x))
    assert calls.index("dot_start") < len(calls) - 1 - calls[::-1].index("axpby") < calls.index("dot_finish")


# The `outs` operand is a buffer of the function's own that nothing mentions afterwards, and the operation needs its old
# elements when it has written new ones.
_NEEDED = {
    "product with its own output": """
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %p = linalg.matvec ins(%A, %a : tensor<?x?xf64, #CSR>, tensor<?xf64>) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        return %p, %z : tensor<?xf64>, f64""",
    "product into zeros of another name's buffer": """
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %b = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>
        %o = linalg.fill ins(%z : f64) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        %p = linalg.matvec ins(%A, %b : tensor<?x?xf64, #CSR>, tensor<?xf64>) outs(%o : tensor<?xf64>) -> tensor<?xf64>
        return %p, %z : tensor<?xf64>, f64""",
    "product and dot into zeros of another name's buffer": """
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %b = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>
        %o = linalg.fill ins(%z : f64) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        %p = linalg.matvec ins(%A, %b : tensor<?x?xf64, #CSR>, tensor<?xf64>) outs(%o : tensor<?xf64>) -> tensor<?xf64>
        %d = linalg.dot ins(%b, %p : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
        %v = tensor.extract %d[] : tensor<f64>
        return %p, %v : tensor<?xf64>, f64""",
    "sum and dot with what it overwrites": """
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %p = linalg.add ins(%a, %x : tensor<?xf64>, tensor<?xf64>) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        %d = linalg.dot ins(%p, %a : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
        %v = tensor.extract %d[] : tensor<f64>
        return %p, %v : tensor<?xf64>, f64""",
    "sum and dot with another name of what it overwrites": """
        %a = linalg.add ins(%x, %x : tensor<?xf64>, tensor<?xf64>) outs(%e : tensor<?xf64>) -> tensor<?xf64>
        %b = func.call @same(%a) : (tensor<?xf64>) -> tensor<?xf64>
        %p = linalg.add ins(%a, %x : tensor<?xf64>, tensor<?xf64>) outs(%a : tensor<?xf64>) -> tensor<?xf64>
        %d = linalg.dot ins(%b, %p : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
        %v = tensor.extract %d[] : tensor<f64>
        return %p, %v : tensor<?xf64>, f64""",
}


@pytest.mark.parametrize("name", _NEEDED)
def test_what_an_operation_needs_while_it_writes_is_not_its_output(name, monkeypatch):
    text = """
    #CSR = #sparse_tensor.encoding<{ map = (d0, d1) -> (d0 : dense, d1 : compressed), posWidth = 32, crdWidth = 32 }>
    module {
      func.func private @same(%%v: tensor<?xf64>) -> tensor<?xf64> {
        return %%v : tensor<?xf64>
      }
      func.func @f(%%A: tensor<?x?xf64, #CSR>, %%x: tensor<?xf64>) -> (tensor<?xf64>, f64) {
        %%c0 = arith.constant 0 : index
        %%z = arith.constant 0.0 : f64
        %%m = tensor.dim %%x, %%c0 : tensor<?xf64>
        %%acc = tensor.splat %%z[] : tensor<f64>
        %%e = tensor.empty(%%m) : tensor<?xf64>
        %s
      }
    }""" % _NEEDED[name].strip()
    a = 2 * _x
    p = A @ a + a if name.endswith("its own output") else A @ a if name.startswith("product") else a + _x
    v = np.dot(a, p) if "dot" in name else 0.0
    for hip in (fake_hip, _fused_hip()):
        written = []  # the stand-ins read all of x before they write y, which a kernel does not: no shared buffer
        for fn in ("spmv", "spmv_overwrite", "spmv_dot_start"):
            if hasattr(hip, fn):
                def check(plan, nrows, ncols, pos, crd, val, x, y, *more, was=getattr(hip, fn)):
                    written.append((x.data_ptr(), y.data_ptr()))
                    return was(plan, nrows, ncols, pos, crd, val, x, y, *more)
                monkeypatch.setattr(hip, fn, check)
        (got, w), _ = _run(text, "f", lambda: [csr(A), vec(_x)], hip)
        assert np.allclose(got.numpy(), p, rtol=1e-13) and np.isclose(w, v, rtol=1e-13)
        assert all(x != y for x, y in written) and bool(written) == name.startswith("product")
