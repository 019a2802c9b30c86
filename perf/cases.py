"""The workloads this library is measured on: CSR SpMV, CSR x dense SpMM, the batched CSRV product, conjugate
gradients, and the generated-module boundary that takes host arrays.

A case is a dict of plain values.  ``listed()`` names the fixed ones, ``draw(rng)`` gives another case of the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call (operands on the device, the plan, the
compiled module), ``run(state)`` is one pass through the public entry points, ``work(case)`` the bytes and
floating-point operations of a pass, ``tolerance(case)`` how far another correct implementation may be off.

Matrix structures (``matrix``):
  grid2d    5-point Laplacian on an nx x nx grid
  grid3d    7-point Laplacian on an nx^3 grid
  fem       3-D elasticity: 27-point node stencil on nx^3 nodes, 3 unknowns per node (81 entries in a full row)
  random    row lengths Poisson(mean), uniformly random distinct columns
  powerlaw  row lengths with an exponent-2 power law of the given mean, capped at n / 10, random columns
"""
import math

import numpy as np
import torch

from lapis_amd import KokkosBackend, hip

_MAX_NNZ = 67_200_000       # entries of the largest matrix
_MAX_DENSE = 67_200_000     # elements of the largest dense operand
_MAX_GATHERED = 2.2e9       # entries x columns of B of the largest SpMM

# A module a user writes in the vocabulary of the front door: the product behind the generated-module boundary.
_SPMV_TEXT = """
#CSR = #sparse_tensor.encoding<{ map = (d0, d1) -> (d0 : dense, d1 : compressed), posWidth = 32, crdWidth = 32 }>
module {
  func.func @spmv(%A: tensor<?x?x{T}, #CSR>, %x: tensor<?x{T}>, %y: tensor<?x{T}>) -> tensor<?x{T}> {
    %0 = linalg.matvec ins(%A, %x: tensor<?x?x{T}, #CSR>, tensor<?x{T}>) outs(%y : tensor<?x{T}>) -> tensor<?x{T}>
    return %0 : tensor<?x{T}>
  }
}"""

# Conjugate gradients as a user's own function: not one of the prebuilt whole functions, so it runs by operation.
_CG_TEXT = """
#CSR = #sparse_tensor.encoding<{ map = (d0, d1) -> (d0 : dense, d1 : compressed), posWidth = 32, crdWidth = 32 }>
#id = affine_map<(d0) -> (d0)>
module {
  func.func private @inner(%a: tensor<?xf64>, %b: tensor<?xf64>) -> f64 {
    %c = arith.constant 0.0 : f64
    %acc = tensor.splat %c[] : tensor<f64>
    %d = linalg.dot ins(%a, %b : tensor<?xf64>, tensor<?xf64>) outs(%acc : tensor<f64>) -> tensor<f64>
    %s = tensor.extract %d[] : tensor<f64>
    return %s : f64
  }
  func.func @cg(%A: tensor<?x?xf64, #CSR>, %b: tensor<?xf64>, %tol: f64, %maxiter: index) -> (tensor<?xf64>, index, f64) {
    %c0 = arith.constant 0 : index
    %c1 = arith.constant 1 : index
    %f0 = arith.constant 0.0 : f64
    %n = tensor.dim %b, %c0 : tensor<?xf64>
    %x0 = tensor.splat %f0[%n] : tensor<?xf64>
    %e0 = tensor.empty(%n) : tensor<?xf64>
    %p0 = linalg.copy ins(%b : tensor<?xf64>) outs(%e0 : tensor<?xf64>) -> tensor<?xf64>
    %bb = func.call @inner(%b, %b) : (tensor<?xf64>, tensor<?xf64>) -> f64
    %bnorm = math.sqrt %bb : f64
    %x, %r, %p, %rr, %its = scf.while (%xi = %x0, %ri = %b, %pi = %p0, %rri = %bb, %i = %c0)
        : (tensor<?xf64>, tensor<?xf64>, tensor<?xf64>, f64, index) -> (tensor<?xf64>, tensor<?xf64>, tensor<?xf64>, f64, index) {
      %nrm = math.sqrt %rri : f64
      %rel = arith.divf %nrm, %bnorm : f64
      %open = arith.cmpf ogt, %rel, %tol : f64
      %more = arith.cmpi slt, %i, %maxiter : index
      %go = arith.andi %open, %more : i1
      scf.condition(%go) %xi, %ri, %pi, %rri, %i : tensor<?xf64>, tensor<?xf64>, tensor<?xf64>, f64, index
    } do {
    ^bb0(%xi: tensor<?xf64>, %ri: tensor<?xf64>, %pi: tensor<?xf64>, %rri: f64, %i: index):
      %e1 = tensor.empty(%n) : tensor<?xf64>
      %z = linalg.fill ins(%f0 : f64) outs(%e1 : tensor<?xf64>) -> tensor<?xf64>
      %Ap = linalg.matvec ins(%A, %pi : tensor<?x?xf64, #CSR>, tensor<?xf64>) outs(%z : tensor<?xf64>) -> tensor<?xf64>
      %pAp = func.call @inner(%pi, %Ap) : (tensor<?xf64>, tensor<?xf64>) -> f64
      %alpha = arith.divf %rri, %pAp : f64
      %xn = linalg.generic {indexing_maps = [#id, #id], iterator_types = ["parallel"]}
          ins(%pi : tensor<?xf64>) outs(%xi : tensor<?xf64>) {
        ^bb0(%pe: f64, %xe: f64):
          %t = arith.mulf %alpha, %pe : f64
          %u = arith.addf %xe, %t : f64
          linalg.yield %u : f64
      } -> tensor<?xf64>
      %e2 = tensor.empty(%n) : tensor<?xf64>
      %rn = linalg.generic {indexing_maps = [#id, #id, #id], iterator_types = ["parallel"]}
          ins(%ri, %Ap : tensor<?xf64>, tensor<?xf64>) outs(%e2 : tensor<?xf64>) {
        ^bb0(%re: f64, %ae: f64, %oe: f64):
          %t = arith.mulf %alpha, %ae : f64
          %u = arith.subf %re, %t : f64
          linalg.yield %u : f64
      } -> tensor<?xf64>
      %rrn = func.call @inner(%rn, %rn) : (tensor<?xf64>, tensor<?xf64>) -> f64
      %beta = arith.divf %rrn, %rri : f64
      %pn = linalg.generic {indexing_maps = [#id, #id], iterator_types = ["parallel"]}
          ins(%rn : tensor<?xf64>) outs(%pi : tensor<?xf64>) {
        ^bb0(%re: f64, %pe: f64):
          %t = arith.mulf %beta, %pe : f64
          %u = arith.addf %re, %t : f64
          linalg.yield %u : f64
      } -> tensor<?xf64>
      %in = arith.addi %i, %c1 : index
      scf.yield %xn, %rn, %pn, %rrn, %in : tensor<?xf64>, tensor<?xf64>, tensor<?xf64>, f64, index
    }
    %nrm = math.sqrt %rr : f64
    %relres = arith.divf %nrm, %bnorm : f64
    return %x, %its, %relres : tensor<?xf64>, index, f64
  }
}"""


def listed():
    return [
        # y += A x with a plan kept over many products.  The smallest: a cache-resident 2-D grid, where the call itself counts.
        {"name": "spmv_grid2d_256_f64", "kind": "spmv", "matrix": "grid2d", "nx": 256, "dtype": "f64"},
        # The two matrices of the reference's published SpMV table whose structure is a formula.
        {"name": "spmv_grid3d_100_f64", "kind": "spmv", "matrix": "grid3d", "nx": 100, "dtype": "f64"},
        {"name": "spmv_fem_60_f64", "kind": "spmv", "matrix": "fem", "nx": 60, "dtype": "f64"},
        # The headline configuration: columns all over a vector that no cache level near the cores holds.
        {"name": "spmv_random_4m_f64", "kind": "spmv", "matrix": "random", "n": 4194304, "mean": 16.0, "dtype": "f64"},
        # Graph-like rows between 1 and 200 000 entries, in single precision.
        {"name": "spmv_powerlaw_2m_f32", "kind": "spmv", "matrix": "powerlaw", "n": 2097152, "mean": 30.0, "dtype": "f32"},
        # C += A B: a block of dense vectors against a matrix without locality, the benchmark's shape ...
        {"name": "spmm_random_1m_k64_f32", "kind": "spmm", "matrix": "random", "n": 1048576, "mean": 32.0, "k": 64, "dtype": "f32"},
        # ... and a handful of right-hand sides (no power of two) against a grid operator in double precision.
        {"name": "spmm_grid3d_97_k10_f64", "kind": "spmm", "matrix": "grid3d", "nx": 97, "k": 10, "dtype": "f64"},
        # Sparse attention weights with a batch of heads times dense values (the batched CSRV product).
        {"name": "bspmm_16k_f32", "kind": "bspmm", "n": 16384, "mean": 32.0, "dh": 32, "nh": 8, "dtype": "f32"},
        # Unpreconditioned CG on a large 3-D grid, exactly 100 iterations.
        {"name": "cg_grid3d_192_f64", "kind": "cg", "nx": 192, "dtype": "f64"},
        # Jacobi-preconditioned CG to a tolerance on a small 2-D problem: bound by launches and scalars.
        {"name": "pcg_grid2d_128_f64", "kind": "pcg", "nx": 128, "dtype": "f64"},
        # The generated-module boundary: host arrays in, host arrays out, one product per call.
        {"name": "module_spmv_grid3d_64_f64", "kind": "module_spmv", "nx": 64, "dtype": "f64"},
        # A user's own CG function compiled from module text and run operation by operation on host arrays.
        {"name": "compiled_cg_grid2d_100_f64", "kind": "compiled_cg", "nx": 100, "iterations": 40, "dtype": "f64"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_matrix(rng, kinds, small=1.0):
    """A matrix of one of the structures, from a thousand rows or so to ``small`` times the largest listed size."""
    matrix = rng.choice(kinds)
    if matrix == "grid2d":
        return {"matrix": matrix, "nx": _log_int(rng, 24, int(2048 * small ** 0.5))}
    if matrix == "grid3d":
        return {"matrix": matrix, "nx": _log_int(rng, 10, int(192 * small ** (1 / 3)))}
    if matrix == "fem":
        return {"matrix": matrix, "nx": _log_int(rng, 6, int(60 * small ** (1 / 3)))}
    mean = round(math.exp(rng.uniform(math.log(6.0), math.log(64.0))), 1) if matrix == "random" else round(rng.uniform(12.0, 40.0), 1)
    top = 4194304 if matrix == "random" else 2097152
    return {"matrix": matrix, "n": _log_int(rng, 1500, int(min(top, _MAX_NNZ / (1.1 * mean)) * small)), "mean": mean}


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "spmv", "spmv", "spmm", "spmm", "bspmm", "cg", "pcg", "module_spmv", "compiled_cg"])
    dtype = rng.choice(["f64", "f32"])
    if kind == "spmv":
        return dict({"kind": kind, "dtype": dtype}, **_draw_matrix(rng, ["grid2d", "grid3d", "fem", "random", "powerlaw"]))
    if kind == "spmm":
        case = dict({"kind": kind, "dtype": dtype}, **_draw_matrix(rng, ["grid3d", "fem", "random"], 0.25))
        rows, nnz = _size(case)
        case["k"] = _log_int(rng, 2, max(2, int(min(128, _MAX_DENSE / rows, _MAX_GATHERED / nnz))))
        return case
    if kind == "bspmm":
        n, mean, nh = _log_int(rng, 300, 65536), round(rng.uniform(6.0, 64.0), 1), _log_int(rng, 1, 16)
        return {"kind": kind, "n": n, "mean": mean, "nh": nh, "dtype": "f32",
                "dh": _log_int(rng, 4, max(4, int(min(128, _MAX_DENSE / (n * nh), 1.0e9 / (n * mean * nh)))))}
    if kind == "cg":
        return {"kind": kind, "nx": _log_int(rng, 32, 191), "dtype": "f64"}
    if kind == "pcg":
        return {"kind": kind, "nx": _log_int(rng, 32, 1024), "dtype": "f64"}
    if kind == "module_spmv":
        return {"kind": kind, "nx": _log_int(rng, 8, 128), "dtype": dtype}
    return {"kind": kind, "nx": _log_int(rng, 16, 256), "iterations": rng.randint(10, 60), "dtype": "f64"}


# ---- inputs -------------------------------------------------------------------------------------------------

def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(seed)


def _uniform(g, shape, dtype, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=g, dtype=dtype, device="cuda") * (hi - lo) + lo


def _positions(lengths):
    pos = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=pos[1:])
    if int(pos[-1]) >= 2 ** 31:
        raise ValueError("the matrix has more entries than 32-bit positions hold")
    return pos.to(torch.int32)


def _grid(nx, offsets, g, dtype, diagonal, unknowns=1):
    """Stencil matrix over a grid with x fastest: ``offsets`` are (dx, dy[, dz]) in ascending column order; off-diagonal
    entries -1, ``diagonal`` on the diagonal (a number, or None: the row's other entries in absolute value plus
    a positive random shift).  ``unknowns`` > 1: that many rows per node, a full block per node pair."""
    dims = len(offsets[0])
    n = nx ** dims
    index = torch.arange(n, dtype=torch.int32, device="cuda")
    at = [(index // nx ** d) % nx for d in range(dims)]
    columns = torch.empty((n, len(offsets)), dtype=torch.int32, device="cuda")
    inside = torch.empty((n, len(offsets)), dtype=torch.bool, device="cuda")
    for j, offset in enumerate(offsets):
        ok = torch.ones(n, dtype=torch.bool, device="cuda")
        for d, o in enumerate(offset):
            if o:
                ok &= (at[d] + o >= 0) & (at[d] + o < nx)
        inside[:, j] = ok
        columns[:, j] = index + sum(o * nx ** d for d, o in enumerate(offset))
    per_node = inside.sum(1)
    if unknowns > 1:
        u = torch.arange(unknowns, dtype=torch.int32, device="cuda")
        columns = (columns[:, None, :, None] * unknowns + u).expand(n, unknowns, len(offsets), unknowns).reshape(n * unknowns, -1)
        inside = inside[:, None, :, None].expand(n, unknowns, len(offsets), unknowns).reshape(n * unknowns, -1)
        per_node = (per_node * unknowns).repeat_interleave(unknowns)
    rows = n * unknowns
    crd = columns[inside]
    row_of = torch.arange(rows, dtype=torch.int32, device="cuda").repeat_interleave(per_node, output_size=crd.numel())
    on_diagonal = crd == row_of
    val = torch.full((crd.numel(),), -1.0, dtype=dtype, device="cuda")
    if diagonal is None:
        val[on_diagonal] = (2.0 * dims) + torch.rand(rows, generator=g, dtype=dtype, device="cuda")
    else:
        val[on_diagonal] = diagonal
    return rows, _positions(per_node), crd, val


_STENCIL2 = [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)]
_STENCIL3 = [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
_STENCIL27 = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]


def _powerlaw_lengths(n, mean, g):
    """Lengths with P(K >= k) = (q + 1) / (k + q), capped at n / 10; q gives the expected length ``mean``."""
    cap = max(64, n // 10)
    lo, hi = 0.0, 64.0
    for _ in range(60):
        q = 0.5 * (lo + hi)
        lo, hi = (q, hi) if (q + 1.0) * math.log((cap + q + 0.5) / (q + 0.5)) < mean else (lo, q)
    u = 1.0 - torch.rand(n, generator=g, dtype=torch.float64, device="cuda")
    return torch.floor((q + 1.0) / u - q).clamp_(1, cap).to(torch.int64)


def _random(n, lengths, g, dtype):
    """Distinct ascending random columns: sorted draws with repetition from [0, n - length], plus their rank in the row."""
    lengths = lengths.clamp(max=n)
    pos = _positions(lengths)
    nnz = int(pos[-1])
    row_of = torch.arange(n, dtype=torch.int64, device="cuda").repeat_interleave(lengths, output_size=nnz)
    key = (torch.rand(nnz, generator=g, dtype=torch.float64, device="cuda") * (n - lengths + 1)[row_of]).to(torch.int64)
    bits = max(1, (n - 1).bit_length())
    key = torch.sort(key | (row_of << bits)).values
    rank = torch.arange(nnz, dtype=torch.int64, device="cuda") - pos[:-1].to(torch.int64)[row_of]
    crd = ((key & ((1 << bits) - 1)) + rank).to(torch.int32)
    del key, rank, row_of
    val = torch.randn(nnz, generator=g, dtype=dtype, device="cuda") if dtype == torch.float32 else _uniform(g, nnz, dtype)
    return n, pos, crd, val


def _matrix(case, g):
    """(rows, positions, coordinates, values) on the device; all structures are square."""
    dtype, matrix = _dtype(case), case["matrix"]
    if matrix == "grid2d":
        return _grid(case["nx"], _STENCIL2, g, dtype, 4.0)
    if matrix == "grid3d":
        return _grid(case["nx"], _STENCIL3, g, dtype, 6.0)
    if matrix == "fem":
        return _grid(case["nx"], _STENCIL27, g, dtype, 100.0, unknowns=3)
    n = case["n"]
    if matrix == "random":
        lengths = torch.poisson(torch.full((n,), case["mean"], device="cuda"), generator=g).to(torch.int64)
    else:
        lengths = _powerlaw_lengths(n, case["mean"], g)
    return _random(n, lengths, g, dtype)


def _size(case):
    """(rows, expected entries) of the case's matrix."""
    nx = case.get("nx", 0)
    matrix = case.get("matrix", "grid3d" if case["kind"] in ("cg", "module_spmv") else "grid2d")
    if case["kind"] == "bspmm" or matrix in ("random", "powerlaw"):
        return case["n"], case["n"] * min(case["mean"], case["n"])
    if matrix == "grid2d":
        return nx ** 2, 5 * nx ** 2 - 4 * nx
    if matrix == "grid3d":
        return nx ** 3, 7 * nx ** 3 - 6 * nx ** 2
    return 3 * nx ** 3, 9 * (3 * nx - 2) ** 3


# ---- one pass -----------------------------------------------------------------------------------------------

def prepare(case, seed):
    g = _generator(seed)
    kind, dtype = case["kind"], _dtype(case)
    state = {"kind": kind}
    if kind in ("spmv", "spmm"):
        n, pos, crd, val = _matrix(case, g)
        plan = hip.CsrPlan(n, n, pos, crd, value_bytes=val.element_size())
        if kind == "spmv":
            plan.analyze(crd, val)  # the matrix will be multiplied many times: the library may lay it out anew
            state.update(x=_uniform(g, n, dtype), y=torch.zeros(n, dtype=dtype, device="cuda"))
        else:
            state.update(B=_uniform(g, (n, case["k"]), dtype), C=torch.zeros((n, case["k"]), dtype=dtype, device="cuda"))
        state.update(plan=plan, n=n, pos=pos, crd=crd, val=val)
    elif kind == "bspmm":
        n, dh, nh = case["n"], case["dh"], case["nh"]
        lengths = torch.poisson(torch.full((n,), case["mean"], device="cuda"), generator=g).to(torch.int64)
        _, pos, crd, _ = _random(n, lengths, g, dtype)
        state.update(n=n, pos=pos, crd=crd, val=torch.rand(crd.numel() * nh, generator=g, dtype=dtype, device="cuda"),
                     V=_uniform(g, (n, dh, nh), dtype), out=torch.zeros((n, dh, nh), dtype=dtype, device="cuda"))
    elif kind in ("cg", "pcg"):
        if kind == "cg":
            n, pos, crd, val = _grid(case["nx"], _STENCIL3, g, dtype, 6.0)
            dinv, tol, maxiter = None, 0.0, 100
        else:
            n, pos, crd, val = _grid(case["nx"], _STENCIL2, g, dtype, None)
            row_of = torch.arange(n, dtype=torch.int32, device="cuda").repeat_interleave(torch.diff(pos), output_size=crd.numel())
            dinv, tol, maxiter = 1.0 / val[crd == row_of], 1e-8, 1000
        plan = hip.CsrPlan(n, n, pos, crd)
        plan.analyze(crd, val)
        state.update(plan=plan, n=n, pos=pos, crd=crd, val=val, b=_uniform(g, n, dtype, 0.0, 1.0), dinv=dinv, tol=tol,
                     maxiter=maxiter, x=torch.empty(n, dtype=dtype, device="cuda"),
                     work=torch.empty(4 * n, dtype=dtype, device="cuda"))
    else:
        stencil = _STENCIL3 if kind == "module_spmv" else _STENCIL2
        n, pos, crd, val = _grid(case["nx"], stencil, g, dtype, 2.0 * len(stencil[0]))
        b = _uniform(g, n, dtype)
        backend = KokkosBackend.KokkosBackend(decompose_tensors=True)
        text = _SPMV_TEXT.replace("{T}", case["dtype"]) if kind == "module_spmv" else _CG_TEXT
        nnz = int(crd.numel())
        state.update(module=backend.compile(text), pos=pos.cpu().numpy(), crd=crd.cpu().numpy(), val=val.cpu().numpy(),
                     spec=((n, n), (n + 1, nnz, nnz)), b=b.cpu().numpy(), y=np.zeros(n, dtype=val.cpu().numpy().dtype),
                     iterations=case.get("iterations"))
    return state


def run(state):
    s, kind = state, state["kind"]
    if kind == "spmv":
        return hip.spmv(s["plan"], s["n"], s["n"], s["pos"], s["crd"], s["val"], s["x"], s["y"])
    if kind == "spmm":
        return hip.spmm(s["n"], s["n"], s["pos"], s["crd"], s["val"], s["B"], s["C"], plan=s["plan"])
    if kind == "bspmm":
        return hip.bspmm_csrv(s["n"], s["n"], s["pos"], s["crd"], s["val"], s["V"], s["out"])
    if kind in ("cg", "pcg"):
        iterations, relres = hip.pcg(s["plan"], s["n"], s["pos"], s["crd"], s["val"], s["b"], s["dinv"], s["tol"],
                                     s["maxiter"], s["x"], work=s["work"])
        return s["x"], iterations, relres
    if kind == "module_spmv":
        return s["module"].spmv(s["pos"], s["crd"], s["val"], s["spec"], s["b"], s["y"])
    x, iterations, relres = s["module"].cg(s["pos"], s["crd"], s["val"], s["spec"], s["b"], 0.0, s["iterations"])
    return x, int(iterations), float(relres)


def work(case):
    n, nnz = _size(case)
    w = 8 if case["dtype"] == "f64" else 4
    matrix = nnz * (4 + w) + 4 * (n + 1)
    kind = case["kind"]
    if kind in ("spmv", "module_spmv"):
        return {"bytes": matrix + 3 * w * n, "flops": 2 * nnz}  # x read, y read and written
    if kind == "spmm":
        return {"bytes": matrix + 3 * w * n * case["k"], "flops": 2 * nnz * case["k"]}
    if kind == "bspmm":
        dense = n * case["dh"] * case["nh"]
        return {"bytes": nnz * (4 + 4 * case["nh"]) + 4 * (n + 1) + 3 * 4 * dense, "flops": 2 * nnz * case["dh"] * case["nh"]}
    # per iteration: the matrix, p read and Ap written by the product; Ap and r read, r written; r, p and x read,
    # p and x written; with a preconditioner also dinv read and z written and read
    iterations = {"cg": 100, "pcg": 41}.get(kind) or case["iterations"]
    vectors = 10 + (3 if kind == "pcg" else 0)
    return {"bytes": iterations * (matrix + vectors * w * n), "flops": iterations * (2 * nnz + 10 * n)}


def tolerance(case):
    if case["kind"] == "pcg":
        # the residual has fallen by 1e-8: what is left of it carries rounding errors that much larger than the vectors' own
        return {"rel": 1e-7}
    if case["kind"] in ("cg", "compiled_cg"):
        return {"rel": 1e-10}  # up to a hundred steps on sums taken in another order
    return {"rel": 1e-12} if case["dtype"] == "f64" else {"rel": 1e-5}
