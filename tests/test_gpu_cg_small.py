"""The one-launch CG of systems that fit the chip's LDS, at the edges of its rows per workgroup and per thread, against
the oracle; a solve that outlives one launch; and the way back to the many-launch solve when a wait runs out."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from gpu_util import dev

pytestmark = pytest.mark.gpu


def _spd(n, per_row, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    k = max(1, min(n, per_row) // 2)
    R = sp.csr_matrix((rng.random(n * k), rng.integers(0, n, n * k), np.arange(0, n * k + 1, k)), shape=(n, n))
    S = R + R.T
    A = sp.csr_matrix(S + sp.diags(np.asarray(abs(S).sum(axis=1)).ravel() + 0.5 + rng.random(n)))
    A.sum_duplicates()
    A.sort_indices()
    return A, rng


def _solve(gpu, A, b, dinv, tol, maxiter):
    n = b.shape[0]
    pos, crd = dev(A.indptr.astype(np.int32)), dev(A.indices.astype(np.int32))
    plan = gpu.CsrPlan(n, n, pos, crd)
    x = torch.full((n,), 7.0, dtype=torch.float64, device="cuda")
    iters, relres = gpu.pcg(plan, n, pos, crd, dev(A.data), dev(b), None if dinv is None else dev(dinv), tol, maxiter, x)
    return x.cpu().numpy(), iters, relres


@pytest.mark.parametrize("preconditioned", [False, True])
@pytest.mark.parametrize("n,per_row", [(1, 1), (2, 2), (63, 6), (511, 6), (512, 6), (513, 6), (1025, 20), (131072, 4), (131073, 4),
                                       (262145, 4), (400000, 4)])
def test_solves_at_the_edges_of_its_shapes(gpu, oracle, n, per_row, preconditioned):
    A, rng = _spd(n, per_row, n)
    b = rng.standard_normal(n)
    dinv = 1.0 / A.diagonal() if preconditioned else None
    print("case", n, per_row, preconditioned, "longest row", np.diff(A.indptr).max(), flush=True)
    for tol, maxiter in ((1e-9, 300), (0.0, 3)):
        xo, io, ro = oracle.pcg(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, b,
                                np.ones(n) if dinv is None else dinv, tol, maxiter)
        xg, ig, rg = _solve(gpu, A, b, dinv, tol, maxiter)
        assert ig == io
        assert np.allclose(xg, xo, rtol=1e-9, atol=1e-12 * np.abs(xo).max())
        assert abs(rg - ro) <= 1e-6 * ro + 1e-16


def test_a_solve_longer_than_one_launch(gpu):
    n = 20000  # a 1-D Laplacian: CG needs about n iterations, so 5000 leave it in the middle
    A = sp.csr_matrix(sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], shape=(n, n)))
    b = np.random.Generator(np.random.PCG64(4)).standard_normal(n)
    x, iters, relres = _solve(gpu, A, b, np.full(n, 0.5), 0.0, 5000)
    assert iters == 5000
    true = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    assert abs(true - relres) <= 1e-7 * max(true, 1.0)
    x1, i1, r1 = _solve(gpu, A, b, None, 0.0, 4097)
    assert i1 == 4097 and abs(np.linalg.norm(b - A @ x1) / np.linalg.norm(b) - r1) <= 1e-7 * max(r1, 1.0)


def test_a_wait_that_runs_out_falls_back_to_the_many_launch_solve(gpu, oracle, monkeypatch):
    A, rng = _spd(3000, 8, 9)
    b = rng.standard_normal(3000)
    want = _solve(gpu, A, b, None, 1e-9, 200)
    monkeypatch.setenv("LAPIS_HIP_CG_SPINS", "0")
    got = _solve(gpu, A, b, None, 1e-9, 200)
    assert got[1] == want[1] and np.allclose(got[0], want[0], rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("n,per_row", [(900, 6), (3000, 90), (540000, 4)])  # one launch; chunks of rows, small and large
def test_a_plan_or_entries_that_do_not_belong_to_the_system_are_refused(gpu, n, per_row, masked):
    A, rng = _spd(n, per_row, n)
    pos, crd, val = dev(A.indptr.astype(np.int32)), dev(A.indices.astype(np.int32)), dev(A.data)
    b, ones = dev(rng.standard_normal(n)), torch.ones(n, dtype=torch.float64, device="cuda")
    x = torch.full((n,), 7.0, dtype=torch.float64, device="cuda")
    plan = gpu.CsrPlan(n, n, pos, crd)

    def solve(plan, n=n, pos=pos, crd=crd, val=val):
        if masked:
            return gpu.pcg_masked(plan, n, pos, crd, val, b, ones, ones, 1e-9, 20, x)
        return gpu.pcg(plan, n, pos, crd, val, b, None, 1e-9, 20, x)
    wide = gpu.CsrPlan(n, n + 1, pos, crd)
    other = gpu.CsrPlan(n, n, pos.clone(), crd)
    for call in (lambda: solve(plan, n=n - 1), lambda: solve(wide), lambda: solve(other), lambda: solve(plan, pos=pos.clone())):
        with pytest.raises(gpu.LapisHipError) as e:
            call()
        assert e.value.status_name == "LAPIS_HIP_ERR_PLAN_MISMATCH"
    for p in (plan, None):
        for call in (lambda: solve(p, crd=None), lambda: solve(p, val=None)):
            with pytest.raises(gpu.LapisHipError) as e:
                call()
            assert e.value.status_name == "LAPIS_HIP_ERR_INVALID_ARGUMENT"
    if n == 900:  # a column-blocked copy stands in for the buffers it was made from only
        plan.build_colblock(crd, val)
        with pytest.raises(gpu.LapisHipError) as e:
            solve(plan, val=val.clone())
        assert e.value.status_name == "LAPIS_HIP_ERR_PLAN_MISMATCH"
    assert torch.equal(x, torch.full_like(x, 7.0))  # refused before anything was written
    solve(plan)
    assert not torch.equal(x, torch.full_like(x, 7.0))


@pytest.mark.parametrize("preconditioned", [False, True])
def test_a_launch_that_is_refused_falls_back_to_the_many_launch_solve(gpu, oracle, monkeypatch, preconditioned):
    A, rng = _spd(3000, 8, 9)
    b = rng.standard_normal(3000)
    dinv = 1.0 / A.diagonal() if preconditioned else None

    def solve():
        gpu.kernel_timing_start(400)  # counts products launched on their own
        result = _solve(gpu, A, b, dinv, 1e-9, 200)
        return result, gpu.kernel_timing_stop()["count"]
    want, products = solve()
    assert products == 0
    monkeypatch.setenv("LAPIS_HIP_CG_ONE_LAUNCH", "0")
    got, products = solve()
    assert products >= got[1] == want[1] and np.allclose(got[0], want[0], rtol=1e-9, atol=1e-12)
    monkeypatch.delenv("LAPIS_HIP_CG_ONE_LAUNCH")
    again, products = solve()
    assert products == 0 and again[1] == want[1] and np.array_equal(again[0], want[0])


def test_the_solution_in_the_right_hand_sides_buffer(gpu, monkeypatch):
    A, rng = _spd(3000, 8, 9)
    n, pos, crd, val = 3000, dev(A.indptr.astype(np.int32)), dev(A.indices.astype(np.int32)), dev(A.data)
    b = rng.standard_normal(n)
    want = _solve(gpu, A, b, None, 1e-9, 200)
    plan = gpu.CsrPlan(n, n, pos, crd)
    for spins in (None, "0"):  # as it comes, and through a one-launch solve that would give up
        if spins:
            monkeypatch.setenv("LAPIS_HIP_CG_SPINS", spins)
        x = dev(b)
        iters, _ = gpu.pcg(plan, n, pos, crd, val, x, None, 1e-9, 200, x)
        assert iters == want[1] and np.allclose(x.cpu().numpy(), want[0], rtol=1e-9, atol=1e-12)
