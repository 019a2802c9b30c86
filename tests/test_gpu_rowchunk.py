"""The SpMV over chunks of whole rows at the edges of its chunks: every chunk size and the longest rows of each, rows of
one entry, runs of empty rows longer than a chunk, chunks at the end of the arrays, buffers at any address."""
import numpy as np
import pytest
import torch

from gpu_util import assert_rows_close, dev, dev_unaligned, from_lengths
from lapis_amd import generators as gen

pytestmark = pytest.mark.gpu

LENGTHS = {
    "one": [1],
    "ones": [1] * 1023,
    "cap256": [64, 63, 64, 64, 64] * 40,
    "cap512": [65, 128, 1, 128] * 50,
    "cap1024": [129, 256, 256, 0, 1, 256] * 30,
    "long_even": [40] * 400,
    "two_lanes_per_row": [16] * 777,
    "empties": [3] + [0] * 3000 + [5, 0, 64] + [0] * 700,
    "mostly_empty": ([0] * 9 + [1]) * 500,
    "mixed": list(np.random.default_rng(5).integers(0, 50, 5000)),
    "uneven": [20, 19, 200, 0, 33, 65, 20, 1, 2, 256, 31, 32] * 60,
    "uneven_ends": [256] + [17] * 300 + [255],
    "too_long": [257] + [2] * 300,
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("name", LENGTHS)
def test_chunks_of_whole_rows(gpu, oracle, name, dtype):
    A = from_lengths(LENGTHS[name], 600, 31, dtype)
    x, y_in = gen.uniform_vector(A.ncols, 1, dtype=dtype), gen.uniform_vector(A.nrows, 2, dtype=dtype)
    want = y_in.copy()
    oracle.spmv(A.pos, A.crd, A.val, x, want)
    scale = oracle.spmv_abs_scale(A.pos, A.crd, A.val, x, y_in)
    for put in (dev, dev_unaligned):
        for value_bytes in (4, 8):  # what the plan was told steers its choices only
            pos, crd, val, dx, y = (put(a) for a in (A.pos, A.crd, A.val, x, y_in))
            plan = gpu.CsrPlan(A.nrows, A.ncols, pos, crd, value_bytes=value_bytes)
            assert (plan.kernel_name() == "spmv_rowchunk_kernel") == (name != "too_long")
            gpu.spmv(plan, A.nrows, A.ncols, pos, crd, val, dx, y)
            assert_rows_close(y.cpu().numpy(), want, scale, dtype, name)
            for kernel in (3, 2, 0):  # other kernels on request, and back to the plan's choice
                plan.set_kernel(kernel)
                y.copy_(torch.from_numpy(y_in))
                gpu.spmv(plan, A.nrows, A.ncols, pos, crd, val, dx, y)
                assert_rows_close(y.cpu().numpy(), want, scale, dtype, "%s kernel %d" % (name, kernel))
            assert (plan.kernel_name() == "spmv_rowchunk_kernel") == (name != "too_long")


def test_matrices_on_both_sides_of_the_last_level_cache_rule(gpu, oracle):
    for n in (1600, 2200):  # 154 MB and 290 MB of matrix: contiguous chunks per XCD, then round-robin
        A = gen.laplace2d(n)
        x = gen.uniform_vector(A.ncols, 3)
        want = np.zeros(A.nrows)
        oracle.spmv(A.pos, A.crd, A.val, x, want)
        pos, crd, y = dev(A.pos), dev(A.crd), dev(np.zeros(A.nrows))
        plan = gpu.CsrPlan(A.nrows, A.ncols, pos, crd)
        gpu.spmv(plan, A.nrows, A.ncols, pos, crd, dev(A.val), dev(x), y)
        scale = oracle.spmv_abs_scale(A.pos, A.crd, A.val, x, np.zeros(A.nrows))
        assert_rows_close(y.cpu().numpy(), want, scale, np.float64, "grid %d" % n)


# a workgroup per group of chunks (1900^2), workgroups that take several (1600, 901), a single short chunk (3)
@pytest.mark.parametrize("nx,iters", [(3, 2), (901, 1), (901, 2), (901, 3), (901, 4), (1600, 3), (1900, 3)])
@pytest.mark.parametrize("preconditioned", [False, True])
def test_cg_leaves_after_odd_and_even_passes(gpu, oracle, monkeypatch, nx, iters, preconditioned):
    monkeypatch.setenv("LAPIS_HIP_CG_SPINS", "0")  # systems that would be solved in one launch take the passes too
    A = gen.laplace2d(nx)
    n = A.nrows
    b = gen.uniform_vector(n, 9)
    dinv = gen.uniform_vector(n, 10, 0.2, 0.3) if preconditioned else np.ones(n)
    x_ref, it_ref, res_ref = oracle.pcg(A.pos, A.crd, A.val, b, dinv, 1e-30, iters)
    for put in (dev, dev_unaligned):
        pos, crd, val, db, x = (put(a) for a in (A.pos, A.crd, A.val, b, np.full(n, 7.0)))
        plan = gpu.CsrPlan(n, n, pos, crd)
        assert plan.kernel_name() == "spmv_rowchunk_kernel"
        it, res = gpu.pcg(plan, n, pos, crd, val, db, put(dinv) if preconditioned else None, 1e-30, iters, x)
        assert it == it_ref == iters and abs(res - res_ref) <= 1e-10 * res_ref
        assert np.linalg.norm(x.cpu().numpy() - x_ref) <= 1e-10 * np.linalg.norm(x_ref)
