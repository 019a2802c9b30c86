"""SpMM and the batched CSRV product at the edges of their launch shapes: k around multiples of the vector width and
of a wavefront's columns, rows longer than the staged window, rows of B at any address, every lanes-per-row split."""
import numpy as np
import pytest
import torch

from gpu_util import TOL, dev, from_lengths
from lapis_amd import generators as gen
from test_gpu_spmm import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 10, 13, 31, 63, 127, 129, 255, 257, 259])
def test_ragged_widths_on_short_and_long_rows(gpu, oracle, dtype, k):
    rng = np.random.default_rng(k)
    short = rng.integers(0, 12, 777)                                     # several rows per wavefront
    long = np.concatenate([rng.integers(90, 240, 37), [0, 383, 384, 385, 0, 768]])  # windows of 384 entries cut inside rows
    for lengths, ncols in ((short, 500), (long, 3000)):
        A = from_lengths(list(lengths), ncols, 7 + k, dtype)
        B = gen.uniform_matrix(ncols, k, 8).astype(dtype)
        C_in = gen.uniform_matrix(A.nrows, k, 9).astype(dtype)
        for plan in (True, False):
            _check(gpu, oracle, A, B, C_in, dtype, "rows of %d.., k=%d plan=%s" % (lengths[0], k, plan), plan=plan)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_rows_of_B_and_C_at_any_address(gpu, oracle, dtype):
    A = from_lengths([5] * 300, 200, 3, dtype)
    for k, ldb, off in ((6, 7, 1), (16, 17, 3), (9, 9, 1)):
        flat_b, flat_c = gen.uniform_matrix(1, 200 * ldb + off, 4)[0].astype(dtype), gen.uniform_matrix(1, 300 * ldb + off, 5)[0].astype(dtype)
        view = lambda t, rows: torch.as_strided(t, (rows, k), (ldb, 1), off)
        dB, dC = dev(flat_b), dev(flat_c)
        B = np.lib.stride_tricks.as_strided(flat_b[off:], (200, k), (ldb * flat_b.itemsize, flat_b.itemsize)).copy()
        want = np.lib.stride_tricks.as_strided(flat_c[off:], (300, k), (ldb * flat_c.itemsize, flat_c.itemsize)).copy()
        oracle.spmm(A.pos, A.crd, A.val, B, want)
        pos, crd = dev(A.pos), dev(A.crd)
        plan = gpu.CsrPlan(A.nrows, A.ncols, pos, crd, value_bytes=np.dtype(dtype).itemsize)
        gpu.spmm(A.nrows, A.ncols, pos, crd, dev(A.val), view(dB, 200), view(dC, 300), plan=plan)
        got = dC.cpu().numpy()
        assert np.allclose(view(dC, 300).cpu().numpy(), want, rtol=1e-5, atol=1e-5)
        untouched = np.ones(got.size, bool)
        untouched[(off + np.arange(300)[:, None] * ldb + np.arange(k)).ravel()] = False
        assert np.array_equal(got[untouched], flat_c[untouched])


@pytest.mark.parametrize("n,mean,k", [(70000, 4, 64), (140000, 16, 64), (140000, 16, 132)])
def test_scattered_columns_over_a_B_larger_than_the_caches(gpu, oracle, n, mean, k):
    A = gen.fixed_degree_random(n, mean, seed=5, dtype=np.float32)
    B = gen.uniform_matrix(n, k, 6)
    _check(gpu, oracle, A, B, np.zeros((n, k), np.float32), np.float32, "scattered n=%d k=%d" % (n, k), plan=True)


@pytest.mark.parametrize("dh,nh", [(1, 1), (3, 1), (4, 1), (5, 1), (2, 3), (5, 7), (31, 8), (32, 8), (64, 4), (65, 4), (9, 300), (1, 1025)])
def test_batched_csrv_product_shapes(gpu, oracle, dh, nh):
    rng = np.random.default_rng(dh * 1000 + nh)
    lengths = np.concatenate([rng.integers(0, 20, 61), [0, 300, 1, 257, 0, 33]])
    A = from_lengths(list(lengths), 400, 17, np.float32)
    values = rng.uniform(-1, 1, A.nnz * nh).astype(np.float32)
    V = rng.uniform(-1, 1, (400, dh, nh)).astype(np.float32)
    out = torch.zeros(A.nrows, dh, nh, dtype=torch.float32, device="cuda")
    print("case", dh, nh, flush=True)
    gpu.bspmm_csrv(A.nrows, 400, dev(A.pos), dev(A.crd), dev(values), dev(V), out)
    assert np.array_equal(out.cpu().numpy(), oracle.bspmm_csrv(A.pos, A.crd, values, V, A.nrows))


@pytest.mark.parametrize("n2,dh,nh", [(11000, 64, 3), (11000, 12, 16), (8400, 32, 8), (8100, 32, 8), (7000, 40, 8), (7000, 40, 9),
                                      (5000, 128, 4), (4200, 64, 9), (17000, 32, 8), (33000, 32, 8)])
def test_batched_csrv_product_in_parts_of_a_row_of_V(gpu, oracle, n2, dh, nh):
    # V on both sides of 8 MB and of 16 MB a part, rows of an even and an odd number of 256 bytes, windows of 32 and more
    # entries and (too many heads) the general path; row lengths around the windows
    rng = np.random.default_rng(n2 + nh)
    A = from_lengths(list(np.concatenate([rng.integers(0, 70, 150), [0, 31, 32, 33, 63, 64, 65, 0, 300]])), n2, 18, np.float32)
    values = rng.uniform(-1, 1, A.nnz * nh).astype(np.float32)
    V = rng.uniform(-1, 1, (n2, dh, nh)).astype(np.float32)
    out = torch.zeros(A.nrows, dh, nh, dtype=torch.float32, device="cuda")
    print("case", n2, dh, nh, flush=True)
    gpu.bspmm_csrv(A.nrows, n2, dev(A.pos), dev(A.crd), dev(values), dev(V), out)
    assert np.array_equal(out.cpu().numpy(), oracle.bspmm_csrv(A.pos, A.crd, values, V, A.nrows))  # the order of the reference's nest: bit-exact


@pytest.mark.parametrize("dh,nh", [(4, 1), (5, 1), (2, 3), (5, 7), (31, 1), (4, 12), (32, 4), (3, 100)])
@pytest.mark.parametrize("rows", [2100, 4200, 17000])
def test_batched_csrv_product_with_several_rows_per_wavefront(gpu, oracle, rows, dh, nh):
    # from one row per wavefront to the most, by the number of rows
    rng = np.random.default_rng(rows + dh * 1000 + nh)
    lengths = rng.integers(0, 9, rows)
    lengths[:: rows // 5] = rng.integers(60, 290, lengths[:: rows // 5].size)
    A = from_lengths(list(lengths), 400, 19, np.float32)
    values = rng.uniform(-1, 1, A.nnz * nh).astype(np.float32)
    V = rng.uniform(-1, 1, (400, dh, nh)).astype(np.float32)
    out = torch.zeros(A.nrows, dh, nh, dtype=torch.float32, device="cuda")
    print("case", rows, dh, nh, flush=True)
    gpu.bspmm_csrv(A.nrows, 400, dev(A.pos), dev(A.crd), dev(values), dev(V), out)
    assert np.array_equal(out.cpu().numpy(), oracle.bspmm_csrv(A.pos, A.crd, values, V, A.nrows))


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("rows_of_B", [(1 << 10) - 1, 1 << 10, 1500])
def test_byte_offsets_into_B_around_two_to_the_32(gpu, oracle, dtype, rows_of_B):
    # rows of B 4 MB apart: 32-bit byte offsets to the last below 4 GB, 64-bit ones from 4 GB on; vectors and single elements,
    # one and several column chunks, even short rows (several per wavefront with a plan) and long ones
    size = np.dtype(dtype).itemsize
    ldb, rng = (1 << 22) // size, np.random.default_rng(rows_of_B)
    whole = torch.empty((rows_of_B - 1) * ldb + 300, dtype=torch.float32 if size == 4 else torch.float64, device="cuda")
    for lengths in ([7] * 150, list(rng.integers(0, 400, 40)) + [0, 385]):
        A = from_lengths(lengths, rows_of_B, 23, dtype)
        A.crd[A.pos[1:][np.diff(A.pos) > 0] - 1] = rows_of_B - 1  # the last row of B in every row of A
        for k in (1, 3, 10, 64, 300):
            B, C_in = rng.uniform(-1, 1, (rows_of_B, k)).astype(dtype), rng.uniform(-1, 1, (A.nrows, k)).astype(dtype)
            view = torch.as_strided(whole, (rows_of_B, k), (ldb, 1))
            view.copy_(dev(B))
            want = C_in.copy()
            oracle.spmm(A.pos, A.crd, A.val, B, want)
            row_of = np.repeat(np.arange(A.nrows), np.diff(A.pos))
            scale = np.abs(C_in) + np.bincount(row_of, np.abs(A.val), A.nrows)[:, None]  # |B| <= 1
            pos, crd, val = dev(A.pos), dev(A.crd), dev(A.val)
            for plan in (None, gpu.CsrPlan(A.nrows, rows_of_B, pos, crd, value_bytes=size)):
                print("case", dtype.__name__, rows_of_B, lengths[0], k, plan is not None, flush=True)
                C = dev(C_in)
                gpu.spmm(A.nrows, rows_of_B, pos, crd, val, view, C, plan=plan)
                assert np.all(np.abs(C.cpu().numpy().astype(np.float64) - want) <= TOL[np.dtype(dtype)] * scale)


@pytest.mark.parametrize("n2,dh,nh", [((1 << 21) - 1, 64, 8), (1 << 21, 64, 8), ((1 << 21) + 5, 64, 8), (2093043, 171, 3), (2093042, 171, 3)])
def test_byte_offsets_into_V_around_two_to_the_32(gpu, oracle, n2, dh, nh):
    # V just below and from 4 GB on, heads in vectors and not; 300 of its rows are used, its first and last among them
    rng = np.random.default_rng(n2)
    used = np.unique(np.concatenate([[0, n2 - 1], rng.integers(0, n2, 298)]))
    A = from_lengths(list(rng.integers(0, 40, 90)) + [0, 150], used.size, 29, np.float32)
    A.crd[A.pos[1:][np.diff(A.pos) > 0] - 1] = used.size - 1
    values = rng.uniform(-1, 1, A.nnz * nh).astype(np.float32)
    small = rng.uniform(-1, 1, (used.size, dh, nh)).astype(np.float32)
    V = torch.empty((n2, dh, nh), dtype=torch.float32, device="cuda")
    V[torch.from_numpy(used).cuda()] = dev(small)
    out = torch.zeros(A.nrows, dh, nh, dtype=torch.float32, device="cuda")
    print("case", n2, dh, nh, flush=True)
    gpu.bspmm_csrv(A.nrows, n2, dev(A.pos), dev(used[A.crd].astype(np.int32)), dev(values), V, out)
    assert np.array_equal(out.cpu().numpy(), oracle.bspmm_csrv(A.pos, A.crd, values, small, A.nrows))
