"""Calls on host arrays at the sizes where their way to the device changes: brought by a kernel, in one transfer, in pieces
on two streams, in rounds of the pinned memory; results worked on in pinned memory or brought back in pieces; the counts
the copying pass makes at the edges of its blocks; several threads at once."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def module(gpu):
    from lapis_amd.module import LAPISModule
    return LAPISModule()


def _matrix(n, m, per_row, dtype, seed):
    rng = np.random.default_rng(seed)
    lengths = rng.integers(0, 2 * per_row + 1, n)
    pos = np.zeros(n + 1, np.int32)
    pos[1:] = np.cumsum(lengths)
    crd = rng.integers(0, m, pos[-1]).astype(np.int32)
    return pos, crd, rng.uniform(-1, 1, pos[-1]).astype(dtype), rng


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("n,m,per_row", [(0, 5, 1), (1, 1, 1), (1023, 7, 3), (16384, 65536, 8), (65535, 65536, 2), (65537, 1000, 3),
                                         (300001, 100000, 4), (1100000, 2000, 5)])
def test_products_of_host_arrays(module, n, m, per_row, dtype):
    pos, crd, val, rng = _matrix(n, m, per_row, dtype, n + m)
    x, y = rng.uniform(-1, 1, m).astype(dtype), rng.uniform(-1, 1, n).astype(dtype)
    A = sp.csr_matrix((val, crd, pos), shape=(n, m))
    want = y + A @ x
    out = module.spmv(pos, crd, val, ((n, m), (n + 1, len(crd), len(val))), x, y)
    tol = 1e-12 if dtype == np.float64 else 2e-5
    assert out.base is y or out is y or n == 0
    assert np.allclose(y, want, rtol=tol, atol=tol * 10)
    if n and n <= 65537:
        B, C = rng.uniform(-1, 1, (m, 5)).astype(dtype), rng.uniform(-1, 1, (n, 5)).astype(dtype)
        want = C + A @ B
        assert np.allclose(module.spmm(pos, crd, val, ((n, m), (n + 1, len(crd), len(val))), B, C), want, rtol=tol, atol=tol * 10)


def test_several_threads(module):
    errors = []

    def work(seed):
        n = 20000 * (seed + 1)
        pos, crd, val, rng = _matrix(n, n, 6, np.float64, seed)
        A = sp.csr_matrix((val, crd, pos), shape=(n, n))
        x = rng.uniform(-1, 1, n)
        want = A @ x
        for _ in range(5):
            y = np.zeros(n)
            module.spmv(pos, crd, val, ((n, n), (n + 1, len(crd), len(val))), x, y)
            if not np.allclose(y, want, rtol=1e-12, atol=1e-11):
                errors.append(seed)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


def test_memory_kept_between_calls_is_bounded_for_all_of_them_together(gpu):
    import torch
    host = np.zeros(25_000_000)  # 200 MB: an arena of 256 MB each
    free = lambda: torch.cuda.mem_get_info()[0]
    torch.cuda.synchronize()
    before = free()
    held = [gpu.stage([host]) for _ in range(3)]
    assert before - free() >= 512 << 20  # one of them may have been there
    del held
    torch.cuda.synchronize()
    assert before - free() <= (256 << 20) + (32 << 20)
    (t,), staged = gpu.stage([host[:1000] + 3.0])  # and the arenas still serve calls
    assert torch.equal(t, torch.full_like(t, 3.0))


def test_a_process_that_gets_no_threads_copies_alone(gpu):
    # a process of its own: the threads are started once
    code = """
import os
os.environ["LAPIS_HIP_STAGING_HELPERS"] = "0"
import numpy as np, scipy.sparse as sp
from lapis_amd.module import LAPISModule
n = 300001
A = sp.csr_matrix(sp.diags([1.0, 2.0, 3.0], [-1, 0, 1], shape=(n, n)))
x, y = np.arange(n) % 7 - 3.0, np.ones(n)
pos, crd = A.indptr.astype(np.int32), A.indices.astype(np.int32)
module = LAPISModule()
for k in range(3):
    module.spmv(pos, crd, A.data, ((n, n), (n + 1, len(crd), len(crd))), x, y)
assert np.array_equal(y, 1.0 + 3.0 * (A @ x)), "wrong product"
print("the same")
"""
    out = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and "the same" in out.stdout, out.stderr
