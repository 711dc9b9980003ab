"""Host-pointer calls return when their answers have arrived: answers that
hold the very word the call waits to be replaced (a NaN of all ones) must
still end the call, and the next call must not see anything of it."""
import time

import numpy as np
import pytest

import oracle as O
from tpr_amd import solvers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["ptpr", "tpr"])
@pytest.mark.parametrize("n,s", [(64, 16), (2048, 512)])
def test_nan_of_all_ones_ends_the_call(method, n, s):
    call = solvers.ptpr_cu if method == "ptpr" else solvers.tpr_cu
    a, b, c, d, _ = O.gen_batch(81, 0, 1, n, O.GEN_DOMINANT)
    a, c, d = a / b, c / b, d / b
    one = np.ones(n, np.float32)
    ref = O.solve_batch(method, a, one, c, d, n, s)
    for bad in (0, n // 2, n - 1):
        print(method, n, s, bad, flush=True)
        e = d.copy()
        e.view(np.uint32)[bad] = 0xFFFFFFFF
        x = np.full(n, 3.0, np.float32)
        start = time.perf_counter()
        call(a, c, e, x, n, s)
        assert time.perf_counter() - start < 5.0
        want = O.solve_batch(method, a, one, c, e, n, s)
        same = (x.view(np.uint32) == want.view(np.uint32)) | (np.isnan(x) & np.isnan(want))
        assert same.all()
        y = np.empty(n, np.float32)
        call(a, c, d, y, n, s)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("method", ["pcr", "cr"])
@pytest.mark.parametrize("n", [64, 2048, 4096])
def test_nan_of_all_ones_ends_the_call_pcr_cr(method, n):
    """The same for the whole-system solvers."""
    call = solvers.pcr_cu if method == "pcr" else solvers.cr_cu
    a, b, c, d, _ = O.gen_batch(82, 0, 1, n, O.GEN_DOMINANT)
    a, c, d = a / b, c / b, d / b
    solve = O.pcr if method == "pcr" else O.cr
    ref = solve(a, c, d)
    for bad in (0, n // 2, n - 1):
        print(method, n, bad, flush=True)
        e = d.copy()
        e.view(np.uint32)[bad] = 0xFFFFFFFF
        x = np.full(n, 3.0, np.float32)
        start = time.perf_counter()
        call(a, c, e, x, n)
        assert time.perf_counter() - start < 5.0
        want = solve(a, c, e)
        assert ((x.view(np.uint32) == want.view(np.uint32)) | (np.isnan(x) & np.isnan(want))).all()
        y = np.empty(n, np.float32)
        call(a, c, d, y, n)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("method", ["ptpr", "tpr"])
def test_calls_of_changing_sizes_after_an_early_return(method):
    """A call that returns with its answers, ahead of its kernel's end, then
    one whose buffers have to grow, one that copies through device memory
    (several workgroups), and small ones again."""
    call = solvers.ptpr_cu if method == "ptpr" else solvers.tpr_cu
    systems = {}
    for k, n in enumerate((64, 2048, 8192, 65536, 131072)):
        s = min(n // 4, 256)
        a, b, c, d, _ = O.gen_batch(83 + k, 0, 1, n, O.GEN_DOMINANT)
        a, c, d = a / b, c / b, d / b
        systems[n] = (a, c, d, s, O.solve_batch(method, a, np.ones(n, np.float32), c, d, n, s))
    for n in (64, 64, 2048, 64, 8192, 2048, 131072, 64, 65536, 2048, 131072, 8192, 64):
        print(method, n, flush=True)
        a, c, d, s, ref = systems[n]
        x = np.full(n, 3.0, np.float32)
        call(a, c, d, x, n, s)
        assert np.array_equal(x.view(np.uint32), ref.view(np.uint32)), n
