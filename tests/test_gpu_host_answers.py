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
