"""Uneven batches whose systems all fit 256 lanes: one workgroup per item,
loads and stores staged with several systems to a wavefront.  Exact results
bit-identical to the oracle, fast ones to the same systems in a batch that
takes the 1024-lane kernel, over counts that leave items partly empty."""
import numpy as np
import pytest
import torch

import oracle as O
from tpr_amd.uneven import UnevenPlan

pytestmark = pytest.mark.gpu


def bits_equal(x, y):
    same = x.view(np.uint32) == y.view(np.uint32)
    return bool(np.all(same | (np.isnan(x) & np.isnan(y))))


def solve(sizes, method, arith, unit, schedule=None):
    plan = UnevenPlan(sizes, method=method, arith=arith, schedule=schedule)
    a, b, c, d, x, xt = [torch.zeros(plan.equations, device="cuda") for _ in range(6)]
    plan.generate("dominant", 91, 0, a, b, c, d, xt)
    if unit:
        a, c, d, b = a / b, c / b, d / b, None
    x.fill_(7.0)
    plan.solve(a, b, c, d, x)
    torch.cuda.synchronize()
    host = [None if v is None else v.cpu().numpy() for v in (a, b, c, d, x)]
    return plan, host


SIZES = [
    [16],
    [32] * 17 + [16],
    [64, 128, 64, 256, 128, 64] * 3 + [64],
    [4096, 256, 2048, 512, 1024, 16, 4096, 256],
    [128] * 33 + [512] * 5,
]


@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("method", ["ptpr", "tpr"])
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "%dx%d" % (len(s), max(s)))
def test_tiles_exact_bit_identical(sizes, method, unit):
    print("tiles", sizes[:4], method, unit, flush=True)
    plan, (a, b, c, d, x) = solve(sizes, method, "exact", unit)
    for k, n in enumerate(sizes):
        lo, hi = plan.offset(k), plan.offset(k + 1)
        one = np.ones(n, np.float32) if b is None else b[lo:hi]
        ref = O.solve_batch(method, a[lo:hi], one, c[lo:hi], d[lo:hi], n, min(n, 256))
        assert bits_equal(x[lo:hi], ref), (k, n)


@pytest.mark.parametrize("method", ["ptpr", "tpr"])
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "%dx%d" % (len(s), max(s)))
def test_tiles_equal_the_persistent_kernel(sizes, method):
    plan, (_, _, _, _, x) = solve(sizes, method, "fast", False)
    # the generator numbers the systems, so these come first in both
    _, (_, _, _, _, y) = solve(sizes + [8192], method, "fast", False)
    assert bits_equal(x, y[: x.size])


@pytest.mark.parametrize("E,L", [(8, 16), (16, 16), (8, 32), (4, 64)])
@pytest.mark.parametrize("method", ["ptpr", "tpr"])
def test_tiles_every_shape(method, E, L):
    s = E * L
    sizes = [s, 2 * s, s, 256 // L * s, s]
    schedule = {n: (s, E, L) for n in set(sizes)}
    plan, (a, b, c, d, x) = solve(sizes, method, "exact", False, schedule)
    for k, n in enumerate(sizes):
        lo, hi = plan.offset(k), plan.offset(k + 1)
        assert bits_equal(x[lo:hi], O.solve_batch(method, a[lo:hi], b[lo:hi], c[lo:hi], d[lo:hi], n, s)), (k, n)


@pytest.mark.parametrize("count", [1, 257, 600, 900])
def test_items_in_turn_and_by_counter(count):
    """Plans of 1024-lane items below, between and above one and three items
    per workgroup (a device of 256 CUs): every answer is written, the same in
    a second solve."""
    sizes = [16384] * count + [64]
    print("items", count, flush=True)
    plan = UnevenPlan(sizes)
    a, b, c, d, x, xt = [torch.zeros(plan.equations, device="cuda") for _ in range(6)]
    plan.generate("dominant", 92, 0, a, b, c, d, xt)
    for _ in range(2):
        x.fill_(7.0)
        plan.solve(a, b, c, d, x)
        torch.cuda.synchronize()
        err = (x.double() - xt.double()).view(-1)
        assert float(err.norm() / xt.double().norm()) < 1e-5
        # a system left out would be all sevens
        assert float(err.abs().max()) < 1e-2
