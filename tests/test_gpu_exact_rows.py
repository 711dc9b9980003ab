"""Exact PTPR with the levels of stage 1 inside the lane (exact_rows.hpp):
bit identity with the oracle on every shape that runs this way, on inputs
that reach its corners -- missing partners at the ends of a slice, signed
zeros, infinities and NaNs beside them, denominators outside the short
reciprocal's range -- and the short reciprocal itself on every float."""
import ctypes
import os
import sys

import numpy as np
import pytest
import torch

import oracle as O
from tpr_amd import batched as B
from tpr_amd import build

pytestmark = pytest.mark.gpu


def bits_equal(x, y):
    same = x.view(np.uint32) == y.view(np.uint32)
    return bool(np.all(same | (np.isnan(x) & np.isnan(y))))


def special_batch(seed, n, s):
    """One kind of special value per system, spread over every position of a
    slice."""
    rng = np.random.default_rng(seed)
    special = [(0.0, -0.0), (-0.0, -0.0), (np.inf, 1.0), (np.nan, 0.0), (1e-39, -0.0), (3e38, 0.0), (-1e20, 1e30),
               (1.0, 1.0)]
    nsys = len(special)
    a, b, c, d, _ = O.gen_batch(seed + 1, 0, nsys, n, O.GEN_DOMINANT)
    a, b, c, d = (v.reshape(nsys, n) for v in (a, b, c, d))
    for k, (off, rhs) in enumerate(special):
        at = np.unique(np.concatenate([rng.integers(0, n, 12), [0, 1, s - 1, s, n - 2, n - 1]]))
        b[k] = 1.0
        for v in (a, c):
            v[k, at] = np.float32(off)
        d[k, at[::2]] = np.float32(rhs)
        if off == 1.0:  # 1 - c a = 0 between neighbours
            a[k, 1::2], c[k, 0::2] = 1.0, 1.0
        a[k, 0] = c[k, n - 1] = 0.0
    return [np.ascontiguousarray(v.ravel(), np.float32) for v in (a, b, c, d)], nsys


def gpu(a, b, c, d, n, s, shape=None, **kw):
    da, db, dc, dd = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (a, b, c, d))
    x = torch.full_like(dd, 7.0)
    B.solve_ex(da, db, dc, dd, x, n, s, arith="exact", shape=shape, **kw)
    torch.cuda.synchronize()
    return x.cpu().numpy()


SHAPES = [(8, 16), (16, 16), (8, 32), (8, 64), (16, 32), (16, 64), (32, 64)]


@pytest.mark.parametrize("E,L", SHAPES)
@pytest.mark.parametrize("m", [1, 4, 16])
def test_shapes_bit_identical(E, L, m):
    s = E * L
    n = s * m
    if m * L > 1024:
        n, m = s * (1024 // L), 1024 // L
    nsys = 5
    print("exact rows", E, L, m, flush=True)
    for kind in (O.GEN_DOMINANT, O.GEN_WEAK):
        a, b, c, d, _ = O.gen_batch(71, 0, nsys, n, kind)
        assert bits_equal(gpu(a, b, c, d, n, s, (E, L)), O.solve_batch("ptpr", a, b, c, d, n, s)), kind


@pytest.mark.parametrize("E,L", SHAPES)
def test_special_values_bit_identical(E, L):
    """One kind of special value per system, spread over every position of a
    slice: zeros of both signs, infinities, NaN, and off-diagonals that make a
    denominator zero, subnormal or beyond 2^126."""
    s = E * L
    m = 2
    n = s * m
    rng = np.random.default_rng(72)
    special = [(0.0, -0.0), (-0.0, -0.0), (np.inf, 1.0), (np.nan, 0.0), (1e-39, -0.0), (3e38, 0.0), (-1e20, 1e30),
               (1.0, 1.0)]
    nsys = len(special)
    a, b, c, d, _ = O.gen_batch(73, 0, nsys, n, O.GEN_DOMINANT)
    a, b, c, d = (v.reshape(nsys, n) for v in (a, b, c, d))
    for k, (off, rhs) in enumerate(special):
        at = np.unique(np.concatenate([rng.integers(0, n, 12), [0, 1, s - 1, s, n - 2, n - 1]]))
        b[k] = 1.0
        for v in (a, c):
            v[k, at] = np.float32(off)
        d[k, at[::2]] = np.float32(rhs)
        if off == 1.0:  # 1 - c a = 0 between neighbours
            a[k, 1::2], c[k, 0::2] = 1.0, 1.0
        a[k, 0] = c[k, n - 1] = 0.0
    a, b, c, d = (np.ascontiguousarray(v.ravel(), np.float32) for v in (a, b, c, d))
    x = gpu(a, b, c, d, n, s, (E, L)).reshape(nsys, n)
    with np.errstate(all="ignore"):
        ref = O.solve_batch("ptpr", a, b, c, d, n, s).reshape(nsys, n)
    for k in range(nsys):
        assert bits_equal(x[k], ref[k]), (k, special[k], np.flatnonzero(x[k].view(np.uint32) != ref[k].view(np.uint32))[:8])


@pytest.mark.parametrize("n,s", [(32768, 128), (65536, 256), (65536, 1024), (65536, 2048)])
def test_multi_workgroup_bit_identical(n, s):
    nsys = 3
    a, b, c, d, _ = O.gen_batch(74, 0, nsys, n, O.GEN_WEAK)
    ref = O.solve_batch("ptpr", a, b, c, d, n, s)
    assert bits_equal(gpu(a, b, c, d, n, s), ref)
    h = [v.astype(np.float16) for v in (a, b, c)]
    wide = [v.astype(np.float32) for v in h]
    assert bits_equal(gpu(*h, d, n, s), O.solve_batch("ptpr", *wide, d, n, s))


def test_short_reciprocal_on_every_float():
    if not os.path.exists(build.DIAG_LIB):
        pytest.fail("libtpr_diag.so is not built")
    L = ctypes.CDLL(build.DIAG_LIB)
    L.tprh_diag_recip_short_check.restype = ctypes.c_int
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    print("short reciprocal over 2^32 inputs", flush=True)
    assert L.tprh_diag_recip_short_check(ctypes.c_void_p(counts.data_ptr()), ctypes.c_void_p(0)) == 0
    torch.cuda.synchronize()
    differ, seen = counts.tolist()
    assert differ == 0
    # 252 binades of both signs, 2^126 itself, and the NaNs
    assert seen == 2 * (252 << 23) + 2 + 2 * ((1 << 23) - 1)
    sys.stdout.flush()


def diag(name):
    if not os.path.exists(build.DIAG_LIB):
        pytest.fail("libtpr_diag.so is not built")
    f = getattr(ctypes.CDLL(build.DIAG_LIB), name)
    f.restype = ctypes.c_int
    return f


def test_short_quotient():
    """n / x for 4096 significands of x, the ends of their range among them,
    against every significand of n."""
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    f = diag("tprh_diag_quot_short_check")
    for first, stride, blocks in ((0, 1, 512), ((1 << 23) - 512, 1, 512), (1777, 2729, 3072)):
        print("short quotient", first, stride, blocks, flush=True)
        assert f(blocks, ctypes.c_uint(first), ctypes.c_uint(stride), ctypes.c_void_p(counts.data_ptr()),
                 ctypes.c_void_p(0)) == 0
        torch.cuda.synchronize()
    assert counts.tolist() == [0, 4096 << 23]


@pytest.mark.parametrize("kind", ["plain", "zeros", "range", "special"])
def test_quotients_of_one_divisor(kind):
    """Whole wavefronts on the short path, and ones that zeros, values at and
    past the ends of its range, infinities and NaNs send to division or not."""
    rng = np.random.default_rng(75)
    blocks = 64
    v = rng.uniform(0.5, 2.0, (blocks, 4, 64, 8)) * rng.choice([-1.0, 1.0], (blocks, 4, 64, 8))
    v = v.astype(np.float32)
    odd = {"plain": [], "zeros": [0.0, -0.0],
           "range": [2.0**-60, np.nextafter(np.float32(2.0**-60), np.float32(0)), 2.0**60,
                     np.nextafter(np.float32(2.0**60), np.float32(np.inf)), 1e-40, -1e-45, 3e38, -2.0**-100],
           "special": [np.inf, -np.inf, np.nan, 0.0, -0.0]}[kind]
    if odd:
        # the first half of the workgroups in a, c, d alone, the rest in b too
        hit = rng.random(v.shape) < 0.02
        hit[: blocks // 2, 3] = False
        v[hit] = rng.choice(np.array(odd, np.float32), int(hit.sum()))
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    ops = torch.from_numpy(np.ascontiguousarray(v)).cuda()
    torch.cuda.synchronize()
    assert diag("tprh_diag_quots_check")(ctypes.c_void_p(ops.data_ptr()), blocks, ctypes.c_void_p(counts.data_ptr()),
                                         ctypes.c_void_p(0)) == 0
    torch.cuda.synchronize()
    assert counts.tolist() == [0, blocks * 64 * 24]


TPR_SHAPES = [(2, 16), (4, 16), (4, 64)] + SHAPES


@pytest.mark.parametrize("E,L", TPR_SHAPES)
def test_tpr_shared_branches_bit_identical(E, L):
    s = E * L
    n = 2 * s
    print("exact tpr", E, L, flush=True)
    (a, b, c, d), nsys = special_batch(76, n, s)
    x = gpu(a, b, c, d, n, s, (E, L), method="tpr").reshape(nsys, n)
    with np.errstate(all="ignore"):
        ref = O.solve_batch("tpr", a, b, c, d, n, s).reshape(nsys, n)
    for k in range(nsys):
        assert bits_equal(x[k], ref[k]), k
    a, b, c, d, _ = O.gen_batch(78, 0, 5, n, O.GEN_WEAK)
    assert bits_equal(gpu(a, b, c, d, n, s, (E, L), method="tpr"), O.solve_batch("tpr", a, b, c, d, n, s))


def zero_batch(seed, n, nsys):
    """Systems whose off-diagonals and most right-hand sides are zeros of
    either sign; the first is all +0 / -0 but for right-hand sides of -1."""
    rng = np.random.default_rng(seed)

    def pick(values):
        return rng.choice(np.array(values, np.float32), nsys * n)

    a, c = pick([0.0, -0.0]), pick([0.0, -0.0])
    b, d = pick([1.0, 1.0, -1.0]), pick([0.0, -0.0, -0.0, 1.0, -1.0])
    a[:n], c[:n], b[:n], d[:n] = 0.0, -0.0, 1.0, -1.0
    d[0] = -0.0
    return a, b, c, d


@pytest.mark.parametrize("method", ["ptpr", "tpr"])
@pytest.mark.parametrize("E,L", SHAPES)
def test_signs_of_zeros_bit_identical(E, L, method):
    """A missing partner must leave a right-hand side of -0 as it is."""
    s = E * L
    for m in (1, 2, 16):
        n = s * m
        if m * L > 1024:
            continue
        print("signs of zeros", method, E, L, m, flush=True)
        a, b, c, d = zero_batch(75 + m, n, 20)
        for diag in (b, np.ones_like(b)):
            ref = O.solve_batch(method, a, diag, c, d, n, s)
            assert bits_equal(gpu(a, diag, c, d, n, s, (E, L), method=method), ref)


@pytest.mark.parametrize("n,s", [(32768, 128), (65536, 256), (65536, 2048)])
def test_signs_of_zeros_multi_workgroup(n, s):
    a, b, c, d = zero_batch(78, n, 3)
    assert bits_equal(gpu(a, b, c, d, n, s), O.solve_batch("ptpr", a, b, c, d, n, s))
