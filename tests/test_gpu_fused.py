"""The one-pass form of fast PTPR and TPR on systems larger than one workgroup
(split_fused.hpp): tiles of 4096 equations that exchange six numbers each.

Sizes at its edges: 8, 16 (one DPP row of tiles), 32 and 64 (several rows in
one wavefront) and 128 and 1024 tiles per system (exchange by groups).
Tolerances: rel-L2 1e-5 against the oracle on dominant systems (the fast
mode's), and on weakly dominant ones twice the two-pass form's error against
the FP64 Thomas solve, or 1e-6.
"""
import ctypes
import os
import sys
import types

import numpy as np
import pytest
import torch

import oracle as O
from tpr_amd import _lib
from tpr_amd import batched as B
from tpr_amd import build

pytestmark = pytest.mark.gpu

FAST_TOL = 1e-5


def say(*args):
    print(*args, flush=True)
    sys.stdout.flush()


def dev(v):
    return torch.from_numpy(np.ascontiguousarray(v)).cuda()


def rel(x, ref, n):
    x = np.asarray(x, np.float64).reshape(-1, n)
    ref = np.asarray(ref, np.float64).reshape(-1, n)
    return float((np.linalg.norm(x - ref, axis=1) / np.linalg.norm(ref, axis=1)).max())


def bits(t):
    return t.view(torch.int32).cpu().numpy()


@pytest.mark.parametrize("n,s,nsys", [(32768, 256, 3), (65536, 256, 5), (65536, 2048, 3), (131072, 512, 3),
                                      (262144, 256, 2), (524288, 1024, 3), (1 << 22, 2048, 1)])
@pytest.mark.parametrize("method", ["ptpr", "tpr"])
def test_one_pass_forms_agree(method, n, s, nsys):
    """Diagonal, unit diagonal, fp16 storage, a shared matrix, a refinement
    step: the one-pass form against the two passes and the oracle, and
    nothing written past x."""
    say("one pass", method, n, s, nsys)
    a, b, c, d, _ = O.gen_batch(61, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    guard = 4096

    def solve(form, coef, **kw):
        x0 = kw.pop("x0", None)
        x = torch.full((nsys * n + guard,), 2.5, device="cuda")
        if x0 is not None:
            x[:nsys * n] = x0
        B.solve_ex(*coef, dd, x[:nsys * n], n, s, split_form=form, method=method, **kw)
        torch.cuda.synchronize()
        assert bool((x[nsys * n:] == 2.5).all())
        return x[:nsys * n].clone()

    x = solve(0, (da, db, dc))
    assert rel(x.cpu().numpy(), O.solve_batch(method, a, b, c, d, n, s), n) <= FAST_TOL
    assert np.array_equal(bits(x), bits(solve(2, (da, db, dc))))
    cases = [((da, db, dc), {}), ((da / db, None, dc / db), {}), ([v.half() for v in (da, db, dc)], {}),
             ([v[:n].contiguous() for v in (da, db, dc)], {"shared": True}),
             ((da, db, dc), {"refine": True, "x0": x * (1 + 1e-3 * torch.rand_like(x))})]
    for coef, kw in cases:
        one, two = solve(0, coef, **kw), solve(1, coef, **kw)
        assert rel(one.cpu().numpy(), two.cpu().numpy(), n) <= FAST_TOL, kw


@pytest.mark.parametrize("n,s,nsys", [(1 << 20, 512, 2), (1 << 21, 1024, 1)])
@pytest.mark.parametrize("method", ["ptpr", "tpr"])
def test_one_pass_refinement_with_many_groups(method, n, s, nsys):
    """A refinement step in the one-pass form on 256 and 512 tiles per system.
    (At three workgroups per CU the device does not hold the 1024 tiles of 4
    Mi equations at once, and that step takes two passes.)"""
    say("one pass, many groups", method, n, s, nsys)
    a, b, c, d, _ = O.gen_batch(68, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    ref = O.thomas_f64_batch(a, b, c, d, n)
    start = dev(O.solve_batch(method, a, b, c, d, n, s)) * 1.001
    err = []
    for form in (0, 1):
        x = start.clone()
        B.solve_ex(da, db, dc, dd, x, n, s, split_form=form, method=method, refine=True)
        torch.cuda.synchronize()
        err.append(rel(x.cpu().numpy(), ref, n))
    say(err)
    assert err[0] <= max(2 * err[1], 1e-7)


@pytest.mark.parametrize("n,s,nsys", [(65536, 256, 70), (524288, 512, 9)])
@pytest.mark.parametrize("method", ["ptpr", "tpr"])
def test_one_pass_weakly_dominant_accuracy(method, n, s, nsys):
    """More tiles than the device holds at once, weakly dominant."""
    say("one pass, weak", method, n, s, nsys)
    t = B.alloc_batch(nsys, n)
    B.generate("weak", 62, 0, nsys, n, t["a"], t["b"], t["c"], t["d"], t["xt"])
    a, b, c, d = (t[k].cpu().numpy() for k in "abcd")
    ref = O.thomas_f64_batch(a, b, c, d, n)
    err = {}
    for form in (0, 1):
        for refine in (False, True):
            B.solve_ex(t["a"], t["b"], t["c"], t["d"], t["x"], n, s, split_form=form, refine=refine, method=method)
            torch.cuda.synchronize()
            err[form, refine] = rel(t["x"].cpu().numpy(), ref, n)
    say(err)
    assert err[0, False] <= max(2 * err[1, False], 1e-6)
    assert err[0, True] <= max(2 * err[1, True], 1e-7)


def test_one_pass_nan_inputs_stay_in_their_system():
    """A NaN of every bit pattern in one system (the exchange marks words not
    yet published with one of them) ends the solve as usual and changes no
    other system."""
    n, nsys = 65536, 6
    a, b, c, d, _ = O.gen_batch(63, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    x = torch.zeros(nsys * n, device="cuda")
    B.solve_ex(da, db, dc, dd, x, n, 256)
    good = x.clone()
    dd.view(torch.int32)[2 * n:3 * n] = -1  # 0xffffffff
    dd[4 * n + 5] = float("inf")
    B.solve_ex(da, db, dc, dd, x, n, 256)
    torch.cuda.synchronize()
    assert bool(torch.isnan(x[2 * n:3 * n]).all())
    for k in (0, 1, 3, 5):
        assert np.array_equal(bits(x[k * n:(k + 1) * n]), bits(good[k * n:(k + 1) * n])), k


def _diag():
    L = ctypes.CDLL(build.DIAG_LIB)
    L.tprh_diag_split_fused.restype = ctypes.c_int
    return L


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("n,nsys,stride,parts,spin", [
    (65536, 3, 48, [(0, 48)], 0),            # every wait gives up at once
    (65536, 3, 16, [(0, 15), (15, 1)], 2),   # one workgroup comes after the others ended
    (65536, 3, 5, [(0, 1), (1, 4)], 1),      # fewer workgroups than tiles of a system, one first
    (1 << 19, 2, 96, [(0, 90), (90, 6)], 2),  # exchange by groups
    (1 << 19, 1, 16, [(3, 1), (0, 3), (4, 12)], 0),
])
def test_one_pass_sweeps_that_are_not_all_there(n, nsys, stride, parts, spin, refine):
    """The workgroups of one solve in several launches, one after the other
    (as when the device has no room for all of them): those that are there
    publish the absent ones' tiles and finish their own; the answers are the
    ordinary launch's bits."""
    if not os.path.exists(build.DIAG_LIB):
        pytest.fail("libtpr_diag.so is not built")
    say("partial sweeps", n, nsys, stride, parts, spin, refine)
    L = _diag()
    a, b, c, d, _ = O.gen_batch(64, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    x0 = dev(O.solve_batch("ptpr", a, b, c, d, n, 256)) * 1.001 if refine else torch.zeros(nsys * n, device="cuda")
    ref = x0.clone()
    B.solve_ex(da, db, dc, dd, ref, n, 256, refine=refine)
    ws = torch.empty(B.workspace_bytes(B.make_desc(da, db, dc, dd, ref, n, 256)), dtype=torch.uint8, device="cuda")
    x = x0.clone()
    torch.cuda.synchronize()
    p = ctypes.c_void_p
    for i, (first, blocks) in enumerate(parts):
        st = L.tprh_diag_split_fused(*(p(v.data_ptr()) for v in (da, db, dc, dd, x)), n, nsys, int(refine),
                                     p(ws.data_ptr()), int(i == 0), first, blocks, stride, spin, p(0))
        assert st == 0
        torch.cuda.synchronize()
    assert np.array_equal(bits(x), bits(ref))


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("n,nsys,stride,parts,spin", [
    (1 << 19, 1, 128, [(0, 64), (64, 64)], 0),    # whole groups of tiles absent, one tile per workgroup
    (1 << 19, 1, 128, [(32, 96), (0, 32)], 1),
    (1 << 17, 2, 64, [(0, 16), (16, 48)], 0),     # of one system one group, of the other none
    (1 << 19, 2, 256, [(112, 16), (128, 128), (0, 112)], 2),
])
def test_one_pass_sweeps_without_whole_groups(n, nsys, stride, parts, spin, refine):
    """Groups none of whose workgroups is there: each launch publishes their
    tiles and their groups and finishes its own."""
    test_one_pass_sweeps_that_are_not_all_there(n, nsys, stride, parts, spin, refine)


@pytest.mark.parametrize("n,nsys,stride,parts,spin", [
    (65536, 2, 16, [(0, 16)], 0),
    (65536, 3, 5, [(0, 1), (1, 4)], 0),
    (1 << 19, 2, 128, [(0, 128)], 0),
    (1 << 19, 1, 128, [(0, 64), (64, 64)], 1),
])
def test_one_pass_answers_over_the_right_hand_sides(n, nsys, stride, parts, spin):
    """x in d's own memory, with workgroups that publish each other's tiles:
    the bits of a solve into memory of its own."""
    say("in place", n, nsys, stride, parts, spin)
    L = _diag()
    a, b, c, d, _ = O.gen_batch(67, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    ref = torch.zeros_like(dd)
    B.solve_ex(da, db, dc, dd, ref, n, 256)
    whole = dd.clone()
    B.solve_ex(da, db, dc, whole, whole, n, 256)
    assert np.array_equal(bits(whole), bits(ref))
    ws = torch.empty(B.workspace_bytes(B.make_desc(da, db, dc, dd, ref, n, 256)), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    p = ctypes.c_void_p
    for i, (first, blocks) in enumerate(parts):
        st = L.tprh_diag_split_fused(*(p(v.data_ptr()) for v in (da, db, dc, dd, dd)), n, nsys, 0, p(ws.data_ptr()),
                                     int(i == 0), first, blocks, stride, spin, p(0))
        assert st == 0
        torch.cuda.synchronize()
    assert np.array_equal(bits(dd), bits(ref))


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("n,nsys,stride,first,blocks", [(65536, 2, 16, 0, 3), (1 << 17, 1, 32, 16, 2)])
def test_one_pass_tile_given_up_is_nan(n, nsys, stride, first, blocks, refine):
    """A workgroup that has used up its tasks answers its tiles with NaN; the
    tiles of those that never came keep what x held."""
    say("given up", n, nsys, stride, first, blocks, refine)
    L = _diag()
    L.tprh_diag_split_fused_bounded.restype = ctypes.c_int
    a, b, c, d, _ = O.gen_batch(66, 0, nsys, n)
    da, db, dc, dd = dev(a), dev(b), dev(c), dev(d)
    x = torch.full((nsys * n,), 2.5, device="cuda")
    ws = torch.empty(B.workspace_bytes(B.make_desc(da, db, dc, dd, x, n, 256)), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    p = ctypes.c_void_p
    st = L.tprh_diag_split_fused_bounded(*(p(v.data_ptr()) for v in (da, db, dc, dd, x)), n, nsys, int(refine),
                                         p(ws.data_ptr()), 1, first, blocks, stride, 0, nsys, p(0))
    assert st == 0
    torch.cuda.synchronize()
    tiles = x.view(-1, 4096)
    there = [k for k in range(nsys * n // 4096) if first <= k % stride < first + blocks]
    nan = torch.isnan(tiles).all(1).cpu().numpy()
    assert sorted(np.flatnonzero(nan)) == there
    assert bool((tiles[~torch.from_numpy(nan).cuda()] == 2.5).all())


def test_one_pass_in_a_graph_and_on_streams():
    """Replays of a captured solve, with eager work between them, and two
    solves overlapping on two streams: the eager answers' bits."""
    n, nsys = 65536, 80
    sets = []
    for k in range(2):
        t = B.alloc_batch(nsys, n)
        B.generate("dominant", 65 + k, 0, nsys, n, t["a"], t["b"], t["c"], t["d"], t["xt"])
        t["ws"] = torch.empty(B.workspace_bytes(B.make_desc(t["a"], t["b"], t["c"], t["d"], t["x"], n, 256)),
                              dtype=torch.uint8, device="cuda")
        sets.append(t)

    def solve(t, **kw):
        B.solve_ex(t["a"], t["b"], t["c"], t["d"], t["x"], n, 256, workspace=t["ws"], **kw)

    eager = []
    for t in sets:
        solve(t)
        eager.append(bits(t["x"]))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        solve(sets[0])
        solve(sets[1])
    for _ in range(4):
        for t in sets:
            t["x"].zero_()
            t["ws"].zero_()
        g.replay()
        torch.cuda.synchronize()
        for t, e in zip(sets, eager):
            assert np.array_equal(bits(t["x"]), e)
    streams = [torch.cuda.Stream() for _ in sets]
    for t in sets:
        t["x"].zero_()
    torch.cuda.synchronize()
    for _ in range(5):
        for t, st in zip(sets, streams):
            solve(t, stream=st)
    torch.cuda.synchronize()
    for t, e in zip(sets, eager):
        assert np.array_equal(bits(t["x"]), e)


def _masked_stream(cus):
    """A stream of default priority on the device's first `cus` CUs."""
    hip = ctypes.CDLL("libamdhip64.so")
    torch.zeros(1, device="cuda")
    words = (ctypes.c_uint32 * ((cus + 31) // 32))(*[(1 << min(32, cus - k)) - 1 for k in range(0, cus, 32)])
    st = ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(st), len(words), words) == 0
    return torch.cuda.ExternalStream(st.value), lambda: hip.hipStreamDestroy(st)


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("n,s,nsys,form", [(65536, 256, 20, 0), (1 << 20, 512, 1, 1)])
def test_one_pass_on_a_stream_with_a_cu_mask(n, s, nsys, form, refine):
    """On 32 CUs: systems that their workgroups hold at once take one pass,
    larger ones two (form: whose bits, on the whole device, the answers are)."""
    say("CU mask", n, s, nsys, refine)
    t = B.alloc_batch(nsys, n)
    B.generate("dominant", 69, 0, nsys, n, t["a"], t["b"], t["c"], t["d"], t["xt"])
    args = (t["a"], t["b"], t["c"], t["d"], t["x"], n, s)
    ws = torch.empty(B.workspace_bytes(B.make_desc(*args)), dtype=torch.uint8, device="cuda")
    got = {}
    st, destroy = _masked_stream(32)
    for name, f, stream in (("one", 0, None), ("two", 1, None), ("masked", 0, st)):
        t["x"].copy_(t["xt"] * 1.001)
        torch.cuda.synchronize()
        B.solve_ex(*args, refine=refine, split_form=f, workspace=ws, stream=stream)
        torch.cuda.synchronize()
        got[name] = bits(t["x"])
    destroy()
    assert not np.array_equal(got["one"], got["two"])
    assert np.array_equal(got["masked"], got["two" if form else "one"])


@pytest.mark.parametrize("handle", [0, 1, 2])
def test_one_pass_on_the_null_streams(handle):
    """The null stream by its handles (default, legacy, per thread)."""
    say("null stream", handle)
    n, nsys = 65536, 2
    t = B.alloc_batch(nsys, n)
    B.generate("dominant", 70, 0, nsys, n, t["a"], t["b"], t["c"], t["d"], t["xt"])
    args = (t["a"], t["b"], t["c"], t["d"], t["x"], n, 256)
    ws = torch.empty(B.workspace_bytes(B.make_desc(*args)), dtype=torch.uint8, device="cuda")
    B.solve_ex(*args, workspace=ws)
    torch.cuda.synchronize()
    want = bits(t["x"])
    t["x"].zero_()
    torch.cuda.synchronize()
    B.solve_ex(*args, workspace=ws, stream=types.SimpleNamespace(cuda_stream=handle))
    torch.cuda.synchronize()
    assert np.array_equal(bits(t["x"]), want)


def test_one_pass_refuses_a_destroyed_stream():
    """As a launch does: an error, before anything runs."""
    say("destroyed stream")
    n, nsys = 65536, 2
    t = B.alloc_batch(nsys, n)
    B.generate("dominant", 71, 0, nsys, n, t["a"], t["b"], t["c"], t["d"], t["xt"])
    args = (t["a"], t["b"], t["c"], t["d"], t["x"], n, 256)
    ws = torch.empty(B.workspace_bytes(B.make_desc(*args)), dtype=torch.uint8, device="cuda")
    t["x"].fill_(2.5)
    st, destroy = _masked_stream(64)
    torch.cuda.synchronize()
    assert destroy() == 0
    with pytest.raises(_lib.TprError):
        B.solve_ex(*args, workspace=ws, stream=types.SimpleNamespace(cuda_stream=st.cuda_stream))
    torch.cuda.synchronize()
    assert bool((t["x"] == 2.5).all())
    B.solve_ex(*args, workspace=ws)
    torch.cuda.synchronize()
    assert rel(t["x"].cpu().numpy(), t["xt"].cpu().numpy(), n) <= FAST_TOL
