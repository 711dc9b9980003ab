"""The work that a user of this framework has it do, as cases that can be timed.

Kinds of case (sizes are powers of two per system, as the solver takes them;
the number of systems is any):

  host     one system in host arrays through the drop-in `ptpr_cu` / `tpr_cu`
           (the reference's documented run is N = 2048, S = 512)
  batch    equal systems resident on the device, `solve_batched`
  f16      the same with a, b, c stored in fp16, `solve_ex`
  refine   one FP64-residual refinement step of an fp32 solution, `solve_ex`
  mixed    the precision run: an fp16-stored solve, then a refinement step
           with the fp32 coefficients
  adi      many right-hand sides of one matrix (`solve_ex`, shared)
  uneven   systems of many sizes in one launch, `UnevenPlan.solve`
  serve    a burst of requests against resident matrices, `Server`

f16, refine, mixed and adi take systems above one workgroup as batch does
not (through the workspace that `solve_ex` allocates).
"""
import random

import numpy as np
import torch

import tpr_amd
from tpr_amd import batched, serve, uneven

MAX_LANES = 1024  # lanes of one workgroup: n / s times the lanes of a slice


def listed():
    return [
        # the reference's documented run, one solve per call from host arrays
        {"name": "host_2048_s512", "kind": "host", "method": "ptpr", "n": 2048, "s": 512},
        # the smallest device call: one system, where launch and host cost count
        {"name": "one_1024", "kind": "batch", "method": "ptpr", "arith": "fast", "n": 1024, "s": 256, "nsys": 1,
         "unit": False, "weak": False},
        # the headline batch
        {"name": "batch_4096x1024", "kind": "batch", "method": "ptpr", "arith": "fast", "n": 1024, "s": 256,
         "nsys": 4096, "unit": False, "weak": False},
        # the other method, a unit diagonal as the reference's GPU entry points have, an odd count
        {"name": "tpr_unit_4093x1024", "kind": "batch", "method": "tpr", "arith": "fast", "n": 1024, "s": 256,
         "nsys": 4093, "unit": True, "weak": False},
        # bit parity with the reference's CPU solver, at the headline size
        {"name": "exact_4096x1024", "kind": "batch", "method": "ptpr", "arith": "exact", "n": 1024, "s": 256,
         "nsys": 4096, "unit": False, "weak": False},
        # the documented run's slice size, batched, an odd count
        {"name": "s512_2047x2048", "kind": "batch", "method": "ptpr", "arith": "fast", "n": 2048, "s": 512,
         "nsys": 2047, "unit": False, "weak": False},
        # systems of N = 2^U{8..14}: the largest case
        {"name": "uneven_20000", "kind": "uneven", "method": "ptpr", "arith": "fast", "nsys": 20000, "lo": 8,
         "hi": 14},
        # systems above one workgroup, weakly dominant: the fp32 solve of the precision run
        {"name": "large_256x65536", "kind": "large", "method": "ptpr", "arith": "fast", "n": 65536, "s": 256,
         "nsys": 256, "weak": True},
        # the whole precision run: fp16-stored solve and one refinement step
        {"name": "mixed_256x65536", "kind": "mixed", "method": "ptpr", "n": 65536, "s": 256, "nsys": 256,
         "weak": True},
        # an ADI sweep over a grid: the lines are right-hand sides of one matrix
        {"name": "adi_4095x4096", "kind": "adi", "method": "ptpr", "n": 4096, "s": 256, "nsys": 4095},
        # a burst of requests as the serving loop gets them: N = 2^U{9..15}, 1..64 right-hand sides each
        {"name": "serve_48", "kind": "serve", "requests": 48, "lo": 9, "hi": 15, "rhs": 64},
        # one large system
        {"name": "large_1x1048576", "kind": "large", "method": "ptpr", "arith": "fast", "n": 1 << 20, "s": 1024,
         "nsys": 1, "weak": False},
    ]


def _log_uniform(rng, lo, hi):
    """A whole number of lo .. hi, uniform in its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _slice(rng, n, lo=16, hi=2048):
    """A slice size of lo .. hi that one workgroup takes for systems of n."""
    sizes = [s for s in (16, 32, 64, 128, 256, 512, 1024, 2048)
             if lo <= s <= min(n, hi) and (n // s) * (16 if s <= 256 else 32 if s == 512 else 64) <= MAX_LANES]
    # 256 and 512 are the slice sizes in use; the others appear too
    common = [s for s in sizes if s in (256, 512)]
    return rng.choice(common) if common and rng.random() < 0.5 else rng.choice(sizes)


def draw(rng):
    kind = rng.choice(["host", "batch", "batch", "batch", "f16", "refine", "mixed", "adi", "uneven", "serve", "large",
                       "large"])
    method = rng.choice(["ptpr", "ptpr", "tpr"])
    arith = rng.choice(["fast", "fast", "exact"])
    if kind == "host":
        n = 1 << rng.randint(9, 16)
        return {"kind": kind, "method": method, "n": n, "s": rng.choice([v for v in (64, 128, 256, 512) if v * v >= n])}
    if kind in ("batch", "f16", "refine"):
        n = 1 << rng.randint(6, 14)
        c = {"kind": kind, "method": method, "arith": arith, "n": n, "s": _slice(rng, n),
             "nsys": _log_uniform(rng, 1, (8 << 20) // n), "unit": rng.random() < 0.25,
             "weak": kind != "f16" and rng.random() < 0.25}
        return c
    if kind == "uneven":
        lo = rng.randint(6, 10)
        return {"kind": kind, "method": method, "arith": arith, "nsys": _log_uniform(rng, 50, 20000), "lo": lo,
                "hi": rng.randint(lo + 1, 14)}
    if kind == "adi":
        n = 1 << rng.randint(8, 16)
        return {"kind": kind, "method": method, "n": n, "s": 256, "nsys": _log_uniform(rng, 2, (16 << 20) // n)}
    if kind == "serve":
        return {"kind": kind, "requests": _log_uniform(rng, 1, 64), "lo": 9, "hi": rng.randint(10, 15),
                "rhs": _log_uniform(rng, 1, 64)}
    # above one workgroup: up to 16 Mi equations
    n = 1 << rng.randint(16, 20)
    s = rng.choice([s for s in (256, 512, 1024, 2048) if n // s <= 2048])
    c = {"kind": kind, "method": method, "n": n, "s": s, "nsys": _log_uniform(rng, 1, (16 << 20) // n),
         "weak": rng.random() < 0.5}
    if kind == "large":
        c["arith"] = arith
    return c


# ---------------------------------------------------------------------------
# Inputs: the benchmark generators (a, c ~ U(-1, 1), b = |a| + |c| + (1 + u) or,
# weakly dominant, + (1e-4 + 0.0099 u); truth ~ U(-1, 1), d = A x), for systems
# of the given sizes back to back.

def _sizes(case):
    if case["kind"] == "uneven":
        r = random.Random(case["nsys"] * 1000 + case["lo"] * 20 + case["hi"])
        return [1 << r.randint(case["lo"], case["hi"]) for _ in range(case["nsys"])]
    if case["kind"] in ("host", "adi"):
        return [case["n"]]
    return [case["n"]] * case["nsys"]


def _requests(case):
    """(n, right-hand sides) of each request of a serve case."""
    r = random.Random(case["requests"] * 1000 + case["hi"] * 70 + case["rhs"])
    return [(1 << r.randint(case["lo"], case["hi"]), r.randint(1, case["rhs"])) for _ in range(case["requests"])]


def _apply(a, b, c, x):
    """A x in 64 bits; a is 0 at every first and c at every last equation."""
    y = b.double() * x
    y[1:] += a[1:].double() * x[:-1]
    y[:-1] += c[:-1].double() * x[1:]
    return y


def _systems(sizes, seed, weak=False, unit=False, f16=False):
    """a, b, c, d on the GPU; unit: rows divided by the diagonal, b is ones."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    ends = torch.as_tensor(np.cumsum(np.asarray(sizes, np.int64)), device="cuda")
    total = int(sum(sizes))

    def uniform():
        return torch.rand(total, generator=g, device="cuda") * 2 - 1

    a, c = uniform(), uniform()
    a[0] = 0
    a[ends[:-1]] = 0
    c[ends - 1] = 0
    u = torch.rand(total, generator=g, device="cuda")
    b = a.abs() + c.abs() + (1e-4 + 0.0099 * u if weak else 1 + u)
    if unit:
        a, c, b = a / b, c / b, torch.ones_like(b)
    if f16:  # stored values that fp16 holds: the system is the stored one
        a, b, c = (v.half() for v in (a, b, c))
    d = _apply(a, b, c, uniform().double()).float()
    return a, b, c, d


def _rhs(count, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed ^ 0x5EED)
    return torch.rand(count, generator=g, device="cuda") * 2 - 1


def _inputs(case, seed):
    kind = case["kind"]
    if kind == "host":
        a, b, c, d = _systems(_sizes(case), seed, unit=True)
        return a, b, c, d
    if kind == "adi":
        a, b, c, _ = _systems(_sizes(case), seed)
        return a, b, c, _rhs(case["n"] * case["nsys"], seed)
    if kind == "serve":
        reqs = _requests(case)
        a, b, c, _ = _systems([n for n, _ in reqs], seed)
        return a, b, c, _rhs(sum(n * k for n, k in reqs), seed)
    return _systems(_sizes(case), seed, case.get("weak", False), case.get("unit", False), kind == "f16")


def prepare(case, seed):
    kind = case["kind"]
    a, b, c, d = _inputs(case, seed)
    st = dict(case, a=a, b=None if case.get("unit") else b, c=c, d=d, x=torch.zeros_like(d))
    if kind == "host":
        st.update(a=a.cpu().numpy(), c=c.cpu().numpy(), d=d.cpu().numpy(), x=np.zeros(case["n"], np.float32))
        st["call"] = {"ptpr": tpr_amd.ptpr_cu, "tpr": tpr_amd.tpr_cu}[case["method"]]
    elif kind == "refine":
        # an iterate with the error of a solve from rounded coefficients; each
        # pass starts from a copy of it, since the step updates x in place
        st["x0"] = _solve64(a, b, c, d, case["n"]).float() * (1 + 1e-3 * _rhs(d.numel(), seed + 1))
    elif kind == "mixed":
        st["h"] = [v.half() for v in (a, b, c)]
    elif kind == "uneven":
        st["plan"] = uneven.UnevenPlan(_sizes(case), method=case["method"], arith=case["arith"])
    elif kind == "serve":
        srv = serve.Server(2 << 30)
        torch.cuda.synchronize()  # the uploads below run on the server's stream
        st["reqs"], at, rt = [], 0, 0
        for n, k in _requests(case):
            m = srv.matrix_upload(a[at:at + n], b[at:at + n], c[at:at + n])
            st["reqs"].append((m, k, d[rt:rt + n * k], st["x"][rt:rt + n * k]))
            at, rt = at + n, rt + n * k
        st["srv"] = srv
    if kind in ("large", "mixed"):
        # the workspace that a program with a fixed batch keeps
        desc = batched.make_desc(a, b, c, d, st["x"], case["n"], case["s"], case["method"], case.get("arith", "fast"))
        need = batched.workspace_bytes(desc)
        st["ws"] = torch.empty(max(1, need), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    return st


def run(st):
    kind = st["kind"]
    if kind == "host":
        st["call"](st["a"], st["c"], st["d"], st["x"], st["n"], st["s"])
        return st["x"]
    if kind == "batch":
        return tpr_amd.solve_batched(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"],
                                     method=st["method"], arith=st["arith"])
    if kind == "f16":
        return batched.solve_ex(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"], method=st["method"],
                                arith=st["arith"])
    if kind == "refine":
        st["x"].copy_(st["x0"])
        return batched.solve_ex(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"], method=st["method"],
                                arith=st["arith"], refine=True)
    if kind == "adi":
        return batched.solve_ex(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"], method=st["method"],
                                shared=True)
    if kind == "large":
        return batched.solve_ex(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"], method=st["method"],
                                arith=st["arith"], workspace=st["ws"])
    if kind == "mixed":
        ha, hb, hc = st["h"]
        batched.solve_ex(ha, hb, hc, st["d"], st["x"], st["n"], st["s"], method=st["method"], workspace=st["ws"])
        return batched.solve_ex(st["a"], st["b"], st["c"], st["d"], st["x"], st["n"], st["s"], method=st["method"],
                                refine=True, workspace=st["ws"])
    if kind == "uneven":
        return st["plan"].solve(st["a"], st["b"], st["c"], st["d"], st["x"])
    srv = st["srv"]
    ids = [srv.submit(m, k, d=d, x=x) for m, k, d, x in st["reqs"]]
    for r in ids:
        srv.wait(r)
        srv.release(r)
    return st["x"]


def work(case):
    """Each input read once and x written once; nine operations an equation
    (the elimination and back-substitution of one right-hand side)."""
    kind = case["kind"]
    if kind == "serve":
        reqs = _requests(case)
        eq = sum(n * k for n, k in reqs)
        return {"bytes": 12 * sum(n for n, _ in reqs) + 8 * eq, "flops": 9 * eq}
    if kind == "adi":
        eq = case["n"] * case["nsys"]
        return {"bytes": 12 * case["n"] + 8 * eq, "flops": 9 * eq}
    eq = sum(_sizes(case))
    per = {"host": 16, "f16": 14, "refine": 24, "mixed": 14 + 24}.get(kind, 20)
    if case.get("unit"):
        per -= 2 if kind == "f16" else 4
    return {"bytes": per * eq, "flops": (18 if kind == "mixed" else 9) * eq}


# ---------------------------------------------------------------------------
# The answers in 64 bits: cyclic reduction of every row at once (each level
# doubles the distance between a row and its neighbours), for any sizes back
# to back, since no row couples across the end of a system.

def _shift(v, k, fill):
    """v[i - k] (k > 0) or v[i + |k|], with `fill` past the ends."""
    w = torch.full_like(v, fill)
    if k > 0:
        w[k:] = v[:-k]
    else:
        w[:k] = v[-k:]
    return w


def _solve64(a, b, c, d, longest):
    a, b, c, d = (v.double() for v in (a, b, c, d))
    k = 1
    while k < longest:
        al = -a / _shift(b, k, 1.0)
        ga = -c / _shift(b, -k, 1.0)
        b = b + al * _shift(c, k, 0.0) + ga * _shift(a, -k, 0.0)
        d = d + al * _shift(d, k, 0.0) + ga * _shift(d, -k, 0.0)
        a, c = al * _shift(a, k, 0.0), ga * _shift(c, -k, 0.0)
        k *= 2
    return d / b


def exact(case, seed):
    a, b, c, d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "adi":
        reqs = [(case["n"], case["nsys"])]
    elif kind == "serve":
        reqs = _requests(case)
    else:
        x = _solve64(a, b, c, d, max(_sizes(case)))
        return x.cpu().numpy() if kind == "host" else x
    out, at, rt = [], 0, 0
    for n, k in reqs:
        m = [v[at:at + n].repeat(k) for v in (a, b, c)]
        out.append(_solve64(*m, d[rt:rt + n * k], n))
        at, rt = at + n, rt + n * k
    return torch.cat(out)
