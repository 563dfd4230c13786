"""Performance cases of the TapasFMM library: the evaluations its users run.

Every case goes through the public binding (tapas-reduce_amd/tfmm.py, a thin
layer over the C ABI).  A program keeps one context per stream of problems,
with its kernel knobs set once, and evaluates bodies that lie on the GPU; the
drop-in path hands over host bodies and takes host fields back.  A pass is the
whole evaluation (tree, upward, traversal, M2L, P2P, downward) with the fields
delivered.  FP64 evaluations return FP64 fields.  Mixed precision computes its
interactions in FP32, and a program that chose it keeps the fields in FP32.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tapas-reduce_amd"))

import datasets  # noqa: E402
import tfmm  # noqa: E402

# The kernel knobs of a program that has tuned them once for its bodies:
# one M2L work unit per tile, the P2P started early as 3 resident waves.
TUNED = {"unit": 0.0, "xcd_run": 8, "p2p_schedule": 2, "p2p_waves": 3}
# the library's own defaults
PLAIN = {"unit": 0.0, "xcd_run": 32, "p2p_schedule": 0, "p2p_waves": 0}


def _case(kind, n, dist="cube", precision="fp64", ncrit=64, theta=0.4, mutual=0, basis="spherical",
          images=0, graph=0, tuned=False, problems=1, targets=0, name=None):
    c = dict(kind=kind, n=n, dist=dist, precision=precision, ncrit=ncrit, theta=theta,
             mutual=mutual, basis=basis, images=images, graph=graph, tuned=tuned,
             problems=problems, targets=targets)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one small problem at a time (a few leaves): launches and latency
        _case("device", 4096, name="cube_4k"),
        # a small time-stepping loop, every step one graph launch
        _case("device", 16384, graph=2, name="cube_16k_graph"),
        # the drop-in path: host array-of-structs bodies in, host fields out
        _case("host", 65537, dist="ellipsoid", name="ellipsoid_64k_host"),
        # an ordinary clustered problem, each pair visited once (mutual)
        _case("device", 262144, dist="plummer", precision="mixed", mutual=1, name="plummer_256k"),
        # an ordinary flat, uneven problem of ragged size in FP64
        _case("device", 500009, dist="ellipsoid", name="ellipsoid_500k"),
        # a uniform million bodies in FP64
        _case("device", 1048576, name="cube_1m"),
        # the headline workload, knobs tuned once
        _case("device", 4194304, dist="plummer", precision="mixed", ncrit=128, theta=0.418,
              tuned=True, name="plummer_4m"),
        # the largest: two clusters
        _case("device", 8388608, dist="two_plummer", precision="mixed", ncrit=128, theta=0.421,
              tuned=True, name="two_plummer_8m"),
        # many independent problems as one forest
        _case("batch", 0, precision="mixed", ncrit=128, tuned=True, problems=256,
              name="batch_256"),
        # the Cartesian Taylor basis
        _case("device", 300000, basis="cartesian", name="cartesian_300k"),
        # periodic boundary conditions with far copies
        _case("device", 100003, images=2, name="periodic_100k"),
        # the accuracy check of a run: direct sums at sampled targets
        _case("direct", 1048576, dist="plummer", targets=4096, name="direct_1m"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["device"] * 6 + ["batch", "direct", "host"])
    dist = rng.choice(["cube", "plummer", "ellipsoid", "two_plummer"])
    precision = rng.choice(["fp64", "mixed"])
    ncrit = rng.choice([32, 64, 128])
    theta = round(rng.uniform(0.36, 0.5), 3)
    if kind == "host":
        return _case(kind, _log_int(rng, 1000, 300000), dist, precision, ncrit, theta)
    if kind == "direct":
        return _case(kind, _log_int(rng, 10000, 2000000), dist,
                     targets=_log_int(rng, 100, 4096))
    if kind == "batch":
        return _case(kind, 0, "cube", precision, 128, theta, tuned=precision == "mixed",
                     problems=_log_int(rng, 4, 128))
    if rng.random() < 0.15:
        return _case(kind, _log_int(rng, 1000, 500000), dist, "fp64", ncrit, theta,
                     basis="cartesian")
    if rng.random() < 0.15:
        return _case(kind, _log_int(rng, 1000, 300000), "cube", precision, ncrit, theta,
                     images=rng.choice([1, 2]))
    n = _log_int(rng, 1000, 2000000 if precision == "fp64" else 4000000)
    return _case(kind, n, dist, precision, ncrit if n < 1000000 else max(ncrit, 64), theta,
                 mutual=rng.choice([0, 0, 1]), graph=rng.choice([0, 0, 0, 2]),
                 tuned=precision == "mixed" and n >= 1000000)


def _sizes(case):
    """Body counts (log-uniform in [2^10, 2^16]) and distributions of a batch's
    problems: part of the case, whatever the bodies."""
    rng = np.random.Generator(np.random.PCG64(case["problems"]))
    n = np.exp(rng.uniform(math.log(1 << 10), math.log(1 << 16), case["problems"])).astype(int)
    return n, rng.integers(0, 3, case["problems"])


def _problems(case, seed):
    """The bodies (x, y, z, q) of every problem, on the host."""
    if case["kind"] != "batch":
        return [datasets.make(case["dist"], case["n"], seed=seed)]
    out = []
    for p, (n, d) in enumerate(zip(*_sizes(case))):
        kw = {} if d == 0 else {"charges": "uniform"}
        out.append(datasets.make(("cube", "plummer", "ellipsoid")[d], int(n),
                                 seed=seed * 65536 + p, **kw))
    return out


def _targets(case, seed, n):
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    return np.sort(rng.choice(n, size=min(n, case["targets"]), replace=False)).astype(np.int64)


def prepare(case, seed):
    probs = _problems(case, seed)
    off = np.zeros(len(probs) + 1, np.int64)
    off[1:] = np.cumsum([len(p[0]) for p in probs])
    ctx = tfmm.Context(0)
    knobs = TUNED if case["tuned"] else PLAIN
    ctx.set_tuning(tfmm.TUNE_M2L_UNIT, knobs["unit"])
    ctx.set_tuning(tfmm.TUNE_M2L_XCD_RUN, knobs["xcd_run"])
    ctx.set_tuning(tfmm.TUNE_P2P_SCHEDULE, knobs["p2p_schedule"])
    ctx.set_tuning(tfmm.TUNE_P2P_WAVES, knobs["p2p_waves"])
    ctx.set_tuning(tfmm.TUNE_GRAPH, case["graph"])
    if case["basis"] == "cartesian":
        ctx.set_basis(tfmm.BASIS_CARTESIAN)
    if case["images"]:
        ctx.set_periodic(case["images"], 1.0)  # the cube's own period
    mixed = case["precision"] == "mixed"
    st = dict(case=case, ctx=ctx, params=tfmm.make_params(
        case["ncrit"], case["theta"], tfmm.MIXED if mixed else tfmm.FP64, case["mutual"]))
    if case["kind"] == "host":
        st["host"] = [np.ascontiguousarray(a) for a in probs[0]]
        return st
    n = int(off[-1])
    st["bodies"] = [torch.from_numpy(np.concatenate([p[k] for p in probs])).cuda()
                    for k in range(4)]
    torch.cuda.synchronize()
    ptrs = [t.data_ptr() for t in st["bodies"]]
    if case["kind"] == "batch":
        ctx.set_batch_device(off, *ptrs)
    else:
        ctx.set_bodies_device(n, *ptrs)
    if case["kind"] == "direct":
        st["targets"] = _targets(case, seed, n)
    else:
        st["fields"] = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    return st


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "direct":
        return ctx.direct(state["targets"])
    if case["kind"] == "host":
        ctx.set_bodies(*state["host"])
        ctx.evaluate(state["params"])
        f = ctx.fields()
        return f.astype(np.float32) if case["precision"] == "mixed" else f
    ctx.evaluate(state["params"])
    ctx.fields_to_device(state["fields"].data_ptr())
    return state["fields"].float() if case["precision"] == "mixed" else state["fields"]


def _bodies(case):
    return float(_sizes(case)[0].sum()) if case["kind"] == "batch" else case["n"]


def work(case):
    """Bodies read and fields written once; the near-field pairs (20 flops
    each) and M2L pairs (9,680 flops each) of an evaluation at these ncrit and
    theta (per body and per leaf as measured on the uniform and clustered
    trees of the listed cases, within about 30 %)."""
    n = _bodies(case)
    if case["kind"] == "direct":
        return {"bytes": 32.0 * n + 40.0 * case["targets"],
                "flops": 20.0 * n * case["targets"]}
    scale = (0.4 / case["theta"]) ** 3
    p2p = n * min(n, 30.0 * case["ncrit"] * scale)
    leaves = n / (0.4 * case["ncrit"])
    m2l = leaves * min(leaves, 160.0 * scale)
    out = 16 if case["precision"] == "mixed" else 32
    return {"bytes": (32.0 + out) * n, "flops": 20.0 * p2p + 9680.0 * m2l}


EXACT_PAIRS = 1.5e11  # what a plain direct sum gets through in a few seconds


def _direct(x, y, z, q, at):
    """pot and acceleration at the bodies `at` from all bodies, 64 bits."""
    src = torch.stack([q, q * x, q * y, q * z], 1)
    out = torch.empty((at.numel(), 4), dtype=torch.float64, device=x.device)
    rows = max(1, (1 << 27) // x.numel())
    for a in range(0, at.numel(), rows):
        i = at[a:a + rows]
        r2 = (x[i, None] - x[None, :]).square_()
        d = y[i, None] - y[None, :]
        r2.addcmul_(d, d)
        torch.sub(z[i, None], z[None, :], out=d)
        r2.addcmul_(d, d)
        r2.masked_fill_(r2 == 0, math.inf)
        w = r2.rsqrt_()
        out[a:a + rows, 0] = w @ q
        torch.mul(w, w, out=d)
        w.mul_(d)
        s = w @ src
        for k, c in enumerate((x, y, z)):
            out[a:a + rows, 1 + k] = s[:, 1 + k] - c[i] * s[:, 0]
    return out


def exact(case, seed):
    probs = _problems(case, seed)
    pairs = sum(float(len(p[0])) ** 2 for p in probs)
    if case["kind"] == "direct":
        pairs = float(case["n"]) * case["targets"]
    if case["images"] or pairs > EXACT_PAIRS:
        return None
    out = []
    for p in probs:
        x, y, z, q = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in p)
        if case["kind"] == "direct":
            at = torch.from_numpy(_targets(case, seed, len(p[0]))).cuda()
        else:
            at = torch.arange(x.numel(), device="cuda")
        out.append(_direct(x, y, z, q, at))
    r = torch.cat(out)
    return r.cpu().numpy() if case["kind"] in ("direct", "host") else r
