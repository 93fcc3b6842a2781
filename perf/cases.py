"""What the speed of this library is measured on.

Each case is one piece of work that a program using amuse_amd has it do,
through the public Python entry points, at a size and precision in the range
such programs use:

  calc      G6.set_j_particles + set_ti + calc: load a list of field particles
            and ask for the forces on a group (BHtree's interaction lists, the
            first force of a worker, a GRAPE call with everything new)
  pass      the same with the field particles themselves as the group
            (calc_self + fetch): the forces of a whole snapshot
  blocks    DeviceHermite4.evolve: ph4's block-step integration over an output
            interval, then the state
  ensemble  Ensemble.start + run + state: a few shared step rounds of many
            small clusters
  pair      pair_force and its gradients (a loss on accelerations and jerks)
  hermite   hermite_integrate and the gradients of a loss on the final state

The mixed path computes forces in FP32, so a program that chooses it keeps
its results in float32 arrays; the FP64 path's results are kept in float64.
"""
import math

import numpy as np
import torch

from amuse_amd import ic
from amuse_amd.blocks import DeviceHermite4
from amuse_amd.diff import hermite_integrate, pair_force
from amuse_amd.ensemble import Ensemble
from amuse_amd.g6 import FP64, MIXED, G6

EPS2 = 1e-4          # softening of the c0/c1 systems
EPS2_CLUSTERS = 1e-6
DT_PARAM = 0.03      # the ensembles' step parameter
KROUPA = (0.08, 20.0)

# ranges of the drawn cases
CALC_NJ, CALC_NI = (500, 60000), (16, 4000)
PASS_N = (8192, 200000)
BLOCKS_N = (256, 60000)
CLUSTERS = (32, 512)
PAIR_N = (500, 20000)


def listed():
    return [
        # a group of a tree code against a short interaction list: launches
        # and host work are the whole cost
        {"name": "calc_fp64_1k", "kind": "calc", "nj": 1000, "ni": 64, "prec": "fp64"},
        # a long list against a large group, no size a multiple of a tile
        {"name": "calc_mixed_30k", "kind": "calc", "nj": 30011, "ni": 1501, "prec": "mixed"},
        # potentials and forces of a 64k snapshot, reference precision
        {"name": "pass_fp64_64k", "kind": "pass", "n": 65536, "prec": "fp64"},
        # the same for a large system in the mixed path
        {"name": "pass_mixed_256k", "kind": "pass", "n": 262144, "prec": "mixed"},
        # ph4's standard small run (N = 1024, eta = 0.01): small blocks, one
        # after another
        {"name": "blocks_fp64_1k", "kind": "blocks", "n": 1024, "prec": "fp64", "lg_dt": -9},
        # the same code at a size whose blocks fill part of the chip
        {"name": "blocks_fp64_16k", "kind": "blocks", "n": 16384, "prec": "fp64", "lg_dt": -11},
        # a large mixed run at ph4's default eta
        {"name": "blocks_mixed_50k", "kind": "blocks", "n": 50021, "prec": "mixed", "lg_dt": -9},
        # cluster ensembles, 16 to 2048 particles each
        {"name": "ensemble_mixed_512", "kind": "ensemble", "nc": 512, "rounds": 16,
         "prec": "mixed"},
        {"name": "ensemble_fp64_100", "kind": "ensemble", "nc": 100, "rounds": 16,
         "prec": "fp64"},
        # a differentiable force evaluation, forward and backward
        {"name": "pair_fp64_5k", "kind": "pair", "n": 5003, "prec": "fp64"},
        {"name": "pair_fp32_16k", "kind": "pair", "n": 16384, "prec": "fp32"},
        # gradient of a short integration (checkpointed)
        {"name": "hermite_fp32_8k", "kind": "hermite", "n": 8192, "steps": 8, "prec": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["calc", "pass", "blocks", "ensemble", "pair", "hermite"])
    if kind == "calc":
        return {"kind": kind, "nj": _log_int(rng, *CALC_NJ), "ni": _log_int(rng, *CALC_NI),
                "prec": rng.choice(["fp64", "mixed"])}
    if kind == "pass":
        return {"kind": kind, "n": _log_int(rng, *PASS_N), "prec": rng.choice(["fp64", "mixed"])}
    if kind == "blocks":
        n = _log_int(rng, *BLOCKS_N)
        prec = rng.choice(["fp64", "mixed"])
        lg = (-9 if n < 4000 else -11 if n < 20000 else -13) if prec == "fp64" else -9
        return {"kind": kind, "n": n, "prec": prec, "lg_dt": lg}
    if kind == "ensemble":
        return {"kind": kind, "nc": _log_int(rng, *CLUSTERS), "rounds": rng.choice([8, 16]),
                "prec": rng.choice(["fp64", "mixed"])}
    if kind == "pair":
        return {"kind": kind, "n": _log_int(rng, *PAIR_N), "prec": rng.choice(["fp32", "fp64"])}
    return {"kind": kind, "n": _log_int(rng, PAIR_N[0], PAIR_N[1] // 2),
            "steps": rng.choice([3, 4, 8]), "prec": rng.choice(["fp32", "fp64"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_unit = None


def _g6():
    """The process's GRAPE-6 unit, opened anew (an empty particle store)."""
    global _unit
    if _unit is None:
        _unit = G6(0)
    _unit.open()
    return _unit


def _plummer(n, seed):
    """Plummer sphere in N-body units with a Salpeter mass spectrum."""
    rng = np.random.Generator(np.random.PCG64(seed))
    _, x, v = ic.plummer_raw(n, rng)
    x, v = ic.to_nbody_units(x, v)
    m = ic.salpeter(n, rng)
    m /= m.sum()
    x, v = ic.center(m, x, v)
    return rng, m, x, v


def _field(case, seed):
    """Field particles with their predictor terms, and the group's rows."""
    n = case["nj"] if case["kind"] == "calc" else case["n"]
    rng, m, x, v = _plummer(n, seed)
    f = {"n": n, "m": m, "x": x, "v": v, "ti": 1.0, "ids": np.arange(1, n + 1, dtype=np.int32),
         "addr": np.arange(n, dtype=np.int32)}
    # particles last stepped up to 1/64 ago, each predicted to ti
    f["tj"] = 1.0 - rng.integers(0, 5, n) / 256.0
    f["a2"] = rng.normal(0.0, 0.2, (n, 3))
    f["j6"] = rng.normal(0.0, 0.2, (n, 3))
    f["k18"] = np.zeros((n, 3))
    if case["kind"] == "calc":
        sel = np.sort(rng.choice(n, min(case["ni"], n), replace=False))
        dt = (f["ti"] - f["tj"][sel])[:, None]
        f["sel"] = sel
        f["id_i"] = f["ids"][sel]
        f["xi"] = x[sel] + v[sel] * dt + f["a2"][sel] * dt ** 2 + f["j6"][sel] * dt ** 3
        f["vi"] = v[sel] + 2 * f["a2"][sel] * dt + 3 * f["j6"][sel] * dt ** 2
    return f


def _clusters(case, seed):
    """Plummer clusters with Kroupa masses, M = 1 each, their sizes spread
    evenly in the logarithm over 16..2048 (the same for every seed), in no
    order."""
    nc = case["nc"]
    counts = np.rint(np.exp(np.linspace(math.log(16), math.log(2048), nc))).astype(np.int32)
    counts = counts[np.random.Generator(np.random.PCG64(nc)).permutation(nc)]
    total = int(counts.sum())
    rng = np.random.Generator(np.random.PCG64(seed))
    _, x, v = ic.plummer_raw(total, rng)
    x, v = ic.to_nbody_units(x, v)
    m = ic.kroupa(total, rng, *KROUPA)
    off = 0
    for n in counts.tolist():
        s = slice(off, off + n)
        m[s] /= m[s].sum()
        x[s], v[s] = ic.center(m[s], x[s], v[s])
        off += n
    return counts, m, x, v


def _prec(case):
    return MIXED if case["prec"] == "mixed" else FP64


def _eta(case):
    # ph4's default step parameter in the mixed path (its FP32 forces do not
    # carry the small one), the accurate setting of the small runs in FP64
    return 0.14 if case["prec"] == "mixed" else 0.01


def _tensors(case, seed):
    _, m, x, v = _plummer(case["n"], seed)
    dtype = torch.float32 if case["prec"] == "fp32" else torch.float64
    t = [torch.tensor(q, dtype=dtype, device="cuda") for q in (x, v, m)]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    # the loss's weights: dL/d(first output), dL/d(second output)
    w = [torch.randn(case["n"], 3, generator=g, dtype=dtype, device="cuda") for _ in range(2)]
    return t, w


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("calc", "pass"):
        return {"case": case, "g6": _g6(), "f": _field(case, seed)}
    if kind == "blocks":
        _, m, x, v = _plummer(case["n"], seed)
        d = DeviceHermite4(precision=_prec(case))
        d.commit(m, x, v, EPS2, eta=_eta(case))
        return {"case": case, "drv": d, "t": 0.0}
    if kind == "ensemble":
        counts, m, x, v = _clusters(case, seed)
        return {"case": case, "ens": Ensemble(counts, m, x, v, eps2=EPS2_CLUSTERS,
                                              dt_param=DT_PARAM, precision=_prec(case))}
    (x, v, m), w = _tensors(case, seed)
    return {"case": case, "x": x.requires_grad_(), "v": v.requires_grad_(),
            "m": m.requires_grad_(), "w": w}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _kept(case, arrays):
    if case["prec"] == "mixed":
        return [a.astype(np.float32) for a in arrays]
    return list(arrays)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("calc", "pass"):
        g6, f = state["g6"], state["f"]
        g6.set_precision(_prec(case))
        g6.set_j_particles(f["addr"], f["ids"], f["tj"], 0.0, f["m"], f["k18"], f["j6"], f["a2"],
                           f["v"], f["x"])
        g6.set_ti(f["ti"])
        if kind == "calc":
            acc, jerk, pot, nn, _ = g6.calc(f["n"], f["id_i"], f["xi"], f["vi"], EPS2)
        else:
            g6.calc_self(f["n"], 0, f["n"], EPS2)
            acc, jerk, pot, nn = g6.fetch(f["n"])
        return _kept(case, (acc, jerk, pot)) + [nn]
    if kind == "blocks":
        state["t"] += 2.0 ** case["lg_dt"]
        state["drv"].evolve(state["t"])
        return _kept(case, state["drv"].state())
    if kind == "ensemble":
        ens = state["ens"]
        ens.start(1.0)
        ens.run(steps_per_graph=case["rounds"], use_graph=False, max_rounds=case["rounds"])
        x, v, t, steps = ens.state()
        return _kept(case, (x, v)) + [t, steps]
    x, v, m, w = state["x"], state["v"], state["m"], state["w"]
    if kind == "pair":
        a, b = pair_force(x, v, m, EPS2)
    else:
        a, b = hermite_integrate(x, v, m, 2.0 ** -9, case["steps"], EPS2, checkpoint_every=4)
    grads = torch.autograd.grad((a, b), (x, v, m), grad_outputs=w)
    return [a.detach(), b.detach(), *grads]


# ---------------------------------------------------------------------------
# what one pass cannot do without: 60 flop per pair interaction (the count of
# the GRAPE literature), 130 per pair of the adjoint
# ---------------------------------------------------------------------------
def _steps_per_time(case):
    """Particle steps per particle and unit time of these systems, roughly
    (measured on them: 3640 at N = 1024 and 4920 at 16384 with the small step
    parameter, 310 at 50021 with ph4's default)."""
    n = case["n"]
    return (3640.0 if case["prec"] == "fp64" else 205.0) * (n / 1024.0) ** 0.108


def work(case):
    kind = case["kind"]
    if kind == "calc":
        nj, ni = case["nj"], min(case["ni"], case["nj"])
        return {"bytes": 140 * nj + 128 * ni, "flops": 60.0 * ni * nj}
    if kind == "pass":
        n = case["n"]
        return {"bytes": 204 * n, "flops": 60.0 * n * n}
    if kind == "blocks":
        n = case["n"]
        psteps = _steps_per_time(case) * 2.0 ** case["lg_dt"] * n
        return {"bytes": 140 * n + 200 * psteps, "flops": 60.0 * psteps * n}
    if kind == "ensemble":
        # counts log-uniform in 16..2048: mean of n and of n^2
        span = math.log(2048 / 16)
        n1, n2 = (2048 - 16) / span, (2048 ** 2 - 16 ** 2) / (2 * span)
        passes = case["rounds"] + 1
        return {"bytes": 100.0 * case["nc"] * n1 * passes, "flops": 60.0 * case["nc"] * n2 * passes}
    n = case["n"]
    size = 4 if case["prec"] == "fp32" else 8
    if kind == "pair":
        return {"bytes": 26 * n * size, "flops": 190.0 * n * n}
    # forward, its recomputation in the backward pass, the adjoint; the
    # initial forces and their adjoint
    s = case["steps"]
    return {"bytes": 26 * n * size * s, "flops": (60.0 * (2 * s + 1) + 130.0 * (s + 1)) * n * n}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from plain torch
# ---------------------------------------------------------------------------
_BUDGET = 1 << 25  # pairs of one chunk


def _dev(*arrays):
    return [torch.as_tensor(np.asarray(a), dtype=torch.float64, device="cuda") for a in arrays]


def _pair_sums(xi, vi, xj, vj, m, eps2, own, collision=None):
    """acc, jerk, pot of rows (xi, vi) from (xj, vj, m); own[i] is the column
    of row i itself (skipped).  collision: the rows' masses; then also the
    largest inverse fourth power of a collision time."""
    acc, jerk, pot = torch.empty_like(xi), torch.empty_like(xi), torch.empty_like(xi[:, 0])
    cmax = 0.0
    step = max(1, _BUDGET // max(1, xj.shape[0]))
    for a in range(0, xi.shape[0], step):
        b = min(a + step, xi.shape[0])
        d = [xj[None, :, k] - xi[a:b, k, None] for k in range(3)]
        s = d[0] * d[0]
        s += d[1] * d[1]
        s += d[2] * d[2]
        r2 = s.clone() if collision is not None else None
        s += eps2
        y = s.rsqrt_()
        y[torch.arange(b - a, device=y.device), own[a:b]] = 0.0
        w = m[None] * y
        pot[a:b] = -w.sum(1)
        y2 = y * y
        w *= y2
        u = [vj[None, :, k] - vi[a:b, k, None] for k in range(3)]
        if collision is not None:
            v2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
            mm = collision[a:b, None] + m[None]
            q = torch.maximum((v2 * y2) ** 2, (mm * y2 * y2) ** 2 * r2)
            cmax = max(cmax, float(q.max()))
        c = d[0] * u[0]
        c += d[1] * u[1]
        c += d[2] * u[2]
        c *= -3.0
        c *= y2
        c *= w
        for k in range(3):
            acc[a:b, k] = (w * d[k]).sum(1)
            jerk[a:b, k] = (w * u[k]).sum(1) + (c * d[k]).sum(1)
    return (acc, jerk, pot) if collision is None else (acc, jerk, pot, cmax)


def _exact_field(case, seed):
    f = _field(case, seed)
    x, v, m, a2, j6, tj = _dev(f["x"], f["v"], f["m"], f["a2"], f["j6"], f["tj"])
    dt = (f["ti"] - tj)[:, None]
    xp = x + v * dt + a2 * dt ** 2 + j6 * dt ** 3
    vp = v + 2 * a2 * dt + 3 * j6 * dt ** 2
    if case["kind"] == "calc":
        xi, vi = _dev(f["xi"], f["vi"])
        own = torch.as_tensor(f["sel"], device="cuda")
    else:
        xi, vi, own = xp, vp, torch.arange(f["n"], device="cuda")
    return [*_pair_sums(xi, vi, xp, vp, m, EPS2, own), None]


def _pow2_below(x):
    """The largest power of two below or at x that ph4's first step takes."""
    f, e = np.frexp(x)
    return np.ldexp(0.5, e)


def _exact_blocks(case, seed):
    """ph4's block steps, from t = 0 to the first output."""
    _, m, x, v = _plummer(case["n"], seed)
    n, eta, t_end = case["n"], _eta(case), 2.0 ** case["lg_dt"]
    x, v, m = _dev(x, v, m)
    every = torch.arange(n, device="cuda")
    a, j, _ = _pair_sums(x, v, x, v, m, EPS2, every)
    # first steps: a power of two, not above 1/32 nor eight times the median
    first = (0.0625 * eta * ((a * a).sum(1) / (j * j).sum(1)).sqrt()).cpu().numpy()
    dt = np.minimum(_pow2_below(first), 0.03125)
    most = 8.0 * np.sort(dt)[n // 2]
    dt = np.minimum(dt, most)
    t = np.zeros(n)
    # the field particles' predictor terms stay zero until a particle's first step
    ja, jj = torch.zeros_like(a), torch.zeros_like(j)
    now = 0.0
    while now < t_end:
        nxt = t + dt
        now = float(nxt.min())
        blk = np.nonzero(nxt == now)[0]
        sel = torch.as_tensor(blk, device="cuda")
        h = torch.as_tensor(now - t, device="cuda")[:, None]
        xp = x + v * h + ja * (h ** 2 / 2) + jj * (h ** 3 / 6)
        vp = v + ja * h + jj * (h ** 2 / 2)
        h = h[sel]
        ao, jo = a[sel], j[sel]
        xi = x[sel] + h * (v[sel] + 0.5 * h * (ao + h * jo / 3))
        vi = v[sel] + h * (ao + 0.5 * h * jo)
        an, jn, _ = _pair_sums(xi, vi, xp, vp, m, EPS2, sel)
        al = -3 * (ao - an) - h * (2 * jo + jn)
        be = 2 * (ao - an) + h * (jo + jn)
        x[sel] = xi + (al / 12 + be / 20) * h ** 2
        v[sel] = vi + (al / 3 + be / 4) * h
        a[sel], j[sel], ja[sel], jj[sel] = an, jn, an, jn
        a2, j2 = (an * an).sum(1), ((h * jn) ** 2).sum(1)
        k2, l2 = ((2 * al) ** 2).sum(1), ((6 * be) ** 2).sum(1)
        new = (eta * h[:, 0] * (((a2 * k2).sqrt() + j2) / ((j2 * l2).sqrt() + k2)).sqrt())
        new, old = new.cpu().numpy(), dt[blk]
        for _ in range(64):
            old = np.where(np.fmod(now, old) != 0, old / 2, old)
        dt[blk] = np.where(new < old, old / 2,
                           np.where((new >= 2 * old) & (np.fmod(now, 2 * old) == 0), 2 * old, old))
        t[blk] = now
    h = torch.as_tensor(now - t, device="cuda")[:, None]
    return [x + h * (v + 0.5 * h * (a + h * j / 3)), v + h * (a + 0.5 * h * j)]


def _exact_ensemble(case, seed):
    """The shared-step Hermite scheme of each cluster, `rounds` steps."""
    counts, m, x, v = _clusters(case, seed)
    x, v, m = _dev(x, v, m)
    xs, vs, ts = [], [], []
    off = 0

    def step_of(cmax, t):
        want = DT_PARAM / math.sqrt(math.sqrt(cmax)) if cmax > 0 else 0.03125
        s = 0.03125
        while s > want or math.fmod(t, s):
            s /= 2
        return s

    for n in counts.tolist():
        xc, vc, mc = x[off:off + n], v[off:off + n], m[off:off + n]
        off += n
        own = torch.arange(n, device="cuda")
        a, j, _, cm = _pair_sums(xc, vc, xc, vc, mc, EPS2_CLUSTERS, own, collision=mc)
        t = 0.0
        h = step_of(cm, t)
        for _ in range(case["rounds"]):
            if t >= 1.0:
                break
            xp = xc + vc * h + a * (h * h / 2) + j * (h ** 3 / 6)
            vp = vc + a * h + j * (h * h / 2)
            a1, j1, _, cm = _pair_sums(xp, vp, xp, vp, mc, EPS2_CLUSTERS, own, collision=mc)
            v1 = vc + (a + a1) * (h / 2) + (j - j1) * (h * h / 12)
            xc = xc + (vc + v1) * (h / 2) + (a - a1) * (h * h / 12)
            vc, a, j = v1, a1, j1
            t += h
            h = step_of(cm, t)
        xs.append(xc)
        vs.append(vc)
        ts.append(t)
    return [torch.cat(xs), torch.cat(vs), torch.tensor(ts, dtype=torch.float64), None]


class _Pair(torch.autograd.Function):
    """acc, jerk in FP64 with gradients, row blocks differentiated one at a
    time (the whole pair matrix would not fit)."""

    @staticmethod
    def rows(x, v, m, a, b):
        d = x[None] - x[a:b, None]
        u = v[None] - v[a:b, None]
        k = torch.arange(b - a, device=x.device)
        y2 = 1.0 / ((d * d).sum(2) + EPS2)
        w = m[None] * y2 * y2.sqrt()
        w = w.index_put((k, k + a), torch.zeros((), dtype=w.dtype, device=w.device))
        c = -3.0 * (d * u).sum(2) * y2
        acc = (w[..., None] * d).sum(1)
        return acc, (w[..., None] * (u + c[..., None] * d)).sum(1)

    @staticmethod
    def blocks(n):
        step = max(1, _BUDGET // 4 // n)
        return [(a, min(a + step, n)) for a in range(0, n, step)]

    @staticmethod
    def forward(ctx, x, v, m):
        ctx.save_for_backward(x, v, m)
        out = [_Pair.rows(x, v, m, a, b) for a, b in _Pair.blocks(x.shape[0])]
        return torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out])

    @staticmethod
    def backward(ctx, ga, gj):
        with torch.enable_grad():
            q = [t.detach().requires_grad_() for t in ctx.saved_tensors]
            total = [torch.zeros_like(t) for t in q]
            for a, b in _Pair.blocks(q[0].shape[0]):
                out = _Pair.rows(*q, a, b)
                g = torch.autograd.grad(out, q, grad_outputs=(ga[a:b], gj[a:b]))
                for s, t in zip(total, g):
                    s += t
        return tuple(total)


def _exact_diff(case, seed):
    (x, v, m), w = _tensors(case, seed)
    x, v, m = (t.double().requires_grad_() for t in (x, v, m))
    a, b = _Pair.apply(x, v, m)
    if case["kind"] == "hermite":
        h = 2.0 ** -9
        xc, vc = x, v
        for _ in range(case["steps"]):
            xp = xc + vc * h + a * (h * h / 2) + b * (h ** 3 / 6)
            vp = vc + a * h + b * (h * h / 2)
            a1, b1 = _Pair.apply(xp, vp, m)
            v1 = vc + (a + a1) * (h / 2) + (b - b1) * (h * h / 12)
            xc = xc + (vc + v1) * (h / 2) + (a - a1) * (h * h / 12)
            vc, a, b = v1, a1, b1
        a, b = xc, vc
    g = torch.autograd.grad((a, b), (x, v, m), grad_outputs=[t.double() for t in w])
    return [a.detach(), b.detach(), *g]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("calc", "pass"):
        return _exact_field(case, seed)
    if kind == "blocks":
        return _exact_blocks(case, seed)
    if kind == "ensemble":
        return _exact_ensemble(case, seed)
    return _exact_diff(case, seed)
