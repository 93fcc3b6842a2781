"""Every unordered pair once, no rounding more: the root mean square error of
the pair-once sums over a system, against 80-bit sums, is not above that of
the pair by ordered pair kernels on the same system.

Both errors are means over thousands of independent roundings.  Over R rows
the ratio of two equal ones scatters by about 1 / sqrt(R) (three components
each, with the tails of close pairs): LIMIT leaves three times that for the
smallest R here, 3000."""
import numpy as np
import pytest

import oracle
from amuse_amd import ic
from conftest import par_oracle, print_case

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

LIMIT = 1.055
EPS2 = 1e-4


def system(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    _, x, v = ic.plummer_raw(n, rng)
    x, v = ic.to_nbody_units(x, v)
    return rng, rng.uniform(0.5, 1.5, n) / n, x, v


class Rms:
    """Errors of the rows of one or more systems, relative to the sums of the
    terms' sizes."""

    def __init__(self):
        self.sq, self.count = {}, {}

    def add(self, name, val, ref, size):
        d = (val - ref).reshape(len(size), -1) / size[:, None]
        self.sq[name] = self.sq.get(name, 0.0) + (d * d).sum()
        self.count[name] = self.count.get(name, 0) + d.size

    def over(self, other):
        out = {}
        for k in self.sq:
            assert self.count[k] == other.count[k]
            out[k] = float(np.sqrt(self.sq[k] / other.sq[k]))
        return out


def check(once, pairs, what):
    ratio = once.over(pairs)
    print(what, "error of pair-once over pair by pair:",
          {k: round(q, 3) for k, q in ratio.items()}, flush=True)
    assert all(q <= LIMIT for q in ratio.values()), (what, ratio)


def sums(ids, row, m, x, v, eps2):
    e = par_oracle(oracle.force_ld, ids[row], x[row], v[row], eps2, ids, m, x, v)
    return dict(zip(("acc", "jerk", "pot"), zip(e[:3], e[3:])))


@pytest.mark.parametrize("prec,sizes", [(0, (8192, 9001)), (0, (20000,)), (1, (13001, 19000))])
def test_full_pass(g6, prec, sizes):
    once, pairs = Rms(), Rms()
    for n in sizes:
        print_case(f"rounding of a full pass prec={prec} n={n}")
        rng, m, x, v = system(n, n)
        ids = np.arange(1, n + 1, dtype=np.int32)
        z = np.zeros((n, 3))
        g6.reset()
        g6.set_precision(prec)
        g6.set_j_particles(np.arange(n), ids, np.zeros(n), 0.0, m, z, z, z, v, x)
        g6.set_ti(0.0)
        row = np.sort(rng.choice(n, 4000, replace=False))
        ref = sums(ids, row, m, x, v, EPS2)
        for tiles, rms in (((0, 0), once), ((4, 1), pairs)):
            g6.set_tiles(*tiles)
            g6.calc_self(n, 0, n, EPS2)
            for (name, (e, s)), val in zip(ref.items(), g6.fetch(n)):
                rms.add(name, val[row], e, s)
    check(once, pairs, f"full pass prec={prec} n={sizes}")


@pytest.mark.parametrize("prec", [0, 1])
def test_clusters(prec):
    from amuse_amd.ensemble import Ensemble
    counts = np.array([129] * 8 + [200] * 6 + [300, 384, 500] * 3 + [777, 1024, 1500, 2048],
                      dtype=np.int32)
    total = int(counts.sum())
    _, m, x, v = system(total, 11)
    ids = np.arange(total, dtype=np.int32)
    off = np.concatenate([[0], np.cumsum(counts)])
    cl = [slice(a, b) for a, b in zip(off[:-1], off[1:])]
    ref = [sums(ids[s], np.arange(s.stop - s.start), m[s], x[s], v[s], EPS2) for s in cl]
    once, pairs = Rms(), Rms()
    for lanes, rms in ((1, once), (2, pairs)):
        print_case(f"rounding of clusters prec={prec} lanes={lanes}")
        ens = Ensemble(counts, m, x, v, eps2=EPS2, dt_param=0.03, precision=prec)
        tiles = ens.tiles()
        tiles[4:] = [lanes] * 4  # 1: the automatic shape, taken pair-once
        ens.set_tiles(tiles)
        out = dict(zip(("acc", "jerk", "pot"), ens.forces(prec)))
        ens.close()
        for s, r in zip(cl, ref):
            for name, (e, size) in r.items():
                rms.add(name, out[name][s], e, size)
    check(once, pairs, f"clusters prec={prec}")


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_differentiable_forward(dtype):
    from amuse_amd import diff
    L = diff._kernels()
    name = "f64" if dtype == torch.float64 else "f32"
    st = torch.cuda.current_stream().cuda_stream
    once, pairs = Rms(), Rms()
    for n in (5003, 6500, 8192, 12000):
        print_case(f"rounding of the forward sums {name} n={n}")
        rng, m, x, v = system(n, n)
        xx, vv, mm = (torch.tensor(q, dtype=dtype, device="cuda") for q in (x, v, m))
        m, x, v = (q.double().cpu().numpy() for q in (mm, xx, vv))
        row = np.sort(rng.choice(n, 2000, replace=False))
        eps2 = 1.0 / 8192  # the same in both precisions
        ref = sums(np.arange(n, dtype=np.int32), row, m, x, v, eps2)
        assert getattr(L, "g6a_forces_workspace_" + name)(n) > 0
        out = [torch.empty_like(xx) for _ in range(2)]
        assert getattr(L, "g6a_forces_" + name)(n, xx.data_ptr(), vv.data_ptr(), mm.data_ptr(), eps2,
                                                out[0].data_ptr(), out[1].data_ptr(), st) == 0
        for val, rms in ((diff.pair_force(xx, vv, mm, eps2), once), (out, pairs)):
            for k, q in zip(("acc", "jerk"), val):
                rms.add(k, q.double().cpu().numpy()[row], *ref[k])
    check(once, pairs, f"forward {name}")
