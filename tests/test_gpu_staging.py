"""Records of g6x_set_j_particles and g6_set_j_particle on their way to the
store: calls between the halves of a force call, a store loaded in slices, and
what the allocation-free call takes after a store was loaded in bulk."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT, print_case

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

N = 8000
EPS2 = 1e-4
G6X_ERR_NOMEM = -6


def records(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    x, v, a2, j6 = (rng.normal(0, 1, (n, 3)) for _ in range(4))
    return dict(ids=np.arange(1, n + 1, dtype=np.int32), tj=1.0 - rng.integers(0, 5, n) / 256.0,
                m=rng.uniform(0.1, 1, n), z=np.zeros((n, 3)), j6=j6, a2=a2, v=v, x=x)


def put(g6, r, sel):
    g6.set_j_particles(sel, r["ids"][sel], r["tj"][sel], 0.0, r["m"][sel], r["z"][sel],
                       r["j6"][sel], r["a2"][sel], r["v"][sel], r["x"][sel])


def put_one(g6, r, k):
    g6.set_j_particle(k, r["ids"][k], r["tj"][k], 0.0, r["m"][k], r["z"][k], r["j6"][k], r["a2"][k],
                      r["v"][k], r["x"][k])


def forces(g6, n):
    g6.set_ti(1.0)
    g6.calc_self(n, 0, n, EPS2)
    return g6.fetch(n)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1000, N])
def test_records_between_the_halves(g6, n, prec):
    """Records given between the two halves of a force call belong to the next
    call: two bulk calls, or a single record and a bulk call, leave the
    latched call's result as it is, and the next call has them."""
    old, new = records(n, 1), records(n, 2)
    every, rows = np.arange(n), np.arange(0, n, 7)
    first, second = every[: n // 2], every[n // 2:]
    g6.set_precision(prec)
    for way in ("bulk, bulk", "single, bulk"):
        print_case(f"between the halves n={n} prec={prec} {way}")
        out = []
        for between in (False, True):
            g6.reset()
            put(g6, old, every)
            g6.set_ti(1.0)
            g6.calc_firsthalf(n, old["ids"][rows], old["x"][rows], old["v"][rows], EPS2)
            if between:
                if way == "bulk, bulk":
                    put(g6, new, first)
                else:
                    put_one(g6, new, 0)
                    put(g6, new, first[1:])
                put(g6, new, second)
            out.append(g6.calc_lasthalf2(n, rows.size, EPS2))
        for a, b in zip(*out):
            assert np.array_equal(a, b)
        got = forces(g6, n)
        g6.reset()
        put(g6, new, every)
        for a, b in zip(got, forces(g6, n)):
            assert np.array_equal(a, b)
    g6.set_precision(0)


@pytest.mark.parametrize("step", [64, 100, 5000, 13000])
def test_store_loaded_in_slices(g6, step):
    """A store loaded in slices is the store loaded at once; the second time
    the library's staging buffers have their size."""
    n = 2 * N
    r = records(n, 3)
    put(g6, r, np.arange(n))
    ref = forces(g6, n)
    for _ in range(2):
        g6.reset()
        for a in range(0, n, step):
            put(g6, r, np.arange(a, min(n, a + step)))
        for a, b in zip(ref, forces(g6, n)):
            assert np.array_equal(a, b)


def noalloc(g6, n):
    out = [torch.zeros(s, dtype=t, device="cuda") for s, t in
           (((n, 3), torch.float64), ((n, 3), torch.float64), ((n,), torch.float64),
            ((n,), torch.int32))]
    torch.cuda.synchronize()
    rc = g6.lib.g6x_calc_self_noalloc(n, 0, n, EPS2, *(t.data_ptr() for t in out))
    g6.sync()
    return rc, [t.cpu().numpy() for t in out]


def child(kind):
    """In a process whose staging buffers have met nothing but bulk loads of N
    records: pending records of `kind`, then the allocation-free call."""
    from amuse_amd.g6 import G6
    g6 = G6(0)
    g6.open()
    old, new = records(N, 4), records(N, 5)
    every = np.arange(N)
    for _ in range(3):
        put(g6, old, every)
        assert g6.lib.g6_flush_jp_buffer(0) == 0
    g6.set_ti(1.0)
    put(g6, old, every)  # pending itself
    sel = {"none": every[:0], "single": every[:1], "few": every[10:73], "many": every[::-1][:5000],
           "all": every[::-1]}[kind]
    if kind == "single":
        put_one(g6, new, 0)
    elif kind != "none":
        put(g6, new, sel)
    print_case(f"allocation-free call after bulk loads, pending: {kind}")
    rc, got = noalloc(g6, N)
    assert rc == 0, (rc, g6.lib.g6x_last_error())
    g6.reset()
    both = {k: np.where(np.isin(every, sel).reshape((-1,) + (1,) * (a.ndim - 1)), new[k], a)
            for k, a in old.items()}
    put(g6, both, every)
    g6.set_ti(1.0)
    assert g6.lib.g6_flush_jp_buffer(0) == 0
    rc, ref = noalloc(g6, N)
    assert rc == 0
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
    # more than was ever flushed: refused, and taken after a flush
    more = records(2 * N, 6)
    put(g6, more, np.arange(2 * N)[::-1])
    assert noalloc(g6, 2 * N)[0] == G6X_ERR_NOMEM
    assert g6.lib.g6_flush_jp_buffer(0) == 0
    assert noalloc(g6, 2 * N)[0] == 0
    print("child ok", flush=True)


@pytest.mark.parametrize("kind", ["none", "single", "few", "many", "all"])
def test_noalloc_after_bulk_loads(kind):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), kind], cwd=ROOT, timeout=100,
                       capture_output=True, text=True)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and "child ok" in r.stdout


if __name__ == "__main__":
    child(sys.argv[1])
