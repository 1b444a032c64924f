"""Drop-ins, uploads, runs and read-backs from several threads at once: they share the kept page-locked buffers
and workspaces, and each gets what it gets alone.  The allocation-free group call is not among them
(its callers serialise it)."""
import threading

import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import lib as L
from openradioss_amd import model as M
from test_zz_no_alloc import group
from test_zz_no_alloc import run as run_group

pytestmark = pytest.mark.gpu


def hexes():
    case = group(8, 4, 4, 1)
    return lambda: [(r[0], *r[2].values(), r[3]) for r in [run_group(*case, nft=0, nel=128, static=False)]][0]


def nodal(nn):
    rng = np.random.default_rng(nn)
    adsky = (np.concatenate([[0], np.cumsum(rng.integers(0, 9, nn))]) + 1).astype(np.int64)
    fsky = rng.standard_normal((int(adsky[-1]) - 1, 8))
    ms = rng.uniform(1.0, 2.0, nn)
    x, v, d = (rng.standard_normal((nn, 3)) for _ in range(3))

    def call():
        ts = L.OrTimeState()
        ts.dt2, ts.dt2old = 1.0e-7, 1.0e-7
        out = [x.copy(), v.copy(), d.copy()]
        E.nodal_update(adsky, fsky, ms, *out, ts, 1.05e-7)
        return out
    return call


def resident(m, precision):
    def call():
        with E.GpuModel(m, precision=precision) as g:
            g.run(7)
            out = list(g.nodes6())
            out += list(g.hex_state().values()) if m.ne_hex else []
            return out + (list(g.q4_state().values()) if m.ne_q4 else [])
    return call


def test_calls_from_several_threads(gpu_lib):
    print("case: 7 threads, 6 rounds of drop-ins, runs and read-backs", flush=True)
    jobs = [hexes(), hexes(), nodal(300), nodal(30011), nodal(30011), resident(M.square_tube(), "fp64"),
            resident(M.block_with_plate(n=12, plate=40, seed=2), "split")]
    want = [j() for j in jobs]
    bad = []

    def work(k):
        try:
            for _ in range(6):
                if not all(np.array_equal(a, b) for a, b in zip(jobs[k](), want[k], strict=True)):
                    bad.append((k, "other values"))
        except Exception as e:  # noqa: BLE001  (reported by the test's thread)
            bad.append((k, repr(e)))

    team = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad, bad
