"""Transfers through page-locked chunks (2 MB): arrays longer than a chunk, ends inside one, both
storage types, and the nodal drop-in's workspace, against what was uploaded or numpy's sums."""
import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import lib as L
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu


def randomised(state, rng, precision):
    out = {k: rng.standard_normal(a.shape) for k, a in state.items()}
    if precision == "split":  # values the FP32 state holds exactly
        out = {k: a.astype(np.float32).astype(np.float64) for k, a in out.items()}
    return out


@pytest.mark.parametrize("precision", ["fp64", "split"])
@pytest.mark.parametrize("name", ["tube", "bar", "tiny"])
def test_read_back_equals_upload(name, precision, gpu_lib):
    print(f"case: read-back, {name}, {precision}", flush=True)
    m = {"tube": lambda: M.square_tube(width=60.0, length=381.0),          # 3 * nn and 25 * ne beyond a chunk
         "bar": lambda: M.hex_model_to_model(M.cantilever_bar(29, 31, 61)),  # 6 * ne beyond a chunk
         "tiny": lambda: M.block_with_plate(n=2, plate=3, seed=1)}[name]()
    rng = np.random.default_rng(9)
    nodes = [rng.standard_normal((m.nn, 3)) for _ in range(4)]
    nodes[0] = m.x + 1e-3 * nodes[0]
    hs = randomised(m.hexp.initial_state(), rng, precision) if m.ne_hex else None
    qs = randomised(m.q4.initial_state(), rng, precision) if m.ne_q4 else None
    g = E.GpuModel(m, precision=precision, hex_state=hs, q4_state=qs, nodes=tuple(nodes))
    for _ in range(2):  # fresh and kept buffers
        x, v, vr, d = g.nodes6()
        assert np.array_equal(x, nodes[0]) and np.array_equal(v, nodes[1]) and np.array_equal(d, nodes[3])
        assert np.array_equal(vr, nodes[2] if m.ne_q4 else np.zeros_like(vr))
        if m.ne_hex:
            out = g.hex_state()
            assert all(np.array_equal(out[k], hs[k]) for k in out)
        if m.ne_q4:
            out = g.q4_state()
            for k in out:  # without the strain-rate filter LBUF EPSD is GBUF EPSD at every point
                want = np.broadcast_to(qs["epsd"], out[k].shape) if k == "epsd_ip" else qs[k]
                assert np.array_equal(out[k], want), k
    g.close()


@pytest.mark.parametrize("nn", [1, 300, 30011])
def test_nodal_drop_in(nn, gpu_lib):
    print(f"case: nodal drop-in, {nn} nodes", flush=True)
    rng = np.random.default_rng(nn)
    deg = rng.integers(0, 9, nn)
    adsky = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    fsky = rng.standard_normal((int(adsky[-1]), 8))
    ms = rng.uniform(1.0, 2.0, nn)
    x, v, d = (rng.standard_normal((nn, 3)) for _ in range(3))
    a, sn = np.zeros((nn, 3)), np.zeros(nn)
    for k in range(8):  # row after row from zero, as ASSPAR4
        on = deg > k
        a[on] += fsky[adsky[:-1][on] + k, :3]
        sn[on] += fsky[adsky[:-1][on] + k, 6]
    ts = L.OrTimeState()
    ts.dt2, ts.dt2old = 1.0e-7, 1.0e-7
    gx, gv, gd, stifn = x.copy(), v.copy(), d.copy(), np.empty(nn)
    E.nodal_update(adsky + 1, fsky, ms, gx, gv, gd, ts, 1.05e-7, stifn=stifn)
    dt12 = 0.5 * (1.0e-7 + ts.dt2)
    vel = v + dt12 * (a * (1.0 / ms)[:, None])
    step = ts.dt2 * vel
    assert np.array_equal(gv, vel) and np.array_equal(gx, x + step) and np.array_equal(gd, d + step)
    assert np.array_equal(stifn, sn)
