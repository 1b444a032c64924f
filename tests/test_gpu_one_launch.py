"""The element tiles of all families and forms in one launch (k_elements, k_node_update_both): the
same bits as one launch for each family.  A family set to the ILP-first variant keeps its own
launch, which gives the reference side."""
import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu


def models():
    # hex elements, shells: below, at and above a tile (256), none of a family
    return [M.block_with_plate(n=4, plate=8, seed=11), M.block_with_plate(n=7, plate=17, seed=3),
            M.hex_model_to_model(M.cantilever_bar(8, 8, 4, v0=1.0e4)), M.square_tube(width=5.0, length=13.0)]


def state(g):
    out = list(g.nodes6())
    out += list(g.hex_state().values()) if g.model.ne_hex else []
    return out + (list(g.q4_state().values()) if g.model.ne_q4 else [])


def same(a, b):
    assert (a.time_state().tt, a.time_state().ncycle) == (b.time_state().tt, b.time_state().ncycle)
    for x, y in zip(state(a), state(b)):
        assert np.array_equal(x, y)


def separate(m, precision):
    g = E.GpuModel(m, precision=precision)
    g.set_variant("hex", 2)
    g.set_variant("q4", 2)
    return g


@pytest.mark.parametrize("precision", ["fp64", "split"])
@pytest.mark.parametrize("k", [0, 1])
def test_model(k, precision, gpu_lib):
    print(f"case: mixed model {k}, {precision}, 40 cycles", flush=True)
    a, b = E.GpuModel(models()[k], precision=precision), separate(models()[k], precision)
    a.run(40)
    b.run(40)
    same(a, b)


@pytest.mark.parametrize("forms", [("fp64",) * 4, ("fp64", "split", "split", "fp64"), ("split", "fp64", "fp64", "split")])
def test_batch(forms, gpu_lib):
    print(f"case: batch of 4 models, {forms}, 40 cycles", flush=True)
    ms = models()
    b = E.GpuBatch()
    gs = [E.GpuModel(m, precision=p) for m, p in zip(ms, forms)]
    for k, g in enumerate(gs):
        b.add(g, 1.0 if k != 1 else 2.0e-6)  # one member stops on the way
    b.run(25)
    b.active()                               # a stopped member leaves the tile lists
    b.run(15)
    for k, (m, p, g) in enumerate(zip(ms, forms, gs)):
        ref = separate(m, p)
        ref.run(g.time_state().ncycle if k == 1 else 40)
        same(g, ref)


@pytest.mark.parametrize("precision", ["fp64", "split"])
@pytest.mark.parametrize("k", [0, 1])
def test_time_history(k, precision, gpu_lib):
    """The instantiations that keep EHOUR (hourglass energy of each tile) and an output cycle's candidates."""
    print(f"case: mixed model {k} with a time history, {precision}, 30 cycles and 3 records", flush=True)
    m = models()[k]
    a, b = E.GpuModel(m, precision=precision), separate(m, precision)
    for g in (a, b):
        g.th_setup(range(0, m.nn, 7), range(0, m.ne_hex, 5), range(0, m.ne_q4, 3))
    for _ in range(3):
        a.run(9)
        b.run(9)
        ra, rb = a.run_th(), b.run_th()
        assert ra["ehour"] != 0.0
        assert all(np.array_equal(ra[n], rb[n]) for n in ra)
        assert a.ehour() == b.ehour() == ra["ehour"]
    same(a, b)
