"""The autotuners: they return variants that are built (no name for the kernel of another variant, which
would only give up the launch that default variants share), advance 4 x cycles a family, and keep results."""
import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu

BUILT = {("fp64", 0): {0, 2}, ("fp64", 1): {0, 2}, ("split", 0): {0, 2, 3}, ("split", 1): {0, 1, 2, 3}}


def models():
    return {"both": M.block_with_plate(n=9, plate=18, seed=3),
            "hexes": M.hex_model_to_model(M.cantilever_bar(5, 5, 12, v0=1.0e4)),
            "shells": M.square_tube(width=6.0, length=20.0)}


def equal(a, b):
    for x, y in zip(a.nodes6(), b.nodes6()):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("precision", ["fp64", "split"])
@pytest.mark.parametrize("name", ["both", "hexes", "shells"])
@pytest.mark.parametrize("cycles", [1, 3])
def test_model(name, precision, cycles, gpu_lib):
    print(f"case: autotune({cycles}), {name}, {precision}", flush=True)
    m = models()[name]
    g, ref = E.GpuModel(m, precision=precision), E.GpuModel(m, precision=precision)
    g.set_variant("q4", 3)  # the search starts from the default variants whatever was set
    families = (m.ne_hex > 0) + (m.ne_q4 > 0)
    for k in range(1, 4):
        chosen = g.autotune(cycles)
        assert all(chosen[f] in BUILT[precision, f] for f in (0, 1))
        assert g.time_state().ncycle == 4 * cycles * families * k
    g.run(5)
    ref.run(g.time_state().ncycle)
    equal(g, ref)
    g.close()
    ref.close()


@pytest.mark.parametrize("forms", [("fp64", "fp64", "fp64"), ("split", "fp64", "split"), ("split", "split", "split")])
def test_batch(forms, gpu_lib):
    print(f"case: batch autotune, {forms}", flush=True)
    ms = list(models().values())
    b = E.GpuBatch()
    gs = [E.GpuModel(m, precision=p) for m, p in zip(ms, forms)]
    for g in gs:
        b.add(g, 1.0)
    chosen = b.autotune(2)
    assert all(chosen[2 * c + f] in BUILT[p, f] for c, p in enumerate(("fp64", "split")) for f in (0, 1))
    families = sum(any(getattr(m, n) > 0 and p == q for m, q in zip(ms, forms))
                   for p in ("fp64", "split") for n in ("ne_hex", "ne_q4"))
    assert gs[0].time_state().ncycle == 8 * families
    b.run(4)
    for g, m, p in zip(gs, ms, forms):
        ref = E.GpuModel(m, precision=p)
        ref.run(8 * families + 4)
        equal(g, ref)
        ref.close()
    b.close()
    for g in gs:
        g.close()
