"""The node update's form for launches of 8,192 blocks and more (2.1 million nodes; loads at their
uses) gives the bits of the one below (loads first): members of a large batch against the same models
alone, and an output cycle of one large model against the oracle."""
import numpy as np
import pytest

import oracle as O
from openradioss_amd import engine as E
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu

BLOCKS = 8192


@pytest.mark.parametrize("precision", ["fp64", "split"])
def test_large_batch_equals_single_models(precision, gpu_lib):
    # hexes with a tied plate; shells with BCs and imposed velocities; hexes alone with a clamped end
    kinds = [M.block_with_plate(n=40, plate=150, seed=5), M.square_tube(),
             M.hex_model_to_model(M.cantilever_bar(20, 21, 80, v0=1.0e4))]
    copies = 13
    nblocks = copies * sum((m.nn + 255) // 256 for m in kinds)
    assert nblocks >= BLOCKS > max(m.nn for m in kinds) // 256
    print(f"case: batch of {3 * copies} models, {nblocks} node blocks, {precision}, 12 cycles", flush=True)
    ref = []
    for m in kinds:
        with E.GpuModel(m, precision=precision) as g:
            g.run(12)
            ref.append(g.nodes6() + (g.time_state().tt,))
    b = E.GpuBatch()
    gs = [E.GpuModel(m, precision=precision) for _ in range(copies) for m in kinds]
    for g in gs:
        b.add(g, 1.0)
    b.run(12)
    for k in (0, 1, 2, 3 * copies - 3, 3 * copies - 2, 3 * copies - 1):
        for x, y in zip(gs[k].nodes6(), ref[k % 3]):
            assert np.array_equal(x, y)
        assert gs[k].time_state().tt == ref[k % 3][4]
    b.close()
    for g in gs:
        g.close()


def test_output_cycle_of_a_large_model(gpu_lib):
    m = M.block_with_plate(n=121, plate=640, seed=5)
    assert (m.nn + 255) // 256 >= BLOCKS
    print(f"case: {m.nn} nodes, 3 cycles and an output cycle against the oracle", flush=True)
    o = O.ModelOracle(m, nthreads=16, math="cr")
    o.cycle(3)
    want = o.cycle_ecrit()
    with E.GpuModel(m) as g:
        g.run(3)
        got = g.run_ecrit()
        x, v, vr, d = g.nodes6()
    assert np.array_equal(d, o.d) and np.array_equal(v, o.v)
    assert (got["itypts"], got["nelts"]) == (want["itypts"], want["nelts"])
    for k in ("enint", "encin", "enrot", "wfext"):
        # sums over n ~ 2e6 terms of one sign: both sides' rounding errors stay below n * 2^-53 = 2.4e-10
        assert abs(got[k] - want[k]) <= 2.5e-10 * abs(want[k]), k
