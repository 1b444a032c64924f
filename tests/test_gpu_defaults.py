"""State arrays that an upload leaves out get their defaults: every value of arrays longer than one
launch of the fill (16,384 blocks, 4.2 million values), in place of what was there."""
import ctypes as C

import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import lib as L
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "split"])
def test_absent_state_is_filled(precision, gpu_lib):
    m = M.square_tube(width=60.0, length=377.0, prop=M.ShellProp(1.5, npt=10))
    print(f"case: {m.ne_q4} shells of 10 points, {50 * m.ne_q4} stresses, {precision}", flush=True)
    assert 50 * m.ne_q4 > 16384 * 256 and (50 * m.ne_q4) % 256
    rng = np.random.default_rng(4)
    st = {k: rng.standard_normal(a.shape) for k, a in m.q4.initial_state().items()}
    with E.GpuModel(m, precision=precision, q4_state=st) as g:
        def p(a, t):
            return np.ascontiguousarray(a, t).ctypes.data_as(C.c_void_p)
        conn, thke = np.ascontiguousarray(m.q4.conn, np.int32), np.ascontiguousarray(m.q4.thke, np.float64)
        L.check(g._lib.or_model_upload_q4(g._h, p(conn, np.int32), p(thke, np.float64), *[None] * 11))
        out = g.q4_state()
    want = dict(offg=1.0, thk=thke.astype(np.float32 if precision == "split" else np.float64))
    for k, a in out.items():
        assert np.array_equal(a, np.broadcast_to(want.get(k, 0.0), a.shape)), k
