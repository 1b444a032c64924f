"""The skyline may be uploaded before the element state (the storage order is then the caller's), and
the state again later: read-backs come in the caller's element order, and a run's bits do not depend on
the order of storage."""
import ctypes as C

import numpy as np
import pytest

from openradioss_amd import engine as E
from openradioss_amd import lib as L
from openradioss_amd import model as M

pytestmark = pytest.mark.gpu


class Resident(E.GpuModel):
    """A model whose handle is filled call by call."""

    def __init__(self, m, precision):
        self.model, self._lib, self.prec = m, L.load(), E.PRECISIONS[precision]
        h = C.c_void_p()
        L.check(self._lib.or_model_create(C.byref(h), 0, m.nn, m.ne_hex, m.ne_q4, m.q4.prop.npt,
                                          self.prec))
        self._h = h


@pytest.mark.parametrize("precision", ["fp64", "split"])
def test_skyline_before_state(precision, gpu_lib):
    m = M.block_with_plate(n=7, plate=17, seed=3)  # more than a tile of each family, Morton order differs
    print(f"case: {m.ne_hex} hexes, {m.ne_q4} shells, skyline first, {precision}", flush=True)
    ref = E.GpuModel(m, precision=precision)
    rng = np.random.default_rng(8)

    def c(a):
        return a.ctypes.data_as(C.c_void_p)

    def drawn(st):
        return {k: rng.standard_normal(a.shape).astype(np.float32).astype(np.float64) for k, a in st.items()}
    hs, qs = m.hexp.initial_state(), m.q4.initial_state()
    marked = drawn(hs), drawn(qs)
    g = Resident(m, precision)
    lib = g._lib
    L.check(lib.or_model_set_hex_params(g._h, C.byref(E.hex_params(m))))
    L.check(lib.or_model_set_q4_params(g._h, C.byref(E.q4_params(m))))
    arrays = [np.ascontiguousarray(a, np.float64) for a in (m.x, m.v, m.vr, m.ms, m.inr)]
    code, vimp = np.ascontiguousarray(m.code, np.int32), np.ascontiguousarray(m.vimp, np.float64)
    L.check(lib.or_model_upload_nodes(g._h, *[a.ctypes.data_as(C.c_void_p) for a in arrays],
                                      code.ctypes.data_as(C.c_void_p), vimp.ctypes.data_as(C.c_void_p)))
    adsky, iads, iadc = (np.ascontiguousarray(a, np.int64) for a in (m.adsky, m.hexp.iads, m.q4.iadc))
    L.check(lib.or_model_upload_skyline(g._h, *[a.ctypes.data_as(C.c_void_p) for a in (adsky, iads, iadc)]))
    hconn, qconn = np.ascontiguousarray(m.hexp.conn, np.int32), np.ascontiguousarray(m.q4.conn, np.int32)
    vol0, thke = np.ascontiguousarray(m.hexp.vol0, np.float64), np.ascontiguousarray(m.q4.thke, np.float64)

    def upload(h, q):
        a = {k: np.ascontiguousarray(v, np.float64) for k, v in h.items()}
        b = {k: np.ascontiguousarray(v, np.float64) for k, v in q.items()}
        L.check(lib.or_model_upload_hex(g._h, c(hconn), c(a["sig"]), c(a["eint"]), c(a["rho"]), c(vol0), c(a["pla"]),
                                        c(a["epsd"]), c(a["offg"]), c(a["qvis"])))
        L.check(lib.or_model_upload_q4(g._h, c(qconn), c(thke), *[c(b[k]) for k in (
            "offg", "thk", "forc", "mom", "gstr", "hourg", "eint", "epsd", "sig", "pla", "epsd_ip")]))

    upload(*marked)
    for got, want in ((g.hex_state(), marked[0]), (g.q4_state(), marked[1])):
        for k, a in got.items():
            if k != "epsd_ip":
                assert np.array_equal(a, want[k]), k
    upload(hs, qs)
    g.run(25)
    ref.run(25)
    for a, b in zip(g.nodes6(), ref.nodes6()):
        assert np.array_equal(a, b)
    for got, want in ((g.hex_state(), ref.hex_state()), (g.q4_state(), ref.q4_state())):
        assert all(np.array_equal(got[k], want[k]) for k in got)
    g.close()
    ref.close()
