"""The HEVI line solves over the orders, column heights and line counts at
their edges (segments with idle lanes, a last group of lines that is not full,
one level), with blocks whose pivots stay on the diagonal (small impl_fac),
leave it on some lines, and leave it everywhere (large impl_fac): one Newton
iteration and Newton to a tolerance against the oracle, bit for bit."""
import numpy as np
import pytest

import fedg
import fedg_oracle as O
from fedg import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def portable_pow():
    with O.pow_mode(O.POW_PORTABLE):
        yield


SHAPES = [(1, 3, 1, 5), (2, 3, 1, 4), (3, 2, 3, 1), (3, 5, 1, 3), (4, 3, 1, 3), (5, 1, 2, 2), (6, 3, 1, 2), (7, 1, 1, 4),
          (7, 3, 1, 1)]


@pytest.mark.parametrize("impl_fac", [0.01, 0.2, 6.0])
@pytest.mark.parametrize("p,NeX,NeY,NeZ", SHAPES)
def test_line_solves_bitwise(p, NeX, NeY, NeZ, impl_fac):
    print(f"line solves p={p} {NeX}x{NeY}x{NeZ} impl_fac={impl_fac}", flush=True)
    m = fedg.BoxMesh(p, NeX, NeY, NeZ, (0.0, 1.0e3 * NeX), (0.0, 1.0e3 * NeY), (0.0, 1.0e3 * NeZ))
    bs = cases.base_state(m, "constBVFreq")
    om = O.OracleMesh(m)
    dm = fedg.DeviceMesh(m)
    n = m.Np * m.Ne

    def state(seed):
        rng = np.random.default_rng(seed)
        q = [m.field() for _ in range(5)]
        for f, amp in zip(q, (1e-3, 0.3, 0.5, 5.0, 1.0)):
            f[:n] = amp * rng.standard_normal(n)
            m.exchange(f)
        return q

    q, q0 = state(p), state(p + 100)
    dev = lambda a: fedg.DevField(a.size, a)  # noqa: E731
    d, d0 = [dev(a) for a in q], [dev(a) for a in q0]
    aux = {k: dev(getattr(bs, k)) for k in ("DENS_hyd", "PRES_hyd", "Rtot", "CVtot", "CPtot")}
    for max_it, rtol in ((None, 0.0), (3, 1e-14)):
        ref, _, _ = om.hevi_cal_vi(q, q0, bs, impl_fac, 1.0, **({} if max_it is None else dict(max_it=max_it, rtol=rtol)))
        out = [dev(m.field()) for _ in range(5)]
        fedg.hevi_cal_vi(dm, out, d[0], d[3], d[4], d[2], d[1], aux["DENS_hyd"], aux["PRES_hyd"], d0[0], d0[3], d0[4],
                         d0[2], d0[1], aux["Rtot"], aux["CVtot"], aux["CPtot"], impl_fac, 1.0, max_it=max_it, rtol=rtol)
        g = [a.download() for a in out]
        for name, a, b in zip(fedg.VARS, [g[0], g[4], g[3], g[1], g[2]], ref):
            assert np.array_equal(a[:n], b[:n], equal_nan=True), f"{name} (max_it={max_it})"
    dm.close()
