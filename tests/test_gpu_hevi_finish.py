"""The line solves that store the tendency and the new stage state themselves
(the last of a fixed number of Newton iterations) against the oracle, bit for
bit, over the orders, with one and two iterations, and with pivots off the
diagonal on some lines (a long step)."""
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


@pytest.mark.parametrize("max_it", [1, 2])
@pytest.mark.parametrize("p", range(1, 8))
def test_fixed_iterations(p, max_it):
    print(f"HEVI fixed iterations p={p} max_it={max_it}", flush=True)
    case = cases.scaled_case(cases.config4(), 3, 1, 3, porder=p)
    mesh, bs, q = cases.build(case)
    om = O.OracleMesh(mesh)
    Dx, Dy = om.calc_phyd_hgrad(bs)
    dm = fedg.DeviceMesh(mesh)
    n = mesh.Np * mesh.Ne
    rng = np.random.default_rng(p)
    for f, amp in zip(q, (1e-3, 0.1, 0.2, 1.0, 1.0)):
        f[:n] += amp * rng.standard_normal(n)
        om.exchange(f)
    for dt in (0.1 * case.dt, case.dt):
        st = fedg.HeviStepper(dm, bs, Dx, Dy, dt, scheme=case.scheme, max_it=max_it)
        st.set_state(q)
        st.run(1)
        g = st.get_state()
        st.close()
        r = [a.copy() for a in q]
        om.hevi_update(r, bs, Dx, Dy, dt, 1, scheme=case.scheme, max_it=max_it)
        for name, a, b in zip(fedg.VARS, g, r):
            assert np.array_equal(a, b[:n], equal_nan=True), f"{name} dt={dt}"
    dm.close()
