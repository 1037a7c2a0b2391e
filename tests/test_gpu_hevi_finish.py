"""The line solves that store the tendency and the new stage state themselves
(the last of a fixed number of Newton iterations) against the oracle, bit for
bit: over the orders with one and two iterations and pivots on the diagonal;
and with steps so long that rows are exchanged in the blocks of some lines and
not of others, on meshes whose lines are all solved by one kernel and on one
whose groups of lines with exchanges are solved by a second kernel after the
first has stored the others (first and later stages, with and without the
copies of the first)."""
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


# (p, NeX, NeY, NeZ, dt): the last one has more groups of lines than a 256-CU chip has SIMDs
MIXED = [(6, 3, 1, 3, 0.2), (7, 3, 1, 4, 0.13), (7, 16, 9, 2, 0.13)]


@pytest.mark.parametrize("max_it", [1, 2])
@pytest.mark.parametrize("p,NeX,NeY,NeZ,dt", MIXED)
def test_fixed_iterations_mixed_pivots(p, NeX, NeY, NeZ, dt, max_it):
    print(f"HEVI fixed iterations, mixed pivots p={p} {NeX}x{NeY}x{NeZ} max_it={max_it}", flush=True)
    mesh = fedg.BoxMesh(p, NeX, NeY, NeZ, (0.0, 1.0e3 * NeX), (0.0, 1.0e3 * NeY), (0.0, 1.0e3 * NeZ))
    bs = cases.base_state(mesh, "constBVFreq")
    om = O.OracleMesh(mesh)
    Dx, Dy = om.calc_phyd_hgrad(bs)
    dm = fedg.DeviceMesh(mesh)
    n = mesh.Np * mesh.Ne
    rng = np.random.default_rng(p)
    q = [mesh.field() for _ in range(5)]
    for f, amp in zip(q, (1e-3, 0.3, 0.5, 1.0, 1.0)):
        f[:n] = amp * rng.standard_normal(n)
        om.exchange(f)
    st = fedg.HeviStepper(dm, bs, Dx, Dy, dt, scheme="IMEX_ARK324", max_it=max_it)
    st.set_state(q)
    st.run(1)
    g = st.get_state()
    st.close()
    r = [a.copy() for a in q]
    with om.pivot_lines() as lines:
        om.hevi_update(r, bs, Dx, Dy, dt, 1, scheme="IMEX_ARK324", max_it=max_it)
    assert 0 < lines.sum() < lines.size
    for name, a, b in zip(fedg.VARS, g, r):
        assert np.array_equal(a, b[:n], equal_nan=True), name
    dm.close()
