"""The two layouts of the element kernel on either side of the mesh size at
which one takes over from the other (p = 4, 5 and 7 on 256 CUs; the sizes beyond
it fill no whole group of eight workgroups), flat and over terrain, against the
oracle bit for bit: the drop-in HEVE and HEVI right-hand sides and the volume
part, and fused steps without and with physics tendencies."""
import dataclasses

import numpy as np
import pytest

import fedg
import fedg_oracle as O
from fedg import cases, constants

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def portable_pow():
    with O.pow_mode(O.POW_PORTABLE):
        yield


# (p, NeX, NeY, NeZ): the largest mesh of one layout and the smallest odd one of the other
SIZES = [(4, 131, 4, 2), (4, 21, 10, 5), (5, 101, 3, 1), (5, 61, 5, 1), (7, 8, 8, 4), (7, 29, 3, 3)]


@pytest.mark.parametrize("terrain", [False, True], ids=["flat", "terrain"])
@pytest.mark.parametrize("p,NeX,NeY,NeZ", SIZES)
def test_layouts_bitwise(p, NeX, NeY, NeZ, terrain):
    print(f"element layouts p={p} {NeX}x{NeY}x{NeZ} terrain={terrain}", flush=True)
    mesh = fedg.BoxMesh(p, NeX, NeY, NeZ, (0.0, 1.0e3 * NeX), (0.0, 1.0e3 * NeY), (0.0, 8.0e2 * NeZ))
    if terrain:
        mesh.set_topography(lambda x, y: 100.0 / (1.0 + ((x - 500.0 * NeX) / 2.0e3) ** 2))
    c = constants.SCALE
    nA, n = mesh.Np * mesh.NeA, mesh.Np * mesh.Ne
    bs = cases.base_state(mesh, "constBVFreq")
    bs = dataclasses.replace(bs, Rtot=np.full(nA, c.Rdry), CVtot=np.full(nA, c.CVdry), CPtot=np.full(nA, c.CPdry))
    rng = np.random.default_rng(p)
    bs.CORIOLIS[:] = 1.0e-4 * (1.0 + 0.3 * rng.standard_normal(bs.CORIOLIS.size))
    om = O.OracleMesh(mesh)
    dm = fedg.DeviceMesh(mesh)
    Dx, Dy = om.calc_phyd_hgrad(bs)
    q = [mesh.field() for _ in range(5)]
    for f, amp in zip(q, (1e-3, 0.3, 0.5, 5.0, 1.0)):
        f[:n] = amp * rng.standard_normal(n)
        om.exchange(f)
    om.apply_bc(q)
    _, DP = om.drhot2pres(q[1], bs)
    dev = lambda a: fedg.DevField(a.size, a)  # noqa: E731
    d = [dev(a) for a in q]
    base = [dev(DP)] + [dev(getattr(bs, k)) for k in ("DENS_hyd", "PRES_hyd", "PRES_hyd_ref", "THERM_hyd", "CORIOLIS",
                                                       "Rtot", "CVtot", "CPtot")] + [dev(Dx), dev(Dy)]
    for fn, ref in ((fedg.heve_cal_tend, om.cal_tend), (fedg.hevi_cal_tend, om.hevi_cal_tend),
                    (fedg.heve_cal_tend_cco, om.cal_tend_cco)):
        out = [dev(mesh.field()) for _ in range(5)]
        fn(dm, out, d[0], d[3], d[4], d[2], d[1], *base)
        g = [a.download() for a in out]
        for name, a, b in zip(("DENS", "MOMX", "MOMY", "MOMZ", "RHOT"), g, ref(q, DP, bs, Dx, Dy)):
            assert np.array_equal(a[:n], b[:n]), f"{fn.__name__} {name}_dt"
    tp = []  # DENS, RHOT, MOMZ, MOMX, MOMY, RHOH
    for amp in (1e-7, 1e-4, 1e-5, 1e-5, 1e-5, 1e-1):
        f = mesh.field()
        f[:n] = amp * rng.standard_normal(n)
        om.exchange(f)
        tp.append(f)
    dtp = [dev(tp[k]) for k in (0, 3, 4, 2, 1, 5)]
    st = fedg.HeveStepper(dm, bs, Dx, Dy, 0.01)
    for phys in (False, True):
        st.set_phys_tend(*(dtp if phys else ()))
        st.set_state(q)
        st.run(1)
        g = st.get_state()
        om.set_phys_tend(tp if phys else None)
        r = [a.copy() for a in q]
        om.heve_update(r, bs, Dx, Dy, 0.01, 1)
        om.set_phys_tend(None)
        for name, a, b in zip(fedg.VARS, g, r):
            assert np.array_equal(a, b[:n]), f"{name} phys={phys}"
    st.close()
    dm.close()


@pytest.mark.parametrize("p", [6, 7])
def test_base_state_with_one_other_node(p):
    """A base state that differs from a horizontally homogeneous one by one unit in the last place of one
    field's last node: the stepper reads that node's own value."""
    mesh = fedg.BoxMesh(p, 3, 3, 2, (0.0, 3.0e3), (0.0, 3.0e3), (0.0, 1.6e3))
    c = constants.SCALE
    nA, n = mesh.Np * mesh.NeA, mesh.Np * mesh.Ne
    bs0 = cases.base_state(mesh, "constT")
    bs0 = dataclasses.replace(bs0, Rtot=np.full(nA, c.Rdry), CVtot=np.full(nA, c.CVdry), CPtot=np.full(nA, c.CPdry))
    om = O.OracleMesh(mesh)
    dm = fedg.DeviceMesh(mesh)
    rng = np.random.default_rng(p)
    q = [mesh.field() for _ in range(5)]
    for f, amp in zip(q, (1e-3, 0.3, 0.5, 5.0, 1.0)):
        f[:n] = amp * rng.standard_normal(n)
        om.exchange(f)
    for field in ("DENS_hyd", "PRES_hyd", "THERM_hyd", "DPhydDx", "DPhydDy", None):
        print(f"base state with one other node, p={p} {field}", flush=True)
        bs = bs0
        Dx, Dy = om.calc_phyd_hgrad(bs)
        if field in ("DPhydDx", "DPhydDy"):
            f = Dx if field == "DPhydDx" else Dy
            f[n - 1] += 1.0e-3
        elif field:
            f = getattr(bs, field).copy()
            f[n - 1] = np.nextafter(f[n - 1], np.inf)
            om.exchange(f)
            bs = dataclasses.replace(bs, **{field: f})
        st = fedg.HeveStepper(dm, bs, Dx, Dy, 0.01)
        st.set_state(q)
        st.run(1)
        g = st.get_state()
        st.close()
        r = [a.copy() for a in q]
        om.heve_update(r, bs, Dx, Dy, 0.01, 1)
        for name, a, b in zip(fedg.VARS, g, r):
            assert np.array_equal(a, b[:n]), f"{name} {field}"
    dm.close()
