"""The element kernel on boxes whose element count fills no last workgroup (18
elements) at every order, against the oracle bit for bit: the drop-in HEVE and
HEVI right-hand sides and the volume part with the flat box's constants and
with loaded metric arrays, and the fused stages with the base state from
per-level tables, from fields that vary in the horizontal, and with the modal
filter in the last stage (two schemes: with and without stages before it)."""
import dataclasses

import numpy as np
import pytest

import fedg
import fedg_oracle as O
from fedg import cases, constants
from fedg.mesh import BND_NOSLIP, BND_NONE, BND_SLIP

pytestmark = pytest.mark.gpu

WALLS = (BND_NONE, BND_SLIP, BND_NONE, BND_SLIP, BND_NOSLIP, BND_SLIP)  # y-, x+, y+, x-, z-, z+


@pytest.fixture(autouse=True)
def portable_pow():
    with O.pow_mode(O.POW_PORTABLE):
        yield


def build(p, box_shape):
    mesh = fedg.BoxMesh(p, 3, 2, 3, (0.0, 3.0e3), (0.0, 2.0e3), (0.0, 1.8e3), periodic=(False, True, False))
    velbc = mesh.velbc(WALLS)
    bs = cases.base_state(mesh, "constBVFreq")
    rng = np.random.default_rng(p)
    bs.CORIOLIS[:] = 1.0e-4 * (1.0 + 0.3 * rng.standard_normal(bs.CORIOLIS.size))
    om = O.OracleMesh(mesh, velbc=velbc)
    dm = fedg.DeviceMesh(mesh, velbc=velbc, box_shape=box_shape)
    n = mesh.Np * mesh.Ne
    q = [mesh.field() for _ in range(5)]
    for f, amp in zip(q, (1e-3, 0.3, 0.5, 5.0, 1.0)):
        f[:n] = amp * rng.standard_normal(n)
        om.exchange(f)
    om.apply_bc(q)
    return mesh, bs, om, dm, q, n, rng


@pytest.mark.parametrize("box_shape", [True, False], ids=["flat", "general"])
@pytest.mark.parametrize("p", range(1, 8))
def test_dropin_bitwise(p, box_shape):
    print(f"element kernel, drop-in, p={p} box_shape={box_shape}", flush=True)
    mesh, bs, om, dm, q, n, _ = build(p, box_shape)
    Dx, Dy = om.calc_phyd_hgrad(bs)
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
    dm.close()


@pytest.mark.parametrize("box_shape", [True, False], ids=["flat", "general"])
@pytest.mark.parametrize("p", range(1, 8))
def test_fused_bitwise(p, box_shape):
    mesh, bs, om, dm, q, n, rng = build(p, box_shape)
    c = constants.SCALE  # the steppers are dry
    nA = mesh.Np * mesh.NeA
    bs = dataclasses.replace(bs, Rtot=np.full(nA, c.Rdry), CVtot=np.full(nA, c.CVdry), CPtot=np.full(nA, c.CPdry))
    F = fedg.modalfilter_matrix(p, 0.0, 0.25, 8)
    dm.setup_modalfilter(F, F)
    dt = 0.02
    for varying in (False, True):
        if varying:
            f = bs.DENS_hyd.copy()
            f[:n] *= 1.0 + 1e-3 * rng.standard_normal(n)
            om.exchange(f)
            bs = dataclasses.replace(bs, DENS_hyd=f)
        Dx, Dy = om.calc_phyd_hgrad(bs)
        for scheme, filt in (("ERK_4s4o", False), ("ERK_4s4o", True), ("ERK_1s1o", True)):
            print(f"element kernel, fused, p={p} box_shape={box_shape} varying={varying} {scheme} filter={filt}", flush=True)
            st = fedg.HeveStepper(dm, bs, Dx, Dy, dt, scheme=scheme)
            st.set_modalfilter(filt)
            st.set_state(q)
            st.run(2)
            g = st.get_state()
            _, Dg = st.get_pressure()
            st.close()
            om.set_modalfilter(*((F, F) if filt else ()))
            r = [a.copy() for a in q]
            om.heve_update(r, bs, Dx, Dy, dt, 2, scheme=scheme)
            for name, a, b in zip(fedg.VARS, g, r):
                assert np.array_equal(a, b[:n]), f"{name} varying={varying} {scheme} filter={filt}"
            assert np.array_equal(Dg, om.drhot2pres(r[1], bs)[1][:n])
    dm.close()
