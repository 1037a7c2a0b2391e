"""The element sums of the tracer kernels at the orders the other tests leave
out (sums with a remainder, one to many elements per workgroup, a last workgroup
that is not full, closed and periodic sides) and the negative fixer over the
number of species and the orders, against the oracle bit for bit."""
import numpy as np
import pytest

import fedg
import fedg_oracle as O
import test_gpu_trcadv as T

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def portable_pow():
    with O.pow_mode(O.POW_PORTABLE):
        yield


@pytest.mark.parametrize("metrics", ["random", "flat"])
@pytest.mark.parametrize("case", [(1, 2, 2, 2, (False, False, True)), (2, 5, 3, 2, (False, True, False)),
                                  (5, 3, 1, 3, (True, False, False)), (6, 2, 3, 2, (True, True, False)),
                                  (7, 3, 3, 1, (False, False, False))], ids=lambda c: f"p{c[0]}")
def test_tracer_kernels(case, metrics):
    T.test_trcadvect_cal_tend_bitwise(case, metrics)
    T.test_trcadvect_fct_tmar_massflux_bitwise(case, metrics)


@pytest.mark.parametrize("p", range(1, 8))
@pytest.mark.parametrize("nq", [1, 4, 5, 8])
def test_negative_fixer(p, nq):
    print(f"negative fixer p={p} nq={nq}", flush=True)
    mesh = fedg.BoxMesh(p, 3, 1, 3, (0.0, 6e3), (0.0, 2e3), (0.0, 4.5e3))
    rng = np.random.default_rng(10 * p + nq)
    n = mesh.Np * mesh.Ne
    om, dm = O.OracleMesh(mesh), fedg.DeviceMesh(mesh)
    thermo = (np.ones(nq), rng.uniform(0.0, 500.0, nq), rng.uniform(1e3, 4e3, nq), rng.uniform(1e3, 4e3, nq))

    def field(base, amp):
        a = mesh.field()
        a[:n] = base + amp * rng.standard_normal(n)
        return a

    Q = [field(2e-5, 2e-5) for _ in range(nq)]
    Q[0][:mesh.Np] = -1e-6  # an element without any of it
    DD, DR, P = field(0.0, 1e-3), field(0.0, 0.1), field(9e4, 1e3)
    R, CV, CP = field(287.0, 1.0), field(718.0, 1.0), field(1005.0, 1.0)
    Dh, Ph = field(1.0, 0.05), field(9e4, 1e3)
    dev = lambda a: fedg.DevField(a.size, a.copy())  # noqa: E731
    z = mesh.height.copy()
    gQ, g = [dev(a) for a in Q], [dev(a) for a in (DD, P, CV, CP, R)]
    gDR = dev(DR)
    fedg.trc_negative_fixer(dm, gQ, *g, dev(Dh), dev(Ph), dev(mesh.J.copy()), dev(z), thermo, QLA=nq - 1, DRHOT=gDR)
    om.trc_negative_fixer(Q, DD, P, CV, CP, R, Dh, Ph, mesh.J, z, thermo, DRHOT=DR)
    for name, a, b in [(f"Q{i}", a, b) for i, (a, b) in enumerate(zip(gQ, Q))] + list(
            zip(("DDENS", "PRES", "CVtot", "CPtot", "Rtot"), g, (DD, P, CV, CP, R))) + [("DRHOT", gDR, DR)]:
        assert np.array_equal(a.download()[:n], b[:n]), name
    dm.close()
