"""The HEVI line solves over the orders, column heights and line counts at
their edges (segments with idle lanes, a last group of lines that is not full,
one level) against the oracle, bit for bit: with blocks whose pivots stay on
the diagonal (small impl_fac) and leave it everywhere (large impl_fac), one
Newton iteration and Newton to a tolerance; with rows exchanged in the blocks of
some lines only, solved in one kernel and in two; and on meshes with more groups
of lines than wavefronts, which walk several groups each."""
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


def mixed_state(m, seed):
    rng = np.random.default_rng(seed)
    n = m.Np * m.Ne
    q = [m.field() for _ in range(5)]
    for f, a in zip(q, (1e-3, 0.3, 0.5, 5.0, 1.0)):
        f[:n] = a * rng.standard_normal(n)
        m.exchange(f)
    return q


# (p, NeX, NeY, NeZ, impl_fac, no-allocation entry, lines with exchanges: none / some / all).  On 256 CUs 16 x 9 x 2
# has more groups of lines than SIMDs (two kernels at p = 7), and more groups than wavefronts have 23 x 23 x 2 and
# 64 x 65 x 1 (4096 wavefronts) and, in the no-allocation entry's scratch, 12 x 12 x 8 (682).
WALKS = [(6, 3, 1, 3, 0.09, False, "some"), (7, 3, 1, 4, 0.06, False, "some"), (7, 16, 9, 2, 0.06, False, "some"),
         (7, 23, 23, 2, 0.01, False, "none"), (7, 23, 23, 2, 0.06, False, "some"), (7, 23, 23, 2, 6.0, False, "all"),
         (7, 12, 12, 8, 0.01, True, "none"), (7, 12, 12, 8, 0.06, True, "some"), (3, 64, 65, 1, 0.05, False, None)]


@pytest.mark.parametrize("p,NeX,NeY,NeZ,impl_fac,noalloc,exchanges", WALKS)
def test_mixed_pivots_and_many_groups(p, NeX, NeY, NeZ, impl_fac, noalloc, exchanges):
    print(f"line solves p={p} {NeX}x{NeY}x{NeZ} impl_fac={impl_fac} noalloc={noalloc}", flush=True)
    m = fedg.BoxMesh(p, NeX, NeY, NeZ, (0.0, 1.0e3 * NeX), (0.0, 1.0e3 * NeY), (0.0, 1.0e3 * NeZ))
    bs = cases.base_state(m, "constBVFreq")
    om = O.OracleMesh(m)
    dm = fedg.DeviceMesh(m)
    n = m.Np * m.Ne
    q, q0 = mixed_state(m, p), mixed_state(m, p + 100)
    with om.pivot_lines() as lines:
        ref, _, _ = om.hevi_cal_vi(q, q0, bs, impl_fac, 1.0)
    if exchanges:
        assert {"none": lines.sum() == 0, "some": 0 < lines.sum() < lines.size, "all": lines.all()}[exchanges]
    if p == 7 and exchanges == "some":  # and groups of eight lines of both kinds
        groups = lines.reshape(-1, 8).any(axis=1)
        assert 0 < groups.sum() < groups.size
    dev = lambda a: fedg.DevField(a.size, a)  # noqa: E731
    d, d0 = [dev(a) for a in q], [dev(a) for a in q0]
    aux = [dev(getattr(bs, k)) for k in ("DENS_hyd", "PRES_hyd", "Rtot", "CVtot", "CPtot")]
    out = [dev(m.field()) for _ in range(5)]
    fedg.hevi_cal_vi(dm, out, d[0], d[3], d[4], d[2], d[1], aux[0], aux[1], d0[0], d0[3], d0[4], d0[2], d0[1], *aux[2:],
                     impl_fac, 1.0, **(dict(max_it=1, noalloc=True) if noalloc else {}))
    g = [a.download() for a in out]
    for name, a, b in zip(fedg.VARS, [g[0], g[4], g[3], g[1], g[2]], ref):
        assert np.array_equal(a[:n], b[:n], equal_nan=True), name
    dm.close()


# the tallest column of every order
TALLEST = {1: 40, 2: 53, 3: 39, 4: 30, 5: 52, 6: 43, 7: 37}


@pytest.mark.parametrize("p", range(1, 8))
def test_tallest_column(p):
    print(f"line solves, tallest column p={p}", flush=True)
    for NeZ in (TALLEST[p], TALLEST[p] + 1):
        m = fedg.BoxMesh(p, 2, 1, NeZ, (0.0, 2.0e3), (0.0, 1.0e3), (0.0, 2.5e2 * NeZ))
        bs = cases.base_state(m, "constBVFreq")
        om = O.OracleMesh(m)
        dm = fedg.DeviceMesh(m)
        n = m.Np * m.Ne
        q, q0 = mixed_state(m, p), mixed_state(m, p + 100)
        dev = lambda a: fedg.DevField(a.size, a)  # noqa: E731
        d, d0 = [dev(a) for a in q], [dev(a) for a in q0]
        aux = [dev(getattr(bs, k)) for k in ("DENS_hyd", "PRES_hyd", "Rtot", "CVtot", "CPtot")]
        for noalloc in (False, True):
            out = [dev(m.field()) for _ in range(5)]
            call = lambda: fedg.hevi_cal_vi(dm, out, d[0], d[3], d[4], d[2], d[1], aux[0], aux[1], d0[0], d0[3],  # noqa: E731
                                            d0[4], d0[2], d0[1], *aux[2:], 0.02, 1.0,
                                            **(dict(max_it=1, noalloc=True) if noalloc else {}))
            if NeZ > TALLEST[p]:
                with pytest.raises(fedg.FedgError, match="too many elements in the vertical"):
                    call()
                continue
            call()
            ref, _, _ = om.hevi_cal_vi(q, q0, bs, 0.02, 1.0)
            g = [a.download() for a in out]
            for name, a, b in zip(fedg.VARS, [g[0], g[4], g[3], g[1], g[2]], ref):
                assert np.array_equal(a[:n], b[:n], equal_nan=True), f"{name} noalloc={noalloc}"
        dm.close()
