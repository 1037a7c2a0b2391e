"""The halo exchange of as many fields as one launch takes, one fewer and more,
against the mesh's own exchange, bit for bit."""
import numpy as np
import pytest

import fedg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfields", [1, 7, 8, 9, 17])
def test_halo_of_many_fields(nfields):
    m = fedg.BoxMesh(2, 3, 2, 2, (0.0, 3.0e3), (0.0, 2.0e3), (0.0, 2.0e3), periodic=(False, True, False))
    dm = fedg.DeviceMesh(m)
    rng = np.random.default_rng(nfields)
    host = [rng.standard_normal(m.Np * m.NeA) for _ in range(nfields)]
    dev = [fedg.DevField(a.size, a) for a in host]
    fedg.halo_exchange(dm, dev)
    for v, (d, a) in enumerate(zip(dev, host)):
        m.exchange(a)
        assert np.array_equal(d.download(), a), f"field {v} of {nfields}"
    dm.close()
