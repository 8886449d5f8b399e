"""The assembled system of meshes whose rows have as many blocks as a slice has
wavefronts, one more or fewer, and many more, and whose blocks have every
remainder of the contributions that are read together, against the oracle."""
import numpy as np
import pytest

import oracle_ffi as of
from acousticsim_amd import capi
from acousticsim_amd import workloads as wl
from obj_fixture import hub_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spokes", [3, 4, 5, 6, 12, 13, 14, 27, 28, 90])
def test_hub_system_matches_oracle(tmp_path, spokes):
    conf, x0 = hub_config(tmp_path / "hub.obj", spokes, precision="fp64")
    W, b = capi.BaraffClothHip(conf, x0).assemble_system()
    systems = []
    for c in (conf, dict(conf, cloth_bending_stiffness=[0, 0, 0])):
        oc = of.OracleCloth(c)
        oc.set_state(x0, x0)
        oc.assemble()
        systems.append((oc.W(), oc.rhs()))
    (Wo, bo), (W0, _) = systems
    rp, cols = oc.pattern()
    pinned = np.zeros(oc.nv, bool)
    pinned[oc.pins()] = True
    rows = np.repeat(np.arange(oc.nv), np.diff(rp))
    free = ~pinned[rows] & ~pinned[cols]
    assert free.sum() and np.all(W[~free] == 0)
    # a bending contribution is rounded to a float, which may differ by an ulp
    # where the device's atan2 does: at most 2^-23 of the largest bending entry
    # each, of up to 2 edges a spoke
    tol = 1e-12 * np.abs(Wo[free]).max() + 2.0 ** -23 * 2 * spokes * np.abs(Wo - W0)[free].max()
    assert np.abs(W[free] - Wo[free]).max() <= tol
    fr = np.repeat(~pinned, 3)
    assert np.abs(b[fr] - bo[fr]).max() <= 1e-12 * np.abs(bo[fr]).max()
    assert np.all(b[~fr] == 0)
