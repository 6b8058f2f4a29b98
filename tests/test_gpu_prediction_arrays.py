"""A prediction's fields are arrays of their own: keeping one case's does not keep
the others', and they are plain C-ordered float32."""
import importlib

import numpy as np
import pytest

from cases import fv

surrogate = importlib.import_module("fvdbm-jax_amd.surrogate")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("project", [False, True])
def test_every_case_gets_its_own_arrays(gpu, project):
    net = surrogate.MeshNet(layers=1, seed=5)
    cases = [fv.porous.make_case(60 + i, fv.porous.STEADY, target_cells=t) for i, t in enumerate((2500, 3301))]
    pred = net.predict(cases, project=project)
    for (r, v), c in zip(pred, cases):
        n = len(c.mesher.points)
        assert r.shape == (n,) and v.shape == (n, 2) and r.dtype == v.dtype == np.float32
        for a in (r, v):
            assert a.base is None and a.flags.owndata and a.flags.c_contiguous and a.flags.writeable
    again = net.predict(cases, project=project)
    kept = pred[0][0].copy()
    again[0][0][:] = 7.0
    assert np.array_equal(pred[0][0], kept)
