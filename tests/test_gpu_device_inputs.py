"""Inputs of a prediction built on the device (fvdbm_nn_device_inputs) against
the host construction of each case: the graph's lists equal, directions and
features to float32 rounding; and the same refusals."""
import copy
import dataclasses

import numpy as np
import pytest

from cases import fv

pytestmark = pytest.mark.gpu

surrogate = __import__("importlib").import_module("fvdbm-jax_amd.surrogate")
porous = fv.porous


def _group(sizes):
    return [porous.make_case(40 + i, porous.STEADY, target_cells=s) for i, s in enumerate(sizes)]


@pytest.mark.parametrize("sizes,grid,resolution", [
    ([3001], (32, 16), True),
    ([2500, 4001, 3203], (32, 16), True),
    ([2500, 3203], (32, 1), False),   # slabs
    ([2500], (1, 1), True),           # one grid node lists every mesh node
    ([4001, 2500], (5, 3), False),
])
def test_device_inputs_match_the_host(gpu, sizes, grid, resolution):
    cases = _group(sizes)
    x, g, mesh, check = surrogate.device_inputs(cases, grid, resolution)
    check()
    ins = [surrogate.case_inputs(c, grid, resolution) for c in cases]
    want = surrogate.concat_graphs([i[1] for i in ins], edge_keys=("w", "ex", "ey"))
    assert g["n"] == want["n"] and np.diff(mesh["nodes"]).tolist() == [i[2] for i in ins]
    for k in ("off", "col", "w"):
        assert np.array_equal(g[k].cpu().numpy(), want[k]), k
    for k in ("ex", "ey"):  # hypot may round differently: one ulp of a value of at most 1
        assert np.abs(g[k].cpu().numpy() - want[k]).max() <= 2**-23, k
    # a feature is (float32(v) - shift) / scale: v and the result each to an ulp
    shift = np.abs(np.concatenate([surrogate.FEATURE_SHIFT, [0, 0], surrogate.SECTION_SHIFT, [0]]))
    scale = np.concatenate([surrogate.FEATURE_SCALE, [1, 1], surrogate.SECTION_SCALE, [1]])
    xh = np.concatenate([i[0] for i in ins])
    bound = 2**-22 * (np.abs(xh) + shift / scale)
    assert (np.abs(x.cpu().numpy() - xh) <= bound).all()


@pytest.mark.parametrize("what", ["edge", "node"])
def test_device_inputs_refuse_what_the_host_refuses(gpu, what):
    cases = _group([2500, 2700])
    mesher = copy.copy(cases[1].mesher)
    if what == "edge":
        mesher.faces = np.array(mesher.faces)
        mesher.faces[17, 1] = len(mesher.points)
    else:
        mesher.points = np.array(mesher.points)
        mesher.points[23, 0] = -0.5
    cases[1] = dataclasses.replace(cases[1], mesher=mesher)
    with pytest.raises(ValueError) as host:
        surrogate.case_inputs(cases[1], (32, 16), True)
    check = surrogate.device_inputs(cases, (32, 16), True)[3]
    with pytest.raises(ValueError) as device:
        check()
    assert str(device.value) == str(host.value)


def test_predicted_fields_match_the_host(gpu):
    """A prediction's fields and calibration equal what numpy makes of the
    network's output: elementwise operations in double, the calibration's sums
    in another order (1e-15 of a factor), stored float32."""
    import torch

    cases = _group([2500, 4001, 3203])
    net = surrogate.MeshNet.load(surrogate.__file__.replace("surrogate.py", "data/surrogate_porous.npz"))
    x, g, mesh, check = surrogate.device_inputs(cases, net.grid, net.resolution)
    with torch.no_grad():
        y = net.forward(x, g).cpu().numpy().astype(np.float64) * net.target_scale
    rows = np.cumsum([0] + [len(c.mesher.points) + net.grid[0] * net.grid[1] + 1 for c in cases])
    plain, scaled = net.predict(cases, calibrate=False), net.predict(cases)
    for c, o, p, s in zip(cases, rows, plain, scaled):
        yy = y[o:o + len(c.mesher.points)] * c.u_in
        r, v = (1.0 + yy[:, 0]).astype(np.float32), yy[:, 1:3].astype(np.float32)
        assert np.array_equal(p[0], r) and np.array_equal(p[1], v)
        r, v = surrogate.apply_calibration(net.calib, c, r, v)
        assert np.abs(s[0] - r).max() <= 2**-23 and np.abs(s[1] - v).max() <= 2**-24  # an ulp below 2, 1
