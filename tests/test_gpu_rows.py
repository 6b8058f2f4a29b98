"""Fields in and out of the device: rows set and read back are the same rows,
on either side of the sizes where the transfer changes its route (1 MB in,
2 MB out), in every precision and lattice, and for a batch whose cases sit in
different buffers."""
import importlib

import numpy as np
import pytest

from cases import fv, ldc_case, porous_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,lattice", [
    (1, "fp32", None), (32, "fp32", None), (32, "fp64", None),
    (120, "fp32", None),   # 28,800 cells: 1.04 MB
    (121, "fp32", None),   # 29,282 cells: 1.05 MB
    (170, "fp32", None),   # 57,800 cells: 2.08 MB
    (171, "fp32", None),   # 58,482 cells: 2.11 MB
    (171, "fp64", None), (120, "fp32", "D2Q13"), (101, "fp64", "D2Q13"),
])
def test_rows_round_trip(gpu, n, precision, lattice):
    dyn, c, f, nd = ldc_case(n=n, lattice=getattr(fv, lattice) if lattice else None)[1:]
    env = fv.Environment(c, f, nd, precision=precision)
    env.init()
    rng = np.random.default_rng(n)
    for obj, name in ((env.cells, "pdf"), (env.nodes, "pdf"), (env.nodes, "rho"), (env.nodes, "vel")):
        want = rng.standard_normal(getattr(obj, name).shape).astype(env.dtype)
        setattr(obj, name, want)
        assert np.array_equal(getattr(obj, name), want), name
    env.close()


def test_batch_rows_follow_each_case(gpu):
    batch = importlib.import_module("fvdbm-jax_amd.batch")
    b = batch.BatchSolver([porous_case(s, target_cells=4000 + 900 * s)[2:] for s in range(3)])
    b.set_active([1, 0, 1])
    b.step(1)  # the stepped cases' state moves to the other buffer
    rng = np.random.default_rng(0)
    want = rng.standard_normal(b.get_pdf().shape).astype(np.float32)
    b.set_pdf(want)
    assert np.array_equal(b.get_pdf(), want)
    b.step(2)
    got = b.get_pdf()
    assert np.array_equal(b.case_pdf(1, got), want[b.cell_off[1]:b.cell_off[2]])
    assert not np.array_equal(b.case_pdf(0, got), want[:b.cell_off[1]])
    b.close()
