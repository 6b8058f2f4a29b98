"""FP64 batches of boundary-heavy porous cases run multi-step tiles at every
block size: tiles whose tables exceed a block's LDS are built as parts, or in
half the size. Bitwise equal to the oracle's single solves."""
import importlib

import numpy as np
import pytest

from cases import fv, oracle_env, oracle_state
from oracle import oracle

batch = importlib.import_module("fvdbm-jax_amd.batch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [128, 256, 512])
def test_fp64_workload_batch_takes_multi_step_tiles(gpu, block):
    cases = [fv.porous.make_case(seed, dist=fv.porous.WORKLOAD, target_cells=t)
             for seed, t in ((11, 20_000), (12, 31_000), (13, 47_000))]
    b = batch.BatchSolver([c.env_tuple() for c in cases], precision="fp64", block=block)
    assert not b.info()["variant"] & 8 and b.info()["launch_classes"] == 1
    b.step(19)
    b.run(10, 5, 0.0)
    pdf = b.get_pdf()
    for k, c in enumerate(cases):
        oenv = oracle_env(c.cells, c.faces, c.nodes, "f64")
        st = oracle_state(oenv, c.nodes, "f64")
        oracle.run(oenv, st, c.dynamics.tau, c.dynamics.delta_t, 29, "f64")
        assert np.isfinite(st["cell_pdf"]).all()
        assert np.array_equal(b.case_pdf(k, pdf), st["cell_pdf"]), (block, k)
    b.close()


def test_tiles_that_join_the_layouts(gpu):
    """A batch of more than 768 cells per CU in tiles of 64 steps in tiles of 128
    cells of one case, whole and ragged: bitwise equal to one step per launch."""
    cases = [fv.porous.make_case(s, dist=fv.porous.STEADY, target_cells=t).env_tuple()
             for s, t in ((1, 90_001), (2, 70_003), (3, 63_005))]
    pdfs = []
    for block, variant in ((64, 0), (64, 8), (192, 0)):
        b = batch.BatchSolver(cases, precision="fp64", block=block, variant=variant)
        assert b.info()["n_cells_padded"] > 768 * 256
        assert bool(b.info()["variant"] & 8) == bool(variant)
        b.step(11)
        b.run(8, 4, 0.0)
        pdfs.append(b.get_pdf())
        b.close()
    assert np.isfinite(pdfs[0]).all()
    assert np.array_equal(pdfs[0], pdfs[1]) and np.array_equal(pdfs[0], pdfs[2])
