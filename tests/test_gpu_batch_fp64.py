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
