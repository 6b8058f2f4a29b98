"""Single steps of meshes and batches too large for one round of multi-step tiles
run in the one-step kernels, between multi-step launches: the same bits as one
step per launch throughout, observables included."""
import importlib

import numpy as np
import pytest

from cases import fv, ldc_case

batch = importlib.import_module("fvdbm-jax_amd.batch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,n,precision", [
    ("D2Q13", 450, "fp32"),  # 405k cells, past the line
    ("D2Q13", 300, "fp64"),  # 180k cells, before it
    ("D2Q9", 300, "fp32"),
])
def test_single_steps_between_longer_runs(gpu, lattice, n, precision):
    _, dyn, c, f, nd = ldc_case(n=n, lattice=getattr(fv, lattice))
    fields = []
    for variant in (0, 8):
        env = fv.Environment(c, f, nd, precision=precision, variant=variant)
        env.init()
        assert bool(env.info()["variant"] & 8) == bool(variant)
        for k in (1, 5, 1, 1, 9, 2, 1):
            print(f"{lattice} {2 * n * n} cells {precision} variant {variant}: {k} steps", flush=True)
            env.step(k)
        env.nodes.vel = np.asarray(env.nodes.vel) * 0.5  # boundary values change after a single step
        env.step(1)
        fields.append([env.cells.pdf, env.cells.rho, env.cells.vel, env.cells.pdf_eq, env.faces.pdf])
        assert env.info()["steps_done"] == 21
        env.close()
    for a, b in zip(*fields):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_single_steps_of_a_batch(gpu, precision):
    cs = [fv.porous.make_case(s, dist=fv.porous.STEADY, target_cells=t).env_tuple()
          for s, t in ((1, 150_000), (2, 130_000), (3, 150_000), (4, 40_001))]
    pdfs, status = [], []
    for variant in (0, 8):
        b = batch.BatchSolver(cs, precision=precision, variant=variant)
        for k in (1, 5, 1, 2):
            print(f"batch {precision} variant {variant}: {k} steps", flush=True)
            b.step(k)
        b.run(6, 2, 0.0)
        b.set_active([1, 0, 1, 1])
        b.run(7, 6, 0.0)
        pdfs.append(b.get_pdf())
        status.append(b.status())
        b.close()
    assert np.isfinite(pdfs[0]).all() and np.array_equal(*pdfs)
    for k in ("steps", "residual", "status"):
        assert np.array_equal(status[0][k], status[1][k]), k
