"""Velocities and equilibria of the multi-step kernels over densities from far
below to far above 1, inside and outside the range where both velocities share
one reciprocal (2^-32 .. 2^32): one and two steps equal the oracle, whose
divisions are IEEE, bit for bit."""
import numpy as np
import pytest

from cases import fv, ldc_case, oracle_env, oracle_state
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quivers", [9, 13])
@pytest.mark.parametrize("exponents", [(-2, 2), (-31, -28), (28, 31), (-40, 40)])
def test_any_density_matches_the_oracle(gpu, quivers, exponents):
    m, dyn, cells, faces, nodes = ldc_case(n=24, lattice=fv.D2Q13 if quivers == 13 else None)
    rng = np.random.default_rng(100 + quivers + exponents[1])
    W = np.asarray(oracle.W13_64 if quivers == 13 else oracle.W64)
    f = W * (1 + 0.3 * rng.uniform(-1, 1, (cells.size, quivers)))
    f *= 2.0 ** rng.uniform(*exponents, (cells.size, 1))
    f = f.astype(np.float32)
    env = fv.Environment(cells, faces, nodes)
    env.init()
    env.cells.pdf = f
    oenv = oracle_env(cells, faces, nodes)
    st = oracle_state(oenv, nodes, "f32", quivers)
    st["cell_pdf"] = f.copy()
    for k in (1, 2):
        env.step(k)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, k, "f32", quivers=quivers)
        assert np.isfinite(st["cell_pdf"]).all()
        for got, want in ((env.cells.pdf, "cell_pdf"), (env.cells.vel, "cell_vel"), (env.cells.pdf_eq, "cell_feq")):
            assert np.array_equal(got, np.asarray(st[want]).reshape(got.shape)), (k, want)
    env.close()
