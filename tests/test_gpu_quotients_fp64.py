"""The FP64 divisions of the multi-step kernels: velocities by a shared reciprocal
for densities inside 2^-32 .. 2^32 and IEEE outside, equilibria by two-operation
constant division below u.u = 1/2 and IEEE from there, and dividends so small
that the brackets absorb them. One and two steps equal the oracle bit for bit."""
import numpy as np
import pytest

from cases import fv, ldc_case, oracle_env, oracle_state
from oracle import oracle

pytestmark = pytest.mark.gpu


def _check(quivers, n, f):
    m, dyn, cells, faces, nodes = ldc_case(n=n, lattice=fv.D2Q13 if quivers == 13 else None)
    env = fv.Environment(cells, faces, nodes, precision="fp64")
    env.init()
    oenv = oracle_env(cells, faces, nodes, "f64")
    for steps in (1, 2):
        env.cells.pdf = f
        st = oracle_state(oenv, nodes, "f64", quivers)
        st["cell_pdf"] = f.copy()
        env.step(steps)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, steps, "f64", quivers=quivers)
        assert np.isfinite(st["cell_pdf"]).all()
        for got, want in ((env.cells.pdf, "cell_pdf"), (env.cells.vel, "cell_vel"), (env.cells.pdf_eq, "cell_feq")):
            assert np.array_equal(got, np.asarray(st[want]).reshape(got.shape)), (steps, want)
    env.close()


@pytest.mark.parametrize("quivers", [9, 13])
@pytest.mark.parametrize("exponents", [(-2, 2), (-33, -28), (28, 33), (-40, 40)])
def test_any_density_matches_the_oracle(gpu, quivers, exponents):
    rng = np.random.default_rng(300 + quivers + exponents[1])
    W = np.asarray(oracle.W13_64 if quivers == 13 else oracle.W64)
    cells = 2 * 24 * 24
    f = W * (1 + 0.3 * rng.uniform(-1, 1, (cells, quivers))) * 2.0 ** rng.uniform(*exponents, (cells, 1))
    _check(quivers, 24, f)


# (rest population or None for W0, {q: added}): q = 1..4 are +x, +y, -x, -y
RECIPES = [
    (None, {}),                                 # u = 0 exactly
    (None, {1: 2.0 ** -50}),                    # momenta of a few ulps of 1
    (1e9, {2: 2.0 ** -40}),                     # u ~ 1e-21, density inside the range
    (4e9, {1: 2.0 ** -20, 4: 2.0 ** -20}),      # ux = -uy: ksi.u of q5 = 0
    (5e9, {1: 2.0 ** -20, 2: 2.0 ** -20}),      # ux = uy, density past the range
    (1e25, {1: 2.0 ** -26}),                    # u ~ 1e-33
    (None, {1: 0.05, 2: 0.02}),                 # moderate
    (None, {1: 2.4142135623730945}),            # u.u on either side of 1/2
    (None, {1: 2.4142135623730954}),
    (None, {1: 3.0, 2: 1.0}),                   # u.u > 1/2 (D2Q9)
]


@pytest.mark.parametrize("quivers", [9, 13])
def test_division_paths_match_the_oracle(gpu, quivers):
    W = np.asarray(oracle.W13_64 if quivers == 13 else oracle.W64)
    f = np.tile(W, (2 * 8 * 8, 1))
    for c in range(len(f)):
        rest, add = RECIPES[c % len(RECIPES)]
        f[c, 0] = f[c, 0] if rest is None else rest
        for q, v in add.items():
            f[c, q] += v
    _check(quivers, 8, f)
