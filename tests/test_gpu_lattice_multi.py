"""Multi-step tiles of the any-lattice handles: D2Q13 runs that end on every
step count of a launch, against the CPU oracle, every observable bitwise:
less than a tile, ragged last tiles, tiles that are all boundary, both flux
schemes and both precisions (whose blocks hold 1024 or 512 cells)."""
import numpy as np
import pytest

from cases import channel_case, fv, ldc_case, meshgen, oracle_env, oracle_state
from oracle import oracle

pytestmark = pytest.mark.gpu


def _case(name, scheme):
    if name.startswith("cavity"):  # 2 n^2 cells
        return ldc_case(n=int(name[6:]), scheme=scheme, lattice=fv.D2Q13)[1:]
    if name == "strip":  # one triangle thick: every tile is boundary, rings are long
        raw = meshgen.jittered_delaunay(2.0, 0.01, [], 0.01, seed=5)
    else:
        raw = meshgen.cylinder_channel(int(name[7:]), seed=2)
    return channel_case(raw, tau=0.6, dt=1e-3, u_max=0.05, dim_multiplier=1.0, scheme=scheme,
                        lattice=fv.D2Q13)[1:]


@pytest.mark.parametrize("name,scheme,precision,block", [
    ("cavity3", "upwind", "fp32", 0),         # 18 cells: less than a tile
    ("cavity11", "upwind", "fp64", 64),       # ragged last tile
    ("cavity91", "upwind", "fp32", 0),        # one cell past the small-tile size
    ("cavity40", "lax_wendroff", "fp32", 448),
    ("cavity40", "lax_wendroff", "fp64", 0),
    ("strip", "upwind", "fp32", 1024),        # the block's tile is a part of it
    ("strip", "lax_wendroff", "fp32", 0),
    ("channel20000", "upwind", "fp64", 512),
    ("channel20000", "upwind", "fp32", 256),
])
def test_every_run_length_matches_the_oracle(gpu, name, scheme, precision, block):
    dyn, c, f, n = _case(name, scheme)
    p = "f64" if precision == "fp64" else "f32"
    env = fv.Environment(c, f, n, precision=precision, block=block)
    env.init()
    assert env.info()["variant"] == 4
    oenv = oracle_env(c, f, n, p)
    st = oracle_state(oenv, n, p, 13)
    done = 0
    nodes = np.asarray(n.type).reshape(-1) != 0
    for k in (2, 3, 1, 4, 5, 6, 7, 8, 9, 17, 130):
        print(f"{name} {scheme} {precision} block {block}: {k} steps", flush=True)
        env.step(k)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, k, p, scheme=scheme, quivers=13)
        done += k
        got = dict(pdf=env.cells.pdf, rho=env.cells.rho, vel=env.cells.vel, feq=env.cells.pdf_eq,
                   flux=env.faces.pdf, node=env.nodes.pdf[nodes])
        want = dict(pdf=st["cell_pdf"], rho=st["cell_rho"], vel=st["cell_vel"], feq=st["cell_feq"],
                    flux=st["face_pdf"], node=st["node_pdf"][nodes])
        for key in got:
            assert np.array_equal(got[key], np.asarray(want[key]).reshape(got[key].shape)), (name, done, key)
    assert np.isfinite(st["cell_pdf"]).all()
    env.close()
