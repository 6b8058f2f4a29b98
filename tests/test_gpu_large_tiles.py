"""Multi-step tiles of more than 64 cells: runs that end on every step count of a
launch against the CPU oracle, every observable bitwise, on meshes above 16384
padded cells, where the tile is the block or a part of it (up to there it is 64
whatever is asked for): both flux schemes, lattices and precisions, tiles that
are no multiple of 128, and blocks whose tile is a part of them."""
import numpy as np
import pytest

from cases import fv, ldc_case, oracle_env, oracle_state, porous_case
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh,lattice,scheme,precision,block", [
    ("cavity", "D2Q9", "lax_wendroff", "fp32", 256),
    ("cavity", "D2Q9", "lax_wendroff", "fp32", 1024),  # tiles of 512
    ("cavity", "D2Q9", "lax_wendroff", "fp64", 256),
    ("cavity", "D2Q9", "lax_wendroff", "fp64", 320),
    ("cavity", "D2Q9", "lax_wendroff", "fp64", 1024),  # tiles of 256
    ("cavity", "D2Q9", "upwind", "fp64", 256),
    ("cavity", "D2Q9", "upwind", "fp64", 448),
    ("cavity", "D2Q9", "upwind", "fp32", 320),
    ("cavity", "D2Q13", "lax_wendroff", "fp32", 448),  # no room for a ring: one step per launch
    ("cavity", "D2Q13", "lax_wendroff", "fp32", 320),
    ("cavity", "D2Q13", "lax_wendroff", "fp64", 256),  # tiles of 128
    ("porous", "D2Q9", "upwind", "fp64", 128),
    ("porous", "D2Q9", "upwind", "fp32", 1024),
])
def test_every_run_length_matches_the_oracle(gpu, mesh, lattice, scheme, precision, block):
    if mesh == "cavity":
        dyn, c, f, nd = ldc_case(n=92, scheme=scheme, lattice=getattr(fv, lattice))[1:]
    else:
        dyn, c, f, nd = porous_case(4, target_cells=20_000, scheme=scheme)[1:]
    p = "f64" if precision == "fp64" else "f32"
    q = int(dyn.NUM_QUIVERS)
    env = fv.Environment(c, f, nd, precision=precision, block=block)
    env.init()
    info = env.info()
    assert info["n_cells_padded"] > 16384 and info["block"] == block
    assert bool(info["variant"] & 8) == ((lattice, block) == ("D2Q13", 448))
    oenv = oracle_env(c, f, nd, p)
    st = oracle_state(oenv, nd, p, q)
    nodes = np.asarray(nd.type).reshape(-1) != 0
    done = 0
    for k in (2, 3, 4, 5, 6, 7, 8, 9, 1, 17, 40):
        print(f"{mesh} {lattice} {scheme} {precision} block {block}: {k} steps", flush=True)
        env.step(k)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, k, p, scheme=scheme, quivers=q)
        done += k
        got = dict(pdf=env.cells.pdf, rho=env.cells.rho, vel=env.cells.vel, feq=env.cells.pdf_eq,
                   flux=env.faces.pdf, node=env.nodes.pdf[nodes])
        want = dict(pdf=st["cell_pdf"], rho=st["cell_rho"], vel=st["cell_vel"], feq=st["cell_feq"],
                    flux=st["face_pdf"], node=st["node_pdf"][nodes])
        for key in got:
            assert np.array_equal(got[key], np.asarray(want[key]).reshape(got[key].shape)), (done, key)
    assert np.isfinite(st["cell_pdf"]).all()
    env.close()
