"""Multi-step tiles (k_multi): runs that end on every step count of a launch,
at the edges of their tiles, against the CPU oracle, every observable
bitwise: meshes smaller than one tile, ragged last tiles, tiles that are all
boundary, tiles split because their ring outgrows the block, both flux
schemes and both precisions."""
import numpy as np
import pytest

from cases import channel_case, fv, ldc_case, meshgen, oracle_env, oracle_state, porous_case
from oracle import oracle

pytestmark = pytest.mark.gpu


def _strip(scheme):  # one triangle thick: every tile is boundary, rings are long
    raw = meshgen.jittered_delaunay(2.0, 0.01, [], 0.01, seed=5)
    m, dyn, c, f, n = channel_case(raw, tau=0.6, dt=1e-3, u_max=0.05, dim_multiplier=1.0, scheme=scheme)
    return dyn, c, f, n


def _case(name, scheme):
    if name == "strip":
        return _strip(scheme)
    if name.startswith("cavity"):  # 2 n^2 cells
        return ldc_case(n=int(name[6:]), scheme=scheme)[1:]
    return porous_case(4, target_cells=int(name[6:]), scheme=scheme)[1:]


def _check(env, st, what):
    nodes = np.asarray(env.nodes.type).reshape(-1) != 0
    got = dict(pdf=env.cells.pdf, rho=env.cells.rho, vel=env.cells.vel, feq=env.cells.pdf_eq,
               flux=env.faces.pdf, node=env.nodes.pdf[nodes])
    want = dict(pdf=st["cell_pdf"], rho=st["cell_rho"], vel=st["cell_vel"], feq=st["cell_feq"],
                flux=st["face_pdf"], node=st["node_pdf"][nodes])
    for k in got:
        assert np.array_equal(got[k], np.asarray(want[k]).reshape(got[k].shape)), (what, k)


@pytest.mark.parametrize("name,scheme,precision,block", [
    ("cavity3", "upwind", "fp32", 0),         # 18 cells: less than a tile
    ("cavity11", "upwind", "fp32", 64),       # ragged last tile
    ("cavity11", "lax_wendroff", "fp32", 0),
    ("cavity91", "upwind", "fp32", 0),        # one cell past the small-tile size
    ("cavity40", "lax_wendroff", "fp64", 128),
    ("strip", "upwind", "fp32", 1024),        # the block's tile is a part of it
    ("strip", "upwind", "fp64", 320),
    ("porous9000", "upwind", "fp32", 128),
    ("porous20000", "upwind", "fp32", 512),
])
def test_every_run_length_matches_the_oracle(gpu, name, scheme, precision, block):
    dyn, c, f, n = _case(name, scheme)
    p = "f64" if precision == "fp64" else "f32"
    env = fv.Environment(c, f, n, precision=precision, block=block)
    env.init()
    assert not env.info()["variant"] & 8
    oenv = oracle_env(c, f, n, p)
    st = oracle_state(oenv, n, p)
    done = 0
    for k in (2, 3, 4, 5, 6, 7, 8, 9, 17, 130):
        print(f"{name} {scheme} {precision} block {block}: {k} steps", flush=True)
        env.step(k)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, k, p, scheme=scheme)
        done += k
        _check(env, st, (name, done))
    assert np.isfinite(st["cell_pdf"]).all()
    env.close()


@pytest.mark.parametrize("block", [64, 128, 256])
def test_batch_intervals_of_every_length(gpu, block):
    """Intervals whose last launch holds 1 to 4 steps, with a case frozen in
    between: each case equals its own solve."""
    batch = __import__("importlib").import_module("fvdbm-jax_amd.batch")
    cs = [porous_case(s, target_cells=3000 + 1100 * s)[1:] for s in range(3)]
    b = batch.BatchSolver([(c, f, n) for _, c, f, n in cs], block=block)
    want = [0, 0, 0]
    for i, k in enumerate((1, 2, 3, 5, 6, 11)):
        mask = np.ones(3, np.int32)
        mask[i % 3] = i < 3
        b.set_active(mask)
        b.run(k, k, 0.0, 0.0) if i % 2 else b.step(k)
        want = [w + k * int(a) for w, a in zip(want, mask)]
    pdf = b.get_pdf()
    for j, (dyn, c, f, n) in enumerate(cs):
        oenv = oracle_env(c, f, n)
        st = oracle_state(oenv, n)
        oracle.run(oenv, st, dyn.tau, dyn.delta_t, want[j], "f32")
        assert np.array_equal(b.case_pdf(j, pdf), st["cell_pdf"]), (block, j)
    b.close()
