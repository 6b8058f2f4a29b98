"""Multi-step launches of meshes whose cells are numbered with wide rings (in the
mesh's order, on a grid, in reverse Cuthill-McKee order): the same bits as one step
per launch, and tables no larger than those of tiles that are mostly whole."""
import numpy as np
import pytest

from cases import build_mesher, fv, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,precision", [(20_000, "fp32"), (60_000, "fp32"), (20_000, "fp64")])
def test_cell_orders(gpu, cells, precision):
    dyn = fv.D2Q9(tau=0.6, delta_t=1e-5)
    m = build_mesher(meshgen.cylinder_channel(cells, seed=1))
    c, f, n = m.to_env(dyn, "upwind", dim_multiplier=1)
    n = m.set_vel_node(n, meshgen.WALL, np.array([0.0, 0.0]))
    n = m.set_vel_node(n, meshgen.INLET, np.array([0.05, 0.0]))
    n = m.set_rho_node(n, meshgen.OUTLET, 1.0)
    size = {}
    for reorder in (0, 1, 2, 3, 4):
        pdf = []
        for variant in (0, 8):
            env = fv.Environment(c, f, n, precision=precision, reorder=reorder, variant=variant)
            env.init()
            if not variant:
                size[reorder] = env.info()["device_bytes"]
            print(f"{cells} cells {precision} order {reorder} variant {variant}", flush=True)
            env.step(21)
            pdf.append(env.cells.pdf)
            env.close()
        assert np.isfinite(pdf[0]).all() and np.array_equal(*pdf), reorder
    if (cells, precision) == (60_000, "fp32"):
        assert size[2] < 1.3 * size[4], size
