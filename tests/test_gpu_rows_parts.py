"""Fields larger than a handle's row buffer cross the bus in parts: every row
arrives both ways, and a read adds no more device memory than the buffer."""
import numpy as np
import pytest

from cases import fv, ldc_case

pytestmark = pytest.mark.gpu

BUFFER = 64 << 20


@pytest.mark.parametrize("lattice,n", [("D2Q9", 690), ("D2Q13", 575)])  # 68.6 and 68.8 MB of FP64 pdf
def test_a_field_larger_than_the_buffer(gpu, lattice, n):
    _, dyn, c, f, nd = ldc_case(n=n, lattice=getattr(fv, lattice))
    env = fv.Environment(c, f, nd, precision="fp64")
    env.init()
    q = int(dyn.NUM_QUIVERS)
    size = c.face_indices.shape[0]
    assert size * q * 8 > BUFFER
    before = env.info()["device_bytes"]
    rng = np.random.default_rng(3)
    pdf = rng.uniform(0.01, 0.5, (size, q))
    env.cells.pdf = pdf
    assert np.array_equal(env.cells.pdf, pdf)
    assert env.info()["device_bytes"] - before <= BUFFER
    env.close()
