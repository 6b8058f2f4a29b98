"""The neighbourhood sums of the surrogate at the edges of their lists: nodes
without edges, lists of one edge, of a whole group and one more, of several
list reads, and node counts that leave the last wave part of its nodes."""
import importlib

import numpy as np
import pytest

from cases import fv  # noqa: F401

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _graph(degrees, seed):
    rng = np.random.default_rng(seed)
    n, off = len(degrees), np.concatenate([[0], np.cumsum(degrees)]).astype(np.int32)
    E = int(off[-1])
    g = dict(off=off, col=rng.integers(0, n, E).astype(np.int32), n=n)
    for k in ("w", "ex", "ey", "wt", "ext", "eyt"):
        g[k] = rng.uniform(-1, 1, E).astype(np.float32)
    return g


def _sum(v, src, n):
    out = np.zeros((n, v.shape[1]))
    np.add.at(out, src, v)
    return out


@pytest.mark.parametrize("degrees", [
    [1], [1, 0], [0, 0, 0, 17], [512, 0, 1], [15, 16, 17, 0, 0, 31, 32, 33],
    [63, 64, 65, 127, 128, 129, 1, 0, 0], [0] * 5 + [600] + [0] * 4, [7] * 258 + [300],
    [2] * 131071 + [100], [3, 0] * 65537 + [65],
], ids=lambda d: f"n{len(d)}_max{max(d)}")
def test_sums_at_list_edges(gpu, degrees):
    import torch
    sg = importlib.import_module("fvdbm-jax_amd.surrogate")
    g = _graph(degrees, len(degrees))
    n, col = g["n"], g["col"]
    deg = np.asarray(degrees)
    src = np.repeat(np.arange(n), deg)
    rng = np.random.default_rng(5)
    h = rng.standard_normal((n, 64)).astype(np.float32)
    dz = rng.standard_normal((n, 256)).astype(np.float32)
    hd = torch.tensor(h, device="cuda", requires_grad=True)
    z = sg.aggregate(hd, sg.graph_to_device(g))
    z.backward(torch.tensor(dz, device="cuda"))

    e = {k: g[k].astype(np.float64)[:, None] for k in ("w", "ex", "ey", "wt", "ext", "eyt")}
    h64, dz64 = h.astype(np.float64), dz.astype(np.float64)
    parts = [e["w"] * h64[col], e["w"] * e["ex"] * h64[col], e["w"] * e["ey"] * h64[col]]
    want = np.concatenate([h64] + [_sum(p, src, n) for p in parts], 1)
    size = np.concatenate([0 * h64] + [_sum(abs(p), src, n) for p in parts], 1)
    # a sum of d terms of two roundings each: (d + 2) roundings of sum |term|
    got = z.detach().cpu().numpy()
    assert np.all(abs(got - want) <= (deg[:, None] + 3) * EPS * size)

    dj = dz64[col]
    terms = [e["wt"] * dj[:, 64:128], e["wt"] * e["ext"] * dj[:, 128:192], e["wt"] * e["eyt"] * dj[:, 192:]]
    want = dz64[:, :64] + _sum(sum(terms), src, n)
    size = abs(dz64[:, :64]) + _sum(sum(abs(t) for t in terms), src, n)
    got = hd.grad.cpu().numpy()
    assert np.all(abs(got - want) <= (deg[:, None] + 4) * EPS * size)
