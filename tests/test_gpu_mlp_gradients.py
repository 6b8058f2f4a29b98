"""All gradients of a two-layer block from one pass, at the edges of its row
tiles (32 rows), of its grid (a block has at least four tiles) and for every
width, with and without the input's gradient, against float64."""
import importlib

import numpy as np
import pytest

from cases import fv  # noqa: F401

pytestmark = pytest.mark.gpu


def _bf16(torch, t):
    return t.to(torch.bfloat16).double()


def _by_parts(torch, sg, x, w1, b1, w2, dy):
    """dx, dw1, db1, dw2, db2 by the separate entry points."""
    lib, p, s = sg._lib.lib(), sg._p, sg._stream()
    (m, k), n = x.shape, w2.shape[1]
    dx, dz, h = torch.empty_like(x), *(torch.empty((m, 64), device="cuda") for _ in range(2))
    ws = torch.empty(-(-m // lib.fvdbm_nn_chunk_rows()) * 64 * max(k, n), device="cuda")
    assert lib.fvdbm_nn_mlp_backward(p(x), m, k, p(w1), p(b1), p(w2), n, p(dy), p(dx), p(dz), p(h), s) == 0
    out = [dx] + [torch.empty(d, device="cuda") for d in ((k, 64), (64,), (64, n), (n,))]
    assert lib.fvdbm_nn_wgrad(p(x), p(dz), m, k, 64, p(ws), p(out[1]), s) == 0
    assert lib.fvdbm_nn_colsum(p(dz), m, 64, p(ws), p(out[2]), s) == 0
    assert lib.fvdbm_nn_wgrad(p(h), p(dy), m, 64, n, p(ws), p(out[3]), s) == 0
    assert lib.fvdbm_nn_colsum(p(dy), m, n, p(ws), p(out[4]), s) == 0
    return out


@pytest.mark.parametrize("k,n_out", [(16, 64), (64, 64), (256, 64), (64, 16)])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 31, 32, 33, 128, 129, 2049, 65536 + 33])
@pytest.mark.parametrize("input_grad", [True, False])
def test_gradients_at_tile_edges(gpu, k, n_out, m, input_grad):
    import torch
    sg = importlib.import_module("fvdbm-jax_amd.surrogate")
    gen = torch.Generator().manual_seed(1000 * k + m)

    def rand(*s, scale=1.0):
        return scale * torch.randn(s, generator=gen)

    x, dy = rand(m, k), rand(m, n_out)
    w1, b1, w2, b2 = rand(k, 64, scale=k ** -0.5), rand(64), rand(64, n_out, scale=0.125), rand(n_out)
    dev = [t.cuda().requires_grad_(input_grad or n > 0) for n, t in enumerate((x, w1, b1, w2, b2))]
    sg.mlp2(*dev).backward(dy.cuda())

    # the separate kernels: dx bit for bit; the sums have the same terms and
    # differ by their order, m roundings of sum |term| a side at most
    parts = [t.cpu().double() for t in _by_parts(torch, sg, *(t.detach() for t in dev[:4]), dy.cuda())]

    # the same products of bf16 operands, exactly summed
    X, DY, W1, W2 = (_bf16(torch, t) for t in (x, dy, w1, w2))
    z = X @ W1 + b1.double()
    s = torch.sigmoid(z)
    h, dz = z * s, (DY @ W2.T) * (s * (1 + z * (1 - s)))
    H, DZ = _bf16(torch, h.float()), _bf16(torch, dz.float())
    # a hidden value or its gradient next to a rounding boundary may round to
    # the other side (2^-8 of itself); every sum is float32 over its terms
    e = 2.0 ** -8
    want = [DZ @ W1.T, X.T @ DZ, dz.sum(0), H.T @ DY, dy.double().sum(0)]
    size = [DZ.abs() @ W1.abs().T, X.abs().T @ DZ.abs(), dz.abs().sum(0), H.abs().T @ DY.abs(),
            dy.double().abs().sum(0)]
    for name, t, v, q, a, tol in zip(("dx", "dw1", "db1", "dw2", "db2"), dev, want, parts, size,
                                  (e, e, 2.0 ** -14, e, 2.0 ** -16)):
        if not t.requires_grad:
            assert t.grad is None
            continue
        err = (t.grad.cpu().double() - v).abs()
        assert bool((err <= tol * a + 1e-30).all()), (name, float((err / (a + 1e-30)).max()))
        order = (t.grad.cpu().double() - q).abs()
        assert bool((order <= (0 if name == "dx" else 2 * m * 2.0 ** -24) * a).all()), name


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 65, 4097])
@pytest.mark.parametrize("input_grad", [True, False])
def test_layer_is_its_parts(gpu, n, input_grad):
    """h + mlp2(aggregate(h)) in one call: forward and dh bit for bit those of
    the separate calls, weight gradients too (the same kernel)."""
    import torch
    sg = importlib.import_module("fvdbm-jax_amd.surrogate")
    rng = np.random.default_rng(n)
    deg = rng.integers(0, 9, n)
    deg[0] += 70
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    g = dict(off=off, col=rng.integers(0, n, off[-1]).astype(np.int32), n=n)
    for k in ("w", "ex", "ey", "wt", "ext", "eyt"):
        g[k] = rng.uniform(-1, 1, off[-1]).astype(np.float32)
    g = sg.graph_to_device(g)

    def rand(*s):
        return torch.tensor(0.1 * rng.standard_normal(s).astype(np.float32), device="cuda")

    host = [rand(n, 64), rand(256, 64), rand(64), rand(64, 64), rand(64)]
    dy = rand(n, 64)
    got, want = ([t.clone().requires_grad_(input_grad or k > 0) for k, t in enumerate(host)] for _ in range(2))
    y = sg.layer(got[0], g, *got[1:])
    v = want[0] + sg.mlp2(sg.aggregate(want[0], g), *want[1:])
    assert torch.equal(y, v)
    y.backward(dy)
    v.backward(dy)
    for a, b in zip(got, want):
        assert (a.grad is None and b.grad is None) or torch.equal(a.grad, b.grad)
