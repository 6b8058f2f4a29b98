"""The message-passing layer refuses blocks of other widths than its kernels'
before anything is launched: they read w2 and b2 as 64 wide whatever is passed."""
import importlib

import pytest

torch = pytest.importorskip("torch")
sg = importlib.import_module("fvdbm-jax_amd.surrogate")

GOOD = dict(h=(5, 64), w1=(256, 64), b1=(64,), w2=(64, 64), b2=(64,))


@pytest.mark.parametrize("name,shape", [
    ("w2", (64, 16)), ("b2", (16,)), ("w1", (64, 64)), ("w1", (256, 32)), ("b1", (16,)),
    ("h", (5, 16)), ("h", (64,)), ("w2", (64, 128)),
])
def test_layer_refuses_other_widths(name, shape, monkeypatch):
    def no_library():
        raise AssertionError("the library was reached")
    monkeypatch.setattr(sg._lib, "lib", no_library)
    t = {k: torch.zeros(s) for k, s in dict(GOOD, **{name: shape}).items()}
    with pytest.raises(RuntimeError, match="unsupported"):
        sg.layer(t["h"], {}, t["w1"], t["b1"], t["w2"], t["b2"])
