"""The step kernels of the built library keep their values in registers: the
code objects' own metadata report no spilled vector register. (A branch in the
FP64 equilibrium once left up to 201 spilled in the one-step kernels, which
took up to twice as long.)"""
import importlib
import struct

import msgpack

_lib = importlib.import_module("fvdbm-jax_amd._lib")
AMDGPU, NOTE_METADATA, PT_NOTE = 224, 32, 4


def _kernels(path):
    """Metadata of every kernel in the code objects embedded in a library."""
    data = open(path, "rb").read()
    at = data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == AMDGPU:
            phoff, = struct.unpack_from("<Q", data, at + 32)
            entsize, count = struct.unpack_from("<HH", data, at + 54)
            for i in range(count):
                head = at + phoff + i * entsize
                if struct.unpack_from("<I", data, head)[0] != PT_NOTE:
                    continue
                off, = struct.unpack_from("<Q", data, head + 8)
                name, desc, kind = struct.unpack_from("<III", data, at + off)
                if kind == NOTE_METADATA:
                    start = at + off + 12 + (name + 3) // 4 * 4
                    yield from msgpack.unpackb(data[start:start + desc])["amdhsa.kernels"]
        at = data.find(b"\x7fELF", at + 4)


def test_step_kernels_spill_no_vector_registers():
    steps = {k[".name"]: k[".vgpr_spill_count"] for k in _kernels(_lib.LIB_PATH)
             if any(s in k[".name"] for s in ("6k_stepI", "10k_lat_stepI", "7k_multiI"))}
    assert len(steps) >= 8 + 8 + 12, sorted(steps)
    assert not {n: s for n, s in steps.items() if s}
