"""The packed pfs_field structs of fluid._on_fields: the layout of ctypes'
struct, swapped pointers written back, errors raised.  Needs no GPU: fields
here are plain objects over CPU tensors, refused or left alone by the library."""
from __future__ import annotations

import ctypes

import pytest

torch = pytest.importorskip("torch")

from probabilistic_fluid_simulation_amd import _lib, fluid  # noqa: E402


class _Field:
    def __init__(self, *shape):
        self.data = torch.zeros(*shape)

    x = property(lambda self: self.data.shape[1])
    y = property(lambda self: self.data.shape[0])
    z = property(lambda self: self.data.shape[2])
    _struct = fluid.VPField._struct


def test_packed_layout_is_the_structs():
    fields = [_Field(3, 5, 4), _Field(7, 2, 1), _Field(1, 1, 3), _Field(9, 9, 4)]
    for n in range(1, 5):
        want = b"".join(bytes(f._struct()) for f in fields[:n])
        vals = []
        for f in fields[:n]:
            vals += f.x, f.y, f.z, f.data.data_ptr()
        buf = fluid._BUFFER[n]()
        fluid._PACK[n].pack_into(buf, 0, *vals)
        assert len(bytes(buf)) == n * ctypes.sizeof(_lib.PfsField) == len(want)
        for k in range(n):  # padding aside
            got = _lib.PfsField.from_buffer_copy(bytes(buf), k * fluid._FIELD_BYTES)
            f = fields[k]
            assert (got.x, got.y, got.z, got.data) == (f.x, f.y, f.z, f.data.data_ptr())


@pytest.mark.parametrize("by_ctypes", [False, True], ids=["packed", "ctypes"])
def test_swapped_pointers_are_written_back(monkeypatch, by_ctypes):
    fields = [_Field(4, 4, 4) for _ in range(4)]
    before = [f.data for f in fields]

    def swap(name, *args):
        s = [ctypes.cast(a, ctypes.POINTER(_lib.PfsField))[0] for a in args[:4]]
        assert [(q.x, q.y, q.z, q.data) for q in s] == [(4, 4, 4, t.data_ptr()) for t in before]
        s[2].data, s[3].data = s[3].data, s[2].data
        assert args[4:] == (0.5, 7)

    monkeypatch.setattr(_lib, "call_fields", swap)
    if by_ctypes:  # the way of sides that do not fit the packing
        class Refuses:
            def pack_into(self, *a):
                raise fluid.struct.error("too large")

            unpack_from = staticmethod(fluid._PACK[4].unpack_from)
        monkeypatch.setattr(fluid, "_PACK", [None] * 4 + [Refuses()])
    fluid._on_fields("any", fields, 0.5, 7)
    assert [f.data is t for f, t in zip(fields, [before[0], before[1], before[3], before[2]])] == [True] * 4


def test_refusals_raise_and_leave_the_fields():
    a, b = _Field(4, 4, 3), _Field(4, 4, 3)  # the step needs 4 channels
    da, db = a.data, b.data
    with pytest.raises(_lib.PfsError, match="pfs_simulate_fluid_step"):
        fluid._on_fields("pfs_simulate_fluid_step", (a, b), 0.1, 0.1, 4, 0)
    assert a.data is da and b.data is db
