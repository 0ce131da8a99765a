"""The packed argument buffers of the C entry points: byte for byte the ctypes
structure's, and refused (not raised as another error) beyond a field's range."""
import ctypes

import pytest

from dan_amd import _native

ENTRIES = [(_native.call_forward, _native.DanTreeAttnArgs), (_native.call_forward_noalloc, _native.DanTreeAttnArgs),
           (_native.call_front, _native.DanQkvFrontArgs), (_native.call_fp8_quantize, _native.DanFp8QuantArgs),
           (_native.call_fp8_gemm, _native.DanFp8GemmArgs), (_native.call_gdn, _native.DanGdnArgs),
           (_native.call_gdn_conv, _native.DanGdnConvArgs), (_native.call_gdn_gated_norm, _native.DanGdnNormArgs),
           (_native.call_gdn_project, _native.DanGdnProjArgs)]


def test_every_entry_is_listed():
    assert {e.name for e, _ in ENTRIES} == {e.name for e in vars(_native).values() if isinstance(e, _native.Entry)}


@pytest.mark.parametrize("entry,args", ENTRIES, ids=[e.name for e, _ in ENTRIES])
def test_fields_lie_where_the_structure_has_them(entry, args):
    values = [{ctypes.c_int32: -7 - i, ctypes.c_int64: -(1 << 40) - i, ctypes.c_float: 0.5 + i,
               ctypes.c_void_p: (1 << 46) + 16 * i}[t] for i, (_, t) in enumerate(args._fields_)]
    packed, filled = args.from_buffer_copy(entry.pack(*values)), args(*values)
    assert [getattr(packed, n) for n, _ in args._fields_] == [getattr(filled, n) for n, _ in args._fields_] == values
    null = [0] * len(values)
    assert entry.pack(*null) == bytes(args())


def test_a_call_reaches_the_library_and_its_refusals():
    fields = [0] * len(_native.DanFp8QuantArgs._fields_)
    with pytest.raises(RuntimeError, match="dan_fp8_quantize failed"):  # ABI version 0
        _native.call_fp8_quantize(0, *fields)
    fields[2] = 2 ** 31  # rows past the field's range
    with pytest.raises(RuntimeError, match="dan_fp8_quantize failed"):
        _native.call_fp8_quantize(0, *fields)


def test_floats_are_rounded_as_a_c_field():
    for x in (1e-6, 1e40, -1e40, 0.1, float("inf")):
        assert _native.f32(x) == ctypes.c_float(x).value
