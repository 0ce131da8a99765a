"""dan_gdn_gated_norm's C ABI without a GPU: the ctypes mirror has the
header's layout, and argument errors come back before any launch."""
import ctypes
import os
import subprocess

import pytest

from dan_amd import _native
from test_abi import GDN_HEADER, lib  # noqa: F401  -- the library fixture


def test_struct_layout(tmp_path):
    cls = _native.DanGdnNormArgs
    src, exe = tmp_path / "p.c", tmp_path / "p"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "dan_gdn.h"\nint main(void) {\n'
                   + 'printf("%zu\\n", sizeof(DanGdnNormArgs));\n'
                   + "".join(f'printf("%zu\\n", offsetof(DanGdnNormArgs, {f}));\n' for f, _ in cls._fields_) + "return 0; }\n")
    subprocess.run(["gcc", "-std=c99", "-I", os.path.dirname(GDN_HEADER), str(src), "-o", str(exe)], check=True)
    got = [int(x) for x in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]
    assert got == [ctypes.sizeof(cls)] + [getattr(cls, f).offset for f, _ in cls._fields_]


@pytest.mark.parametrize("kw,status,needle", [
    (dict(abi_version=1), _native.ERR_VERSION, "abi_version"), (dict(dtype=_native.DTYPE_F32), _native.ERR_UNSUPPORTED, "dtype"),
    (dict(v_dim=96), _native.ERR_UNSUPPORTED, "v_dim"), (dict(eps=float("nan")), _native.ERR_INVALID_ARGUMENT, "eps"),
    (dict(gate_stride=250), _native.ERR_INVALID_ARGUMENT, "strides"), (dict(out_stride=260), _native.ERR_INVALID_ARGUMENT, "strides"),
    (dict(x=4098), _native.ERR_INVALID_ARGUMENT, "aligned"), (dict(weight=None), _native.ERR_INVALID_ARGUMENT, "NULL"),
    (dict(num_tokens=-1), _native.ERR_INVALID_ARGUMENT, "num_tokens"), (dict(num_tokens=0, x=None), _native.OK, "")])
def test_argument_errors(lib, kw, status, needle):  # noqa: F811
    a = _native.DanGdnNormArgs()
    base = dict(abi_version=_native.GDN_ABI_VERSION, dtype=_native.DTYPE_BF16, num_tokens=3, num_v_heads=2, v_dim=128, eps=1e-6,
                x=4096, gate=4096, weight=4096, out=4096, x_stride=256, gate_stride=256, out_stride=256)
    for k, v in {**base, **kw}.items():
        setattr(a, k, v)
    assert lib.dan_gdn_gated_norm(ctypes.byref(a), None) == status
    assert needle in _native.last_error(lib)
