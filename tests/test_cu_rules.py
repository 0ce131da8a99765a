"""The DeltaNet kernels' choices by the device's compute units (csrc/cus.h),
compiled for the host: the state columns of the bf16 scan (16 while two work
groups per CU hold every one) and the rows of the narrow projections (16 while
there is at most one work group per CU), on a whole device and on partitions."""
import os
import subprocess

from dan_amd import _build

CASES = [(cus, n) for cus in (256, 128, 64, 32) for n in (1, cus // 64, cus // 64 + 1, cus // 8, cus)]


def test_rules_follow_the_compute_units(tmp_path):
    src = tmp_path / "rules.cpp"
    calls = "".join(f'printf("%d %d\\n", dan::scan_columns({n}, 16, 128, {cus}), dan::project_rows(16 * {n}, 16, {cus}));' for cus, n in CASES)
    src.write_text('#include <stdio.h>\n#include "cus.h"\nint main() { ' + calls + " }")
    exe = tmp_path / "rules"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(_build.HERE, "csrc"), str(src), "-o", str(exe)], check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()
    want = [f"{16 if n * 16 * 8 <= 2 * cus else 32} {16 if n <= cus else 32}" for cus, n in CASES]
    assert got == want
    kernels = [open(os.path.join(_build.HERE, "csrc", f)).read() for f in ("gdn_chunk.hip", "gdn_proj.hip")]
    assert "dan::scan_columns(" in kernels[0] and "dan::project_rows(" in kernels[1]
