// What the DeltaNet kernels choose by the device's compute units (host code).
#pragma once
#include <stdint.h>

namespace dan {

int num_cus();  // fp8_gemm.hip: compute units of the current device (0: unknown)

// State columns per work group of the bf16 scan (gdn_chunk.hip): 16 while all
// groups are resident at once, two per CU, else 32. A chunk's step of 16 columns is the
// shorter, so the longest run ends sooner, but the groups' total work is more.
// The whole rule (16 value heads of 128 columns, 256 CUs), microseconds at 16 / 32 columns:
// 1 run of 1462 tokens (128 groups) 55.4 / 71.4, 2000 + 300 + 900 (384) 82.9 / 99.8,
// 3 of 1500 87.8 / 87.0, 4 of 1000 (512) 63.6 / 63.1; past that it depends on how
// unequal the runs are: 5 of 286-1843 (640) 92 / 108, but 5 of 1000 91 / 80, 6 of
// 400-1900 116 / 111, 8 of 800 95 / 79, 45 branches of 16-96 77 / 62.
inline int scan_columns(int64_t runs, int64_t v_heads, int64_t v_dim, int cus) {
  return runs * v_heads * (v_dim / 16) <= 2 * (int64_t)cus ? 16 : 32;
}

// Rows of x per work group of the narrow projections (gdn_proj.hip): 16 while
// that is at most one group per CU, else 32. 2048 hidden values, 256 CUs, 16 / 32 rows,
// microseconds: 834 x 16 7.2 / 9.0 and 2779 x 16 7.4 / 9.1, but 8192 x 16 12.8 / 9.7
// and 2779 x 32 12.7 / 9.6.
inline int project_rows(int64_t rows, int64_t cols, int cus) {
  return (rows + 15) / 16 * ((cols + 15) / 16) <= cus ? 16 : 32;
}

}  // namespace dan
