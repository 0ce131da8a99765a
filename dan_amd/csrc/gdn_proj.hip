// The two narrow projections of a Gated DeltaNet layer on gfx950 (MI355X,
// CDNA4): b = x Wb^T and a = x Wa^T (dan/models/qwen3_5.py:186-189), one value
// head a column, rounded once from fp32 sums.
//
// Bound by the CU's address unit: a load covers 16 rows, 64 bytes of each, and
// takes about 43 cycles. 834 rows of 2048 take 7.2 us for 16 columns each and 8192
// rows 9.7; as two library products they took 10.5 and 16.7, and the host 2 x 20 us
// where one call takes 3. A work group takes whole 16-column tiles of both
// matrices; its 8 waves split the hidden dimension (128 bytes of every row at a
// time, so that a row's lines are read whole) and add their partial sums in LDS,
// in the waves' order. With one wave a row block, 834 rows would be 53 waves on
// 1024 SIMDs, each with a chain of 64 products. 64 rows or 32 columns a group:
// 13 and 10 us for 834 rows, 13.6 and 11.2 for 8192.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cus.h"
#include "dan_gdn.h"

namespace dan {
int fail(int status, const char *fmt, ...);  // tree_attn.hip: sets the thread's last-error message
extern thread_local char g_err[512];
}  // namespace dan

namespace dan_gproj {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

#define DAN_GLOBAL __attribute__((address_space(1)))

constexpr int kWaves = 8;
constexpr int kStep = 32, kPair = 2;  // hidden values a product; products of one 128-byte line
constexpr int kAhead = 4;             // lines of a row a wave has in flight

template <typename T>
struct V;
template <>
struct V<__bf16> {
  typedef bf16x4 x4;
  static __device__ inline f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <>
struct V<_Float16> {
  typedef f16x4 x4;
  static __device__ inline f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

struct Params {
  const void *x, *w0, *w1;
  void *y0, *y1;
  int64_t x_st, w0_st, w1_st, y0_st, y1_st;
  int32_t M, N, K;
};

// A work group: 16 RB rows of x, 16 columns of w0 and of w1. Lane l16 + 16 g4
// loads row l16 of a 16-row block, hidden values 8 g4 .. + 7 of a product; it ends
// with columns 4 g4 .. + 3 of x's row l16.
template <typename T, int RB>
__global__ __launch_bounds__(64 * kWaves) void proj_kernel(const Params p) {
  constexpr int kTiles = 2 * RB;  // (rows, matrix)
  __shared__ __attribute__((aligned(16))) float part[kWaves][kTiles][64][4];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = 16 * RB * (int)blockIdx.x, col0 = 16 * (int)blockIdx.y, n = min(col0 + l16, p.N - 1);
  const T *x[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) x[r] = static_cast<const T *>(p.x) + min(row0 + 16 * r + l16, p.M - 1) * p.x_st + 8 * g4;
  const T *w[2] = {static_cast<const T *>(p.w0) + n * p.w0_st + 8 * g4, static_cast<const T *>(p.w1) + n * p.w1_st + 8 * g4};
  const int steps = p.K / kStep;
  f32x4 acc[RB][2] = {};
  for (int s0 = kPair * wave; s0 < steps; s0 += kPair * kWaves * kAhead) {
    u32x4 xv[kAhead][kPair][RB] = {}, wv[kAhead][kPair][2] = {};
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
#pragma unroll
      for (int j = 0; j < kPair; ++j) {
        const int s = s0 + kPair * kWaves * i + j;
        if (s >= steps) continue;  // the same for the wave; its products add zero
#pragma unroll
        for (int r = 0; r < RB; ++r) xv[i][j][r] = *(const DAN_GLOBAL u32x4 *)(x[r] + kStep * s);
#pragma unroll
        for (int c = 0; c < 2; ++c) wv[i][j][c] = *(const DAN_GLOBAL u32x4 *)(w[c] + kStep * s);
      }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
#pragma unroll
      for (int j = 0; j < kPair; ++j)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[r][c] = V<T>::mma(wv[i][j][c], xv[i][j][r], acc[r][c]);
  }
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) *reinterpret_cast<f32x4 *>(part[wave][r * 2 + c][lane]) = acc[r][c];
  __syncthreads();
  for (int t = wave; t < kTiles; t += kWaves) {  // a wave adds up and stores whole tiles
    const int r = t / 2, c = t % 2;
    f32x4 sum = *reinterpret_cast<const f32x4 *>(part[0][t][lane]);
#pragma unroll
    for (int v = 1; v < kWaves; ++v) sum += *reinterpret_cast<const f32x4 *>(part[v][t][lane]);
    const int row = row0 + 16 * r + l16, col = col0 + 4 * g4;
    if (row >= p.M || col >= p.N) continue;
    T *y = c == 0 ? static_cast<T *>(p.y0) + row * p.y0_st : static_cast<T *>(p.y1) + row * p.y1_st;
    *(DAN_GLOBAL typename V<T>::x4 *)(y + col) = __builtin_convertvector(sum, typename V<T>::x4);
  }
}

template <typename T, int RB>
void launch(const Params &p, hipStream_t s) {
  const dim3 grid((unsigned)(((int64_t)p.M + 16 * RB - 1) / (16 * RB)), (unsigned)((p.N + 15) / 16));
  hipLaunchKernelGGL((proj_kernel<T, RB>), grid, dim3(64 * kWaves), 0, s, p);
}

template <typename T>
void run(const Params &p, hipStream_t s) {
  if (dan::project_rows(p.M, p.N, dan::num_cus()) == 16) launch<T, 1>(p, s);
  else launch<T, 2>(p, s);
}

}  // namespace dan_gproj

extern "C" int dan_gdn_project(const DanGdnProjArgs *a, void *stream) {
  using dan::fail;
  dan::g_err[0] = 0;
  if (!a) return fail(DAN_ERR_INVALID_ARGUMENT, "args is NULL");
  if (a->abi_version != DAN_GDN_ABI_VERSION)
    return fail(DAN_ERR_VERSION, "abi_version %d, delta rule speaks %d", a->abi_version, DAN_GDN_ABI_VERSION);
  if (a->dtype != DAN_DTYPE_BF16 && a->dtype != DAN_DTYPE_F16) return fail(DAN_ERR_UNSUPPORTED, "dtype %d: bf16 or f16", a->dtype);
  if (a->rows < 0 || a->cols <= 0 || a->hidden <= 0) return fail(DAN_ERR_INVALID_ARGUMENT, "need rows >= 0, cols > 0 and hidden > 0");
  if (a->cols % 4 || a->hidden % dan_gproj::kStep) return fail(DAN_ERR_UNSUPPORTED, "cols must be a multiple of 4, hidden of %d", dan_gproj::kStep);
  if (a->cols > 16 * 65535) return fail(DAN_ERR_UNSUPPORTED, "too many columns");
  if (a->rows == 0) return DAN_OK;
  if (!a->x || !a->w0 || !a->w1 || !a->y0 || !a->y1) return fail(DAN_ERR_INVALID_ARGUMENT, "NULL pointer");
  for (int64_t st : {a->x_stride, a->w0_stride, a->w1_stride})
    if (st < a->hidden || st % 8) return fail(DAN_ERR_INVALID_ARGUMENT, "row strides of x, w0 and w1 must hold a row and be multiples of 8");
  for (int64_t st : {a->y0_stride, a->y1_stride})
    if (st < a->cols || st % 4) return fail(DAN_ERR_INVALID_ARGUMENT, "row strides of y0 and y1 must hold a row and be multiples of 4");
  for (const void *ptr : {a->x, a->w0, a->w1})
    if ((uintptr_t)ptr & 15) return fail(DAN_ERR_INVALID_ARGUMENT, "x, w0 and w1 must be 16-byte aligned");
  for (const void *ptr : {(const void *)a->y0, (const void *)a->y1})
    if ((uintptr_t)ptr & 7) return fail(DAN_ERR_INVALID_ARGUMENT, "y0 and y1 must be 8-byte aligned");
  dan_gproj::Params p;
  p.x = a->x; p.w0 = a->w0; p.w1 = a->w1; p.y0 = a->y0; p.y1 = a->y1;
  p.x_st = a->x_stride; p.w0_st = a->w0_stride; p.w1_st = a->w1_stride; p.y0_st = a->y0_stride; p.y1_st = a->y1_stride;
  p.M = a->rows; p.N = a->cols; p.K = a->hidden;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == DAN_DTYPE_BF16) dan_gproj::run<__bf16>(p, s);
  else dan_gproj::run<_Float16>(p, s);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(DAN_ERR_LAUNCH, "projection launch failed: %s", hipGetErrorString(err));
  return DAN_OK;
}
