// The output side of a Gated DeltaNet layer on gfx950 (MI355X, CDNA4): the
// gated RMS norm of dan/fused.py:52-56 over every (token, value head) row,
//
//   y = rnd(weight * rnd(x * rsqrt(mean(x^2) + eps))) * silu(gate)
//
// rnd() rounding to the I/O type as the eager ops do; sums, silu and the last
// product in fp32, rounded once more at the store.
//
// One pass over x and gate, bound by HBM: 8192 x 16 rows of 128 take 18.1 us
// (100.7 MB, 5.6 TB/s in repeated calls; a large copy reaches 5.0), 759 x 16 rows 3.8 us. As nine
// eager launches the chain moved about ten times these bytes: it cost the
// 8192-token layer 180 us (886 -> 707) and one mixed-type product alone took
// 73 us of the 759-token layer. A row of Dv values takes Dv / 8 lanes (16
// bytes each), so a wave reads whole rows; a lane takes two rows
// 256 / (Dv / 8) apart and loads both rows' operands before any math (what
// the front end's kernel measured best for the same shape of work).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dan_gdn.h"

// The products are rounded before the next one, as the eager ops are.
#pragma clang fp contract(off)

namespace dan {
int fail(int status, const char *fmt, ...);  // tree_attn.hip: sets the thread's last-error message
bool finite_nonnegative(float x);             // tree_attn.hip: decided from the float's bits
extern thread_local char g_err[512];
}  // namespace dan

namespace dan_gnorm {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define DAN_GLOBAL __attribute__((address_space(1)))

template <typename T>
struct V;
template <>
struct V<__bf16> {
  typedef bf16x8 x8;
};
template <>
struct V<_Float16> {
  typedef f16x8 x8;
};

template <typename T>
__device__ inline f32x8 to_f32(u32x4 raw) {
  return __builtin_convertvector(__builtin_bit_cast(typename V<T>::x8, raw), f32x8);
}
template <typename T>
__device__ inline u32x4 from_f32(f32x8 x) {
  return __builtin_bit_cast(u32x4, __builtin_convertvector(x, typename V<T>::x8));
}
template <typename T>
__device__ inline f32x8 rnd(f32x8 x) {
  return to_f32<T>(from_f32<T>(x));
}

// Sum of v over the L consecutive lanes of a row (L = 4, 8, 16 or 32), in every
// one of them: DPP quad swaps and mirrors, one cross-row shuffle at L = 32.
#define DAN_DPP(x, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), ctrl, 0xF, 0xF, false))
template <int L>
__device__ inline float row_sum(float v) {
  v += DAN_DPP(v, 0xB1);   // quad_perm 1, 0, 3, 2
  v += DAN_DPP(v, 0x4E);   // quad_perm 2, 3, 0, 1
  if constexpr (L >= 8) v += DAN_DPP(v, 0x141);   // row_half_mirror
  if constexpr (L >= 16) v += DAN_DPP(v, 0x140);  // row_mirror
  if constexpr (L >= 32) v += __shfl_xor(v, 16, 32);
  return v;
}

// silu(g) = g / (1 + exp(-g)) to about three fp32 ulps for |g| < 87: exp(-g) as 2^p,
// p = -g log2(e) rounded, times 1 + (what the rounding of p and of log2(e) left) ln 2,
// without which up to 44 ulps are lost. Within 87, 1 + exp(-g) and its reciprocal are normal.
// 8192 x 16 rows of 128, microseconds: 18.1; 17.1 with the bare exp2 of the rounded product,
// 19.3 with silu_any and a Newton step on every gate, 22.4 with expf and a division.
__device__ inline float silu_near(float g) {
  const float p = g * -1.4426950408889634f;
  const float left = __builtin_fmaf(g, -1.925963033500011e-08f, __builtin_fmaf(g, -1.4426950216293335f, -p));
  const float e = __builtin_amdgcn_exp2f(p);
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_fmaf(e, left * 0.6931471805599453f, e));
}
// The same for every g, from e = exp(-|g|) = 2^n 2^f: 1 + e lies in [1, 2], and 2^n is
// applied to g 2^f, since e alone is subnormal from g = -87.4 on (the hardware exp2
// and reciprocal flush there: -88 came out as 0, and silu(-88) is a normal bf16).
__device__ inline float silu_any(float g) {
  const float a = fabsf(g);
  const float n = fmaxf(__builtin_rintf(a * -1.4426950408889634f), -300.0f);  // finite: -inf leaves f = -inf, m = 0 and NaN
  const float f = __builtin_fmaf(a, -1.925963033500011e-08f, __builtin_fmaf(a, -1.4426950216293335f, -n));
  const float m = __builtin_amdgcn_exp2f(f);
  const int k = (int)n;
  return (g >= 0.0f ? g : __builtin_ldexpf(g * m, k)) * __builtin_amdgcn_rcpf(1.0f + __builtin_ldexpf(m, k));
}
// Whether every one of a lane's eight gates lies within (-87, 87): their bits without
// the sign, largest first (a NaN's are the largest).
template <typename T>
__device__ inline bool all_near(u32x4 raw) {
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  const u16x8 x = __builtin_bit_cast(u16x8, raw) & (uint16_t)0x7fff;
  const u16x4 x4 = __builtin_elementwise_max(x.lo, x.hi);
  const u16x2 x2 = __builtin_elementwise_max(x4.lo, x4.hi);
  return max(x2[0], x2[1]) < __builtin_bit_cast(uint16_t, (T)87.0f);
}

struct Params {
  const void *x, *gate, *weight;
  void *out;
  int64_t x_st, g_st, o_st;
  int32_t N, H;
  float eps;
};

constexpr int kVecs = 2;

template <typename T, int D>
__global__ __launch_bounds__(256) void gated_norm_kernel(const Params p) {
  constexpr int L = D / 8, VPB = 256 / L;
  const int slot = threadIdx.x / L, j = threadIdx.x % L;
  const int64_t rows = (int64_t)p.N * p.H, v0 = (int64_t)blockIdx.x * (kVecs * VPB) + slot;
  if (v0 >= rows) return;  // whole rows leave together: the lane exchanges stay inside live rows
  const f32x8 w = to_f32<T>(*(const DAN_GLOBAL u32x4 *)(static_cast<const T *>(p.weight) + 8 * j));
  u32x4 xr[kVecs], gr[kVecs];
  T *dst[kVecs];
  bool ok[kVecs];
#pragma unroll
  for (int k = 0; k < kVecs; ++k) {
    const int64_t v = v0 + k * VPB;
    ok[k] = v < rows;
    const int64_t vc = ok[k] ? v : rows - 1;  // a row past the end is computed on the last one and not stored
    const int64_t n = vc / p.H, col = vc % p.H * D + 8 * j;
    xr[k] = *(const DAN_GLOBAL u32x4 *)(static_cast<const T *>(p.x) + n * p.x_st + col);
    gr[k] = *(const DAN_GLOBAL u32x4 *)(static_cast<const T *>(p.gate) + n * p.g_st + col);
    dst[k] = static_cast<T *>(p.out) + n * p.o_st + col;
  }
#pragma unroll
  for (int k = 0; k < kVecs; ++k) {
    const f32x8 x = to_f32<T>(xr[k]), g = to_f32<T>(gr[k]);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(x[i], x[i], ss);
    const float r = rsqrtf(row_sum<L>(ss) * (1.0f / (float)D) + p.eps);
    const f32x8 n = rnd<T>(w * rnd<T>(x * r));
    f32x8 y;
    if (__all(all_near<T>(gr[k]))) {
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = n[i] * silu_near(g[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = n[i] * silu_any(g[i]);
    }
    if (ok[k]) *(DAN_GLOBAL u32x4 *)dst[k] = from_f32<T>(y);
  }
}

template <typename T, int D>
void launch(const Params &p, hipStream_t s) {
  constexpr int VPB = kVecs * (256 / (D / 8));
  const int64_t rows = (int64_t)p.N * p.H;
  hipLaunchKernelGGL((gated_norm_kernel<T, D>), dim3((unsigned)((rows + VPB - 1) / VPB)), dim3(256), 0, s, p);
}

template <typename T>
void by_dim(const Params &p, int d, hipStream_t s) {
  if (d == 32) launch<T, 32>(p, s);
  else if (d == 64) launch<T, 64>(p, s);
  else if (d == 128) launch<T, 128>(p, s);
  else launch<T, 256>(p, s);
}

}  // namespace dan_gnorm

extern "C" int dan_gdn_gated_norm(const DanGdnNormArgs *a, void *stream) {
  using dan::fail;
  dan::g_err[0] = 0;
  if (!a) return fail(DAN_ERR_INVALID_ARGUMENT, "args is NULL");
  if (a->abi_version != DAN_GDN_ABI_VERSION)
    return fail(DAN_ERR_VERSION, "abi_version %d, delta rule speaks %d", a->abi_version, DAN_GDN_ABI_VERSION);
  if (a->dtype != DAN_DTYPE_BF16 && a->dtype != DAN_DTYPE_F16) return fail(DAN_ERR_UNSUPPORTED, "dtype %d: bf16 or f16", a->dtype);
  const int d = a->v_dim;
  if (d != 32 && d != 64 && d != 128 && d != 256) return fail(DAN_ERR_UNSUPPORTED, "v_dim %d: 32, 64, 128 or 256", d);
  if (a->num_tokens < 0 || a->num_v_heads <= 0) return fail(DAN_ERR_INVALID_ARGUMENT, "need num_tokens >= 0 and num_v_heads > 0");
  if (!dan::finite_nonnegative(a->eps)) return fail(DAN_ERR_INVALID_ARGUMENT, "eps must be finite and >= 0");
  if (a->num_tokens == 0) return DAN_OK;
  if (!a->x || !a->gate || !a->weight || !a->out) return fail(DAN_ERR_INVALID_ARGUMENT, "NULL pointer");
  const int64_t row = (int64_t)a->num_v_heads * d;
  for (int64_t st : {a->x_stride, a->gate_stride, a->out_stride})
    if (st < row || st % 8) return fail(DAN_ERR_INVALID_ARGUMENT, "token strides must hold the heads and be multiples of 8");
  for (const void *ptr : {a->x, a->gate, a->weight, (const void *)a->out})
    if ((uintptr_t)ptr & 15) return fail(DAN_ERR_INVALID_ARGUMENT, "x, gate, weight and out must be 16-byte aligned");
  if ((int64_t)a->num_tokens * a->num_v_heads > 0x7fffffffLL * 16) return fail(DAN_ERR_INVALID_ARGUMENT, "too many rows");
  dan_gnorm::Params p;
  p.x = a->x; p.gate = a->gate; p.weight = a->weight; p.out = a->out;
  p.x_st = a->x_stride; p.g_st = a->gate_stride; p.o_st = a->out_stride;
  p.N = a->num_tokens; p.H = a->num_v_heads; p.eps = a->eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == DAN_DTYPE_BF16) dan_gnorm::by_dim<__bf16>(p, d, s);
  else dan_gnorm::by_dim<_Float16>(p, d, s);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(DAN_ERR_LAUNCH, "gated norm launch failed: %s", hipGetErrorString(err));
  return DAN_OK;
}
