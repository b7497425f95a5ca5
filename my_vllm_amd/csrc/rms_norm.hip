// RMSNorm and fused residual-add RMSNorm for gfx950.
//
// Semantics follow the reference's native path (nanovllm/layers/layernorm.py:
// 31-52, the compiled torch restatement its CUDA providers must match):
//   rms_norm:      x32 = float(x); y = T(T(x32 * rsqrt(mean(x32^2) + eps)) * w)
//   add_rms_norm:  s32 = float(x) + float(residual); residual_out = T(s32);
//                  y = T(T(s32 * rsqrt(mean(s32^2) + eps)) * w)
// i.e. the statistics use the fp32 sum (not the rounded residual), the scaled
// row is rounded to the storage type T before the weight multiply, and the
// product is rounded again (torch multiplies two T tensors in fp32 and rounds
// once).  `w` is T or fp32.
//
// HBM-bound: each lane keeps its 16-byte chunks of a row in registers between
// the sum of squares and the output, so a row is read once and written once,
// and an in-place call (out == x, residual_out == residual) is safe: every
// element is read before any element of its row is written.
#include "mva_capi.h"
#include "mva_common.h"

#include <algorithm>

namespace mva {
namespace {

// Row r of a call is row (r % rows_per_group) of group (r / rows_per_group):
// x + (r / rows_per_group) * x_group_stride + (r % rows_per_group) * x_stride
// (likewise for out; the fused form uses one group per row).
struct RmsArgs {
  const void* x;
  int64_t x_stride;  // elements between rows of a group
  const void* residual;  // nullptr: plain RMSNorm
  int64_t res_stride;
  const void* weight;
  void* out;
  int64_t out_stride;
  void* residual_out;
  int64_t res_out_stride;
  int64_t rows;
  int hidden;
  float eps;
  int64_t rows_per_group;
  int64_t x_group_stride;
  int64_t out_group_stride;
  int64_t first_row;  // of this launch (launch_rows)
};

// Rows and rows per group below 2^31 (the usual case) divide in 32 bits: a
// 64-bit division is about a hundred instructions at the start of every row.
__device__ inline int64_t row_offset(int64_t r, int64_t per_group, int64_t group_stride, int64_t stride) {
  const bool narrow = ((uint64_t)r | (uint64_t)per_group) >> 31 == 0;
  const int64_t g = narrow ? (int64_t)((uint32_t)r / (uint32_t)per_group) : r / per_group;
  return g * group_stride + (r - g * per_group) * stride;
}

__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

template <typename W>
__device__ inline void load_w8(const W* w, float (&f)[8]);
template <>
__device__ inline void load_w8<float>(const float* w, float (&f)[8]) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(w);
  const f32x4 b = *reinterpret_cast<const f32x4*>(w + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = a[i];
    f[4 + i] = b[i];
  }
}
template <>
__device__ inline void load_w8<__bf16>(const __bf16* w, float (&f)[8]) {
  const bf16x8 a = *reinterpret_cast<const bf16x8*>(w);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = (float)a[i];
}
template <>
__device__ inline void load_w8<_Float16>(const _Float16* w, float (&f)[8]) {
  const f16x8 a = *reinterpret_cast<const f16x8*>(w);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = (float)a[i];
}

// Vector path: hidden % 8 == 0, 16-byte aligned rows, hidden <= 512 * kWaves *
// kChunks (at most 8192: larger rows take the scalar path).  kWaves 1: four
// rows per workgroup, a wavefront each.  kWaves > 1: a workgroup of kWaves
// wavefronts per row, whose partial sums meet in LDS.  The row, the residual
// and the weight are all requested before the sum, one memory round trip.
template <typename T, typename W, int kWaves, int kChunks, bool kAdd>
__global__ __launch_bounds__(kWaves == 1 ? 256 : 64 * kWaves) void rms_norm_vec_kernel(RmsArgs a) {
  typedef typename Elem<T>::v8 V;
  __shared__ float part[kWaves];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t row = a.first_row + (kWaves == 1 ? (int64_t)blockIdx.x * 4 + w : (int64_t)blockIdx.x);
  if (row >= a.rows) return;
  const int j0 = kWaves == 1 ? lane : (int)threadIdx.x;
  const int nvec = a.hidden >> 3;
  const T* xr = (const T*)a.x +
                (kAdd ? row * a.x_stride : row_offset(row, a.rows_per_group, a.x_group_stride, a.x_stride));
  const T* rr = kAdd ? (const T*)a.residual + row * a.res_stride : nullptr;
  const W* wp = (const W*)a.weight;
  V xv[kChunks], rv[kChunks];
  float wf[kChunks][8];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int j = j0 + 64 * kWaves * c;
    if (j < nvec) {
      xv[c] = *reinterpret_cast<const V*>(xr + 8 * j);
      if constexpr (kAdd) rv[c] = *reinterpret_cast<const V*>(rr + 8 * j);
      load_w8<W>(wp + 8 * j, wf[c]);
    }
  }
  float v[kChunks][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    if (j0 + 64 * kWaves * c < nvec) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f = (float)xv[c][i];
        if constexpr (kAdd) f += (float)rv[c][i];
        v[c][i] = f;
        ss += f * f;
      }
    }
  }
  ss = wave_sum(ss);
  if constexpr (kWaves > 1) {
    if (lane == 0) part[w] = ss;
    __syncthreads();
    ss = part[0];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) ss += part[k];
  }
  const float r = 1.0f / __builtin_sqrtf(ss / (float)a.hidden + a.eps);
  T* orow = (T*)a.out +
            (kAdd ? row * a.out_stride : row_offset(row, a.rows_per_group, a.out_group_stride, a.out_stride));
  T* ro = kAdd ? (T*)a.residual_out + row * a.res_out_stride : nullptr;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int j = j0 + 64 * kWaves * c;
    if (j < nvec) {
      V o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (T)((float)(T)(v[c][i] * r) * wf[c][i]);
      if constexpr (kAdd) {
        V s;
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = (T)v[c][i];
        __builtin_nontemporal_store(s, reinterpret_cast<V*>(ro + 8 * j));
      }
      __builtin_nontemporal_store(o, reinterpret_cast<V*>(orow + 8 * j));
    }
  }
}

// Any width and alignment: two passes over the row per wavefront (the first
// only reads), so in-place calls stay correct.
template <typename T, typename W, bool kAdd>
__global__ __launch_bounds__(256) void rms_norm_scalar_kernel(RmsArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = a.first_row + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.rows) return;
  const T* xr = (const T*)a.x + row_offset(row, a.rows_per_group, a.x_group_stride, a.x_stride);
  const T* rr = kAdd ? (const T*)a.residual + row * a.res_stride : nullptr;
  float ss = 0.f;
  for (int i = lane; i < a.hidden; i += 64) {
    float f = (float)xr[i];
    if constexpr (kAdd) f += (float)rr[i];
    ss += f * f;
  }
  ss = wave_sum(ss);
  const float r = 1.0f / __builtin_sqrtf(ss / (float)a.hidden + a.eps);
  T* orow = (T*)a.out + row_offset(row, a.rows_per_group, a.out_group_stride, a.out_stride);
  T* ro = kAdd ? (T*)a.residual_out + row * a.res_out_stride : nullptr;
  const W* w = (const W*)a.weight;
  for (int i = lane; i < a.hidden; i += 64) {
    float f = (float)xr[i];
    if constexpr (kAdd) f += (float)rr[i];
    const T y = (T)((float)(T)(f * r) * (float)w[i]);
    if constexpr (kAdd) ro[i] = (T)f;
    orow[i] = y;
  }
}

// A launch of 2^32 threads or more runs some of its rows only (and reports
// nothing), so more rows than that (8.4 million at 512 threads a row) take
// several.
void launch_rows(void (*kernel)(RmsArgs), RmsArgs a, int rows_per_block, int threads, hipStream_t s) {
  const int64_t most = 0xffffffffLL / threads * rows_per_block;
  for (a.first_row = 0; a.first_row < a.rows; a.first_row += most) {
    const int64_t rows = std::min(most, a.rows - a.first_row);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((rows + rows_per_block - 1) / rows_per_block)), dim3(threads), 0, s, a);
  }
}

template <typename T, typename W, bool kAdd, int kWaves, int kChunks>
void launch_vec(const RmsArgs& a, hipStream_t s) {
  launch_rows(rms_norm_vec_kernel<T, W, kWaves, kChunks, kAdd>, a, kWaves == 1 ? 4 : 1, kWaves == 1 ? 256 : 64 * kWaves,
              s);
}

template <typename T, typename W, bool kAdd>
int launch_rms(const RmsArgs& a, hipStream_t s) {
  if ((a.rows + 3) / 4 > 0x7fffffffLL) return set_error("rms_norm: too many rows");
  uint64_t bits = (uint64_t)(uintptr_t)a.x | (uint64_t)(uintptr_t)a.out | (uint64_t)(uintptr_t)a.weight |
                  (uint64_t)(a.x_stride * (int64_t)sizeof(T)) | (uint64_t)(a.out_stride * (int64_t)sizeof(T)) |
                  (uint64_t)(a.x_group_stride * (int64_t)sizeof(T)) |
                  (uint64_t)(a.out_group_stride * (int64_t)sizeof(T));
  if (kAdd)
    bits |= (uint64_t)(uintptr_t)a.residual | (uint64_t)(uintptr_t)a.residual_out |
            (uint64_t)(a.res_stride * (int64_t)sizeof(T)) | (uint64_t)(a.res_out_stride * (int64_t)sizeof(T));
  const int nvec = a.hidden / 8;
  if (a.hidden % 8 == 0 && bits % 16 == 0 && nvec <= 64 * 16) {
    // One 16-byte chunk a lane up to 8 wavefronts a row, two beyond.  One
    // wavefront a row with 8 chunks a lane (hidden 4096) left 61 rows on 16 CUs
    // (6.2 us a launch) and read and wrote 4096 rows in two separate bursts (33 us):
    // see pick_prologue_kernel for a layer's launches.  Non-temporal stores: 110.4
    // against 120.9 us for those of 4000 tokens, where nothing reads them.  The
    // reader pays that back: norm of 4099 x 4096 20.7 / 22.1 us, with the GEMM
    // (4096 x 6144) on its output 203.8 / 201.9; 2048 rows 100.8 / 101.3; norm,
    // GEMM, prologue, copy, norm and GEMM of 4099 446.0 / 446.8.
    if (nvec <= 64) launch_vec<T, W, kAdd, 1, 1>(a, s);
    else if (nvec <= 128) launch_vec<T, W, kAdd, 2, 1>(a, s);
    else if (nvec <= 256) launch_vec<T, W, kAdd, 4, 1>(a, s);
    else if (nvec <= 512) launch_vec<T, W, kAdd, 8, 1>(a, s);
    else launch_vec<T, W, kAdd, 8, 2>(a, s);
  } else {
    launch_rows(rms_norm_scalar_kernel<T, W, kAdd>, a, 4, 256, s);
  }
  return check_launch("rms_norm");
}

template <bool kAdd>
int dispatch(const RmsArgs& a, int dtype, int weight_dtype, hipStream_t s) {
  if (a.rows < 0 || a.hidden <= 0) return set_error("rms_norm: invalid shape");
  if (a.rows == 0) return 0;
  const bool wf32 = weight_dtype == kF32;
  if (!wf32 && weight_dtype != dtype) return set_error("rms_norm: weight must be fp32 or the input dtype");
  if (dtype == kBF16) return wf32 ? launch_rms<__bf16, float, kAdd>(a, s) : launch_rms<__bf16, __bf16, kAdd>(a, s);
  if (dtype == kF16)
    return wf32 ? launch_rms<_Float16, float, kAdd>(a, s) : launch_rms<_Float16, _Float16, kAdd>(a, s);
  return set_error("rms_norm: dtype must be bf16 or fp16");
}

}  // namespace
}  // namespace mva

extern "C" int mva_rms_norm(const void* x, int64_t x_group_stride, int64_t x_row_stride, const void* weight,
                            void* out, int64_t out_group_stride, int64_t out_row_stride, int64_t rows,
                            int64_t rows_per_group, int64_t hidden, float eps, int dtype, int weight_dtype,
                            void* stream) {
  using namespace mva;
  if (hidden > 0x7fffffffLL) return set_error("rms_norm: hidden too large");
  if (rows_per_group <= 0) return set_error("rms_norm: rows_per_group must be positive");
  RmsArgs a{x, x_row_stride, nullptr, 0, weight, out, out_row_stride, nullptr, 0, rows, (int)hidden, eps,
            rows_per_group, x_group_stride, out_group_stride};
  return dispatch<false>(a, dtype, weight_dtype, (hipStream_t)stream);
}

extern "C" int mva_fused_add_rms_norm(const void* x, int64_t x_row_stride, const void* residual,
                                      int64_t residual_row_stride, const void* weight, void* out,
                                      int64_t out_row_stride, void* residual_out,
                                      int64_t residual_out_row_stride, int64_t rows, int64_t hidden, float eps,
                                      int dtype, int weight_dtype, void* stream) {
  using namespace mva;
  if (hidden > 0x7fffffffLL) return set_error("rms_norm: hidden too large");
  if (residual == nullptr || residual_out == nullptr) return set_error("rms_norm: missing residual buffers");
  RmsArgs a{x, x_row_stride, residual, residual_row_stride, weight, out, out_row_stride,
            residual_out, residual_out_row_stride, rows, (int)hidden, eps, 1, x_row_stride, out_row_stride};
  return dispatch<true>(a, dtype, weight_dtype, (hipStream_t)stream);
}
