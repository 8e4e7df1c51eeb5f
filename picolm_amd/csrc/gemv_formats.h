// gemv_formats.h -- what the weight GEMV kernels (gemv.hip) and the batched
// ones on the matrix cores (gemm.hip) share: type ids, launch arguments and
// the small device helpers of the packed formats.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attn_common.h"

namespace plh {

constexpr int kThreads = 256;
constexpr int kTypeQ8_0 = 8, kTypeQ4K = 12, kTypeQ6K = 14;
constexpr size_t kPlaneAlign = 256;
constexpr size_t kMaxPacked = (size_t)1 << 31;  // 32-bit plane offsets

struct GemvArgs {
  const uint8_t* w;     // packed matrix
  const float* x;       // [n]
  float* out;           // [d]
  int d;
  int nb;               // blocks per row
  int units;            // lane units per row
  int uspan;            // units covered by one pass of the threads (<= 256)
  int row_par;          // rows worked side by side (kThreads / uspan)
  int unit_iters;       // passes over the units
  int rows_per_wg;      // rows of one workgroup (row_par * rows per thread)
  int terms;            // chained terms per row
  int tpitch;           // LDS pitch of a row's terms
  uint32_t off0, off1, off2, scales_off, d_off;  // plane offsets (bytes)
  // Epilogue, in the reference's order (tensor.c:256-264, 605-657):
  // v = dot; v = v + bias[i] (bias_mode 1) or v + 0.0f (bias_mode 2, a
  // zero-filled bias); v = silu(gate[i]) * v; v = resid[i] + v.
  const float* bias;
  const float* gate;
  const float* resid;
  int bias_mode;
  // Prologue (gemv_kernel<..., true>): x is rmsnorm(x, norm_w) of length n
  // (tensor.c:425-492), formed by every workgroup itself.
  const float* norm_w;
  float norm_eps;
  int n;
  int xs_off;  // floats from the LDS base to the staged rmsnorm(x)
  float* xn_out;  // workgroup 0 also stores rmsnorm(x) here (or null)
  // Gate/up pair (gemv_body<..., true>): virtual row 2r is row r of w (gate),
  // 2r + 1 row r of w2 (up, same type and shape); out[r] = silu(gate) * up.
  const uint8_t* w2;
};

// tensor.c:605-609: x / (1 + expf(-x)).  expf is the device library's, not
// glibc's (which is not correctly rounded), so results can differ from the
// host's in the last place.
__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }

__device__ __forceinline__ float hsum8(const float (&v)[8]) {
  const float a0 = v[0] + v[4], a1 = v[1] + v[5], a2 = v[2] + v[6], a3 = v[3] + v[7];
  return (a0 + a2) + (a1 + a3);
}

__device__ __forceinline__ float4 ld4(const float* p) { return *(const float4*)p; }

template <class T>
__device__ __forceinline__ T ld(const uint8_t* w, uint32_t off) {
  return *(const T*)(w + off);
}

// byte B of a word as a float, exact (v_cvt_f32_ubyteB: one instruction)
template <int B>
__device__ __forceinline__ float ubyte(uint32_t w) {
  float r;
  if constexpr (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(r) : "v"(w));
  if constexpr (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(r) : "v"(w));
  if constexpr (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(r) : "v"(w));
  if constexpr (B == 3) asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(r) : "v"(w));
  return r;
}
__device__ __forceinline__ float ubyte(uint32_t w, int b) {
  switch (b) {
    case 0: return ubyte<0>(w);
    case 1: return ubyte<1>(w);
    case 2: return ubyte<2>(w);
    default: return ubyte<3>(w);
  }
}
__device__ __forceinline__ float sbyte(uint32_t w, int b) {
  return (float)(int)(int8_t)((w >> (8 * b)) & 0xFFu);
}

// A batched launch: tokens, floats between x rows / out rows, tiles.
struct BatchShape {
  int n_tok, x_stride, out_stride;
  int row_tiles, tok_tiles;
};

// gemm.hip: the batched GEMV on the matrix cores, x rows x_stride apart, out
// rows (and gate, resid) out_stride apart; pair: gate a.w, up a.w2.  0 or -1.
int gemm_mfma(int qtype, bool pair, const GemvArgs& a, int n_tok, int x_stride, int out_stride);
// Three matrices over the same x in one launch, K quants only or Q8_0 only, and
// whether that is faster than three launches.
bool gemm_mfma_multi_pays(const int* qtype, const GemvArgs* a, int n_tok);
int gemm_mfma_multi(const int* qtype, const GemvArgs* a, int n_tok, int x_stride,
                    const int* out_stride);
// Whether it is the faster of the two batched kernels for this shape.
bool gemm_mfma_pays(int qtype, const GemvArgs& a, int n_tok, bool pair);

}  // namespace plh
