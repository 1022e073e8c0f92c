// Shared helpers for the gfx950 kernels and the C-ABI implementation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>

#include "cdml.h"

namespace cdml {

// Thread-local last-error message (cdml_last_error()).
void set_error(const char *fmt, ...);
int fail(int code, const char *fmt, ...);

// Makes the library's device current on the calling thread.
int ensure_device();

// Finds this device's copy of the static scratch behind the no-allocation
// entry points (hipGetSymbolAddress); called by cdml_init with `device`
// current.  It does not touch the thread's last error: a failure is
// described in `msg` and reported by the entry point that needs the scratch.
int noalloc_scratch_setup(int device, char *msg, size_t msg_bytes);

// Compute units of the current device (queried once; 256 on MI355X).
int num_cus();

// Checks the launch that was just enqueued.
int check_launch(const char *what);

inline hipStream_t as_hip(cdml_stream s) { return reinterpret_cast<hipStream_t>(s); }

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Launch geometry for gfx950: 8 XCDs, and hardware hands workgroup i to XCD
// i % 8.  xcd_remap() turns the hardware id into a logical id such that each
// XCD receives one contiguous range of logical work, so neighbouring tiles
// (same head, same weight panel) share an L2.
constexpr int kNumXcd = 8;

__device__ __forceinline__ int xcd_remap(int hw_id, int padded_total) {
  const int per_xcd = padded_total / kNumXcd;
  return (hw_id % kNumXcd) * per_xcd + hw_id / kNumXcd;
}

inline int pad_to_xcd(int n) { return (n + kNumXcd - 1) / kNumXcd * kNumXcd; }

// fp32 MFMA 32x32x2: D = A(32x2) * B(2x32) + C, one block.
// Operand layout (lane l, half h = l / 32):
//   A[i][k]: i = l % 32, k = h      B[k][j]: j = l % 32, k = h
//   D[i][j]: j = l % 32, i = 8*(r/4) + 4*h + (r%4) for accumulator r = 0..15
typedef float floatx16 __attribute__((ext_vector_type(16)));
// Native 4-float vector for register staging: unlike HIP's float4 struct it
// is always kept in registers (no private-memory copies of staging arrays).
typedef float vf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 mfma32x32x2(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// fp32 products on the bf16 matrix cores.  An fp32 value is the sum of three
// bf16 values, h = bf16(x), m = bf16(x - h), l = x - h - m, each rounded to
// nearest: 8 + 8 + 8 significant bits hold all 24.  Operands are multiplied by
// kSplitScale = 2^16 on their way into the split, and the sums by 2^-32 at the end:
// the last bit of the smallest fp32 value, 2^-149, then lies at 2^-133, the last
// bit of the smallest bf16 value (the MFMA keeps subnormal operands and sums), so
// the split loses nothing at all.  (Unscaled, l underflows below 2^-110: an operand
// of rms 2^-118 had an error of 9e-6, one of 2^-124 6e-4.)  Of the nine products
// of two split operands, hh + hm + mh + mm + hl + lh are summed in fp32; ml, lm
// and ll are below 2^-24 of |a b| together.  Six bf16 products take 6/16 of one
// fp32 product's matrix-core cycles.
//
// The bf16 MFMA adds eight products at a time to its accumulator, one rounding
// each: with all six products in one accumulator a K of 16 takes 12 roundings
// of the whole sum, where the fp32 MFMA takes 16, and fewer where operands are
// zero (behind a ReLU the single-accumulator form came out 8% worse than fp32,
// so it was not kept).  hh has an accumulator of its own and the five
// corrections, 2^-8 and less of it, another: two roundings of the whole sum per
// 16.  Error against float64 (2-norm, N(0, 1) operands, 256 x 256 outputs): K =
// 64 0.5e-7, 1024 1.9e-7, 8192 5.8e-7, where the fp32 MFMA has 1.4e-7, 5.7e-7 and
// 16e-7 (positive operands, K = 8192: 4.2e-7 against 11.9e-7).
//
// The bf16 MFMA aligns its addends to the largest of them and drops the bits
// below by rounding down, so a long sum drifts towards minus infinity by about
// 1e-8 of its size: nothing next to an element's own rounding error, but the
// same sign in every element, which a column sum over many rows collects (a
// bias gradient over 130816 rows had 5.8e-6 instead of 4.5e-7).  The kernels
// therefore compute every other row and column of a product negated (the operands
// change their sign as they are split, at no cost), which turns the drift round,
// and undo the sign at the end; along the queries of the attention output and the
// keys of dV, whose other operand, the probabilities, is not scaled, every other
// workgroup does.
//
// An infinity, a NaN or a value of 2^112 and more (above the largest bf16 once
// scaled) leaves inf - inf in m, and a sum of 2^96 and more overflows, so every
// result that one reaches comes out non-finite; the kernels test their results for
// that (any_nonfinite) and recompute such blocks with mfma32x32x2, whose
// infinities and NaNs are those of the fp32 sum.  That walks K serially from memory:
// one NaN takes a 16384 x 1024 -> 4096 product from 0.79 to 1.5 ms, its input gradient
// from 0.78 to 2.8, its weight gradient from 0.71 to 6.3, and an attention backward of
// 4 x 4096 from 2.3 to 9.3.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t vu2 __attribute__((ext_vector_type(2)));
typedef uint32_t vu4 __attribute__((ext_vector_type(4)));
constexpr int kSplitProducts = 6;
constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};  // piece of A (0 = h, 1 = m, 2 = l)
constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};  // piece of B
constexpr int kSplitMain = 5;                                // hh; the others are its corrections

constexpr float kSplitScale = 65536.f;             // 2^16, of either operand
constexpr float kSplitUnscale = 1.f / 65536.f;     // of a sum with one scaled operand
constexpr float kSplitUnscale2 = kSplitUnscale * kSplitUnscale;  // with two

// (bf16(a), bf16(b)) in the low and high half, rounded to nearest even.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef float vf2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((vf2{a, b}), bf16x2));
}

// The three pieces of a (low halves) and b (high halves).
__device__ __forceinline__ void split_bf16x3(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
  h = pack_bf16(a, b);
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = pack_bf16(ra, rb);
  l = pack_bf16(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}

// The three pieces of eight values as MFMA operands.
__device__ __forceinline__ void split_operand(const float (&x)[8], float scale, bf16x8 (&p)[3]) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) split_bf16x3(x[2 * i] * scale, x[2 * i + 1] * scale, h[i], m[i], l[i]);
  p[0] = __builtin_bit_cast(bf16x8, (vu4{h[0], h[1], h[2], h[3]}));
  p[1] = __builtin_bit_cast(bf16x8, (vu4{m[0], m[1], m[2], m[3]}));
  p[2] = __builtin_bit_cast(bf16x8, (vu4{l[0], l[1], l[2], l[3]}));
}

// bf16 MFMA 32x32x16: D = A(32x16) * B(16x32) + C.  Lane l holds eight
// consecutive k, 8 * (l / 32) + 0..7, of row (A) or column (B) l % 32; D as
// mfma32x32x2.
__device__ __forceinline__ floatx16 mfma32x32x16(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 0 when every value of v is finite, NaN otherwise (summed into s).
__device__ __forceinline__ float nonfinite_sum(const floatx16 &v, float s) {
#pragma unroll
  for (int r = 0; r < 16; ++r) s = fmaf(v[r], 0.f, s);
  return s;
}
// Whether any lane's nonfinite_sum found one (wave-uniform).
__device__ __forceinline__ bool any_nonfinite(float s) { return __builtin_amdgcn_ballot_w64(s != s) != 0; }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The forward attention launcher (flash_attn.hip) for callers that have
// validated their arguments.  With lse non-NULL it also writes each row's
// log2 softmax normaliser ([batch * heads][lq]; head dims up to 128).
// causal: key j is visible to query i iff j <= i (lq may differ from lk).
int flash_forward(const float *q, int ldq, const float *k, int ldk, const float *v, int ldv,
                  float *o, int ldo, float *lse, int batch, int lq, int lk, int dim, int num_heads,
                  float scale, bool causal, const uint8_t *mask, hipStream_t st);

}  // namespace cdml
