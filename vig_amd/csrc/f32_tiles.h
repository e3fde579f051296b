// Building blocks of the fp32 GLA kernels on the bf16 matrix cores (gfx950): an fp32 value is the exact sum of three
// bf16 pieces (8 + 8 + 8 significand bits, each rounded to nearest), and a product is the six piece products that
// matter, x*y = h*h + (h*m + m*h) + (m*m + h*l + l*h), accumulated in fp32.  What is left out (m*l, l*m, l*l) is below
// 2^-25 of the product, under fp32's own rounding.  Six v_mfma_f32_32x32x16_bf16 take 6 x 32 clocks for what
// v_mfma_f32_32x32x2_f32 needs 8 x 64 clocks for: 2.7 times the rate of the fp32 matrix instruction, 157 TFLOP/s.
#pragma once
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {
namespace {

typedef float f32x8_t __attribute__((ext_vector_type(8)));

struct P3 {  // eight contraction slots in three bf16 pieces (high, middle, low)
  u32x4_t p[3];
};

__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& a, uint32_t& b, uint32_t& c) {
  a = pack_bf16x2(x0, x1);
  const float r0 = x0 - bf16lo_to_f32(a), r1 = x1 - bf16hi_to_f32(a);  // (exact)
  b = pack_bf16x2(r0, r1);
  c = pack_bf16x2(r0 - bf16lo_to_f32(b), r1 - bf16hi_to_f32(b));
}
__device__ __forceinline__ P3 split8(f32x8_t x) {
  P3 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a, b, c;
    split_pair(x[2 * i], x[2 * i + 1], a, b, c);
    o.p[0][i] = a, o.p[1][i] = b, o.p[2][i] = c;
  }
  return o;
}
// the six products: the leading one into one accumulator, the five that correct it into another, so that the large sum
// is rounded once per contraction step and not six times
__device__ __forceinline__ void mfma6(const P3& a, const P3& b, f32x16_t& big, f32x16_t& small) {
  small = mfma(a.p[2], b.p[0], small);
  big = mfma(a.p[0], b.p[0], big);
  small = mfma(a.p[0], b.p[2], small);
  small = mfma(a.p[1], b.p[1], small);
  small = mfma(a.p[1], b.p[0], small);
  small = mfma(a.p[0], b.p[1], small);
}

// three LDS units (64 lanes x 16 bytes each) of an operand
__device__ __forceinline__ void store_p3(char* region, int u, int lane, const P3& x) {
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4_t*>(unit_ptr(region, 3 * u + i, lane)) = x.p[i];
}
__device__ __forceinline__ P3 load_p3(char* region, int u, int lane) {
  P3 x;
#pragma unroll
  for (int i = 0; i < 3; ++i) x.p[i] = *reinterpret_cast<const u32x4_t*>(unit_ptr(region, 3 * u + i, lane));
  return x;
}

// inclusive prefix sum over the 32 lanes of each half: four shifts inside the rows of sixteen, then the first row's
// total into the second one
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_or_zero(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float prefix32(float x) {
  x += dpp_or_zero<0x111, 0xf>(x);
  x += dpp_or_zero<0x112, 0xf>(x);
  x += dpp_or_zero<0x114, 0xf>(x);
  x += dpp_or_zero<0x118, 0xf>(x);
  x += dpp_or_zero<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
  return x;
}

// raw fp32 rows of one 32-token tile: lane (r, h) reads token r, channels [8*NG*h, +8*NG)
template <int NG>
__device__ __forceinline__ void load_rows_f32(rsrc_t rows, int r, int h, f32x8_t (&x)[NG]) {
  const unsigned base = (unsigned)r * (64u * NG) + 32u * NG * h;
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    const f32x4_t a = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rows, base + 32u * c, 0, 0));
    const f32x4_t b = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rows, base + 32u * c + 16u, 0, 0));
    x[c] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
}
__device__ __forceinline__ f32x8_t lds_f32x8(const float* p) {
  const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
// values of one tile for transposed fragments (tokens in the contraction slots): x[p][t][e] = channel
// 2*cpair<4>(r) + p of token jmap(t, h, e)
__device__ __forceinline__ void load_pairs_f32(rsrc_t rows, int r, int h, f32x8_t (&x)[2][2]) {
  const unsigned base = (4u * h) * 256u + 8u * cpair<4>(r);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const u32x2_t w = __builtin_amdgcn_raw_buffer_load_b64(rows, base + (unsigned)jmap(t, 0, e) * 256u, 0, 0);
      x[0][t][e] = __uint_as_float(w[0]), x[1][t][e] = __uint_as_float(w[1]);
    }
}
__device__ __forceinline__ f32x8_t octet(const float (&x)[16], int t) {
  f32x8_t y;
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = x[8 * t + e];
  return y;
}
__device__ __forceinline__ float sum_abs(f32x8_t x) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += fabsf(x[e]);
  return s;
}
// registers 8t .. 8t + 7 of an accumulator
template <int T>
__device__ __forceinline__ f32x8_t half_of(const f32x16_t& P) {
  return __builtin_shufflevector(P, P, 8 * T, 8 * T + 1, 8 * T + 2, 8 * T + 3, 8 * T + 4, 8 * T + 5, 8 * T + 6, 8 * T + 7);
}

// element of a state slot (kGlaStateFloats) that holds S[key channel ch][value channel vch]
template <int NG>
__device__ __forceinline__ int state_index(int ch, int vch) {
  const int h = ch / (8 * NG), cq = (ch >> 3) & (NG - 1), m = (ch >> 1) & 3, pk = ch & 1;
  const int pv = vch & 1, cp = vch >> 1;
  const int r = ((cp >> 4) << 2) | (((cp >> 2) & 3) << 3) | (cp & 3);
  return (((pk * 2 + pv) * 4 + cq) * 64 + 32 * h + r) * 4 + m;
}

}  // namespace
}  // namespace vig
