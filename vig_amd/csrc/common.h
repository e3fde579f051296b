// Shared device helpers for the gfx950 GLA kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vig {

typedef __bf16 bf16_t;
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// bf16 <-> f32 through the native type: hipcc lowers the narrowing conversion to
// the round-to-nearest-even hardware convert of gfx950.
__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  bf16_t h = (bf16_t)f;
  return __builtin_bit_cast(uint16_t, h);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  f32x2_t x = {lo, hi};
  bf16x2_t y = __builtin_convertvector(x, bf16x2_t);
  return __builtin_bit_cast(uint32_t, y);
}
__device__ __forceinline__ float bf16lo_to_f32(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16hi_to_f32(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// eight channels as stored (no conversion): what a kernel that only moves them keeps in registers
template <typename T> struct Raw8;
template <> struct Raw8<uint16_t> {
  u32x4_t a;
  __device__ __forceinline__ void zero() { a = u32x4_t{0u, 0u, 0u, 0u}; }
  __device__ __forceinline__ void load(const uint16_t* p) { a = *reinterpret_cast<const u32x4_t*>(p); }
  __device__ __forceinline__ void store(uint16_t* p) const { *reinterpret_cast<u32x4_t*>(p) = a; }
  __device__ __forceinline__ void unpack(float (&x)[8]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = bf16lo_to_f32(a[i]);
      x[2 * i + 1] = bf16hi_to_f32(a[i]);
    }
  }
};
template <> struct Raw8<float> {
  f32x4_t a, b;
  __device__ __forceinline__ void zero() { a = b = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const f32x4_t*>(p);
    b = *reinterpret_cast<const f32x4_t*>(p + 4);
  }
  __device__ __forceinline__ void store(float* p) const {
    *reinterpret_cast<f32x4_t*>(p) = a;
    *reinterpret_cast<f32x4_t*>(p + 4) = b;
  }
  __device__ __forceinline__ void unpack(float (&x)[8]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a[i];
      x[4 + i] = b[i];
    }
  }
};

// Channel octets of token rows dealt out to workgroups: a workgroup owns `tokens` consecutive rows of [B * L] tokens of nv octets each
// and numbers their octets through, so that neighbouring lanes hold neighbouring octets whatever the width and every lane has one.
struct OctetRows {
  int b, l, n;    // first token, and octets to do
  __device__ __forceinline__ OctetRows(int B, int L, int nv, int tokens) {
    const unsigned first = blockIdx.x * (unsigned)tokens;
    b = (int)(first / (unsigned)L), l = (int)(first - (unsigned)b * L);
    n = (int)min((unsigned)tokens, (unsigned)B * L - first) * nv;
  }
};
struct Octet {
  int b, l, cv;  // batch element, token and octet of its row
  __device__ __forceinline__ Octet(const OctetRows& rows, int x, int nv, int L) {
    const unsigned dt = (unsigned)x / (unsigned)nv;
    cv = x - (int)dt * nv, b = rows.b;
    unsigned at = rows.l + dt;
    if (at >= (unsigned)L) b += at / (unsigned)L, at %= (unsigned)L;
    l = (int)at;
  }
};

// Typed element access used by the dtype-generic (non-MFMA) kernels.
template <typename T> struct Elem;
template <> struct Elem<float> {
  static __device__ __forceinline__ float load(const float* p) { return *p; }
  static __device__ __forceinline__ void store(float* p, float v) { *p = v; }
};
template <> struct Elem<uint16_t> {  // bf16 storage
  static __device__ __forceinline__ float load(const uint16_t* p) { return bf16_to_f32(*p); }
  static __device__ __forceinline__ void store(uint16_t* p, float v) { *p = f32_to_bf16(v); }
};

// (hardware reciprocal, 1 ulp: a full-precision division costs ten instructions more per value)
// e^-|..| style arguments only need the bare hardware instructions (2^x and log2 x, 1 ulp): results below the
// normal range flush to zero, which is exact enough next to 1, and the guards the library versions wrap around them
// (range tests, rescaling) cost more than the instructions themselves.
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float sigmoidf_(float x) { return __builtin_amdgcn_rcpf(1.0f + exp_fast(-x)); }
// log(sigmoid(x)) = min(x, 0) - log(1 + e^-|x|); the log's argument lies in [1, 2]
__device__ __forceinline__ float logsigmoidf_(float x) {
  return fminf(x, 0.f) - 0.6931471805599453f * __builtin_amdgcn_logf(1.f + exp_fast(-fabsf(x)));
}

// out[c] = sum over the n rows of partials [n, C].  The rows were written by every XCD, so a load is a trip to memory: a workgroup of 1024 takes
// 16 columns, a thread every 64th row of one, eight loads under way at a time.  Measured with the
// kernel in front of it, 512 to 1024 rows of 128: 3.7 us less than with 64 columns a workgroup and four loads.
__device__ __forceinline__ void sum_columns(const float* partials, float* out, int n, long long C, int block, float (*red)[17]) {
  const int col = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const long long c = (long long)block * 16 + col;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (c < C) {
    for (int i = slice; i < n; i += 512) {
      float x[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = i + 64 * k < n ? partials[(size_t)(i + 64 * k) * C + c] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] += x[k];
    }
  }
  red[slice][col] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  __syncthreads();
  if (threadIdx.x < 64) {  // four threads a column, 16 slices each
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[4 * k + (threadIdx.x >> 4)][col];
    t += __shfl_xor(t, 16);
    t += __shfl_xor(t, 32);
    if (threadIdx.x < 16 && c < C) out[c] = t;
  }
}

// 16 bytes per lane from memory straight into LDS: lane i lands 16 i bytes behind lds_base (wave-uniform byte offset in the
// workgroup's LDS).  In assembly, because the compiler answers the builtin of this load with waits of its own in front of
// every later LDS read it cannot tell apart from the destination, down to vmcnt(0), which also drains the stores and the
// loads of stages further ahead.  The caller waits (wait_vmem), counting what it has issued since.  (m0 is reserved, so it
// cannot be named as changed: no kernel mixes this with the builtin.)
__device__ __forceinline__ void load_to_lds16(const void* p, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(p) : "memory");
}
// (base: wave-uniform; 32-bit byte offset a lane.)  The base has to come out of scalar arithmetic.  One in vector registers does not
// assemble; one that v_readfirstlane has just brought over may be read as a load's address five wait states later at the earliest, which the
// compiler sees to between its own instructions, but not into an asm block, where there are two: tests/test_isa_hazards.py goes through
// the compiled callers for that.  (Five wait states in here cost the weight gradients 1 %: 25088 rows, 2048 x 384 67.2 -> 68.0 us.)
__device__ __forceinline__ void load_to_lds16(const void* base, uint32_t offset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(offset), "s"(base) : "memory");
}
// at most N vector memory operations (loads and stores, in the order of issue) still out
template <int N>
__device__ __forceinline__ void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

}  // namespace vig
