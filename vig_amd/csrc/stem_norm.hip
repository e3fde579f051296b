// The layer norms of the patch embedding in training, with the bias of the convolution in front and the SiLU behind
// (classification/models/vig.py:619-624,651-656): rows of channels-last maps,
//   s = x + pre_bias,  z = (s - mean) rstd weight + bias,  y = z or z sigmoid(z),
// everything between the stored x and the stored y in fp32, and the gradients of all five in one pass over x and dy.  As separate
// operators under mixed precision each norm was a cast to fp32, the norm, the activation, a cast back, and backwards two passes for the weights and
// one for the input in fp32; the bias another pass each way: 860 us of a training pass of ViG-S (128 images of 224 px).
// HBM-bound: x and y once forward, x, dy and dx once backward.  us (TB/s), forward / backward with its column sum: 100 352 rows of 192, bf16 20.4 (3.8)
// / 38.9 (3.0); 25 088 of 384, fp32 y 12.9 (4.5) / 21.2 (3.6); 6272 of 768 8.5 / 20.2 (of its two octets a lane 128 registers spilled: 35).  ms a training pass under bf16 autocast, before / after: ViG-S,
// 128 images of 224 px 10.83 / 10.29, ViG-B, 32 9.60 / 9.49, ViG-T, 128 6.31 / 6.13.
#include "common.h"
#include "launch.h"

namespace vig {

namespace {

template <typename T> struct Row8;
template <> struct Row8<uint16_t> {
  static __device__ __forceinline__ void store(uint16_t* p, const float (&x)[8]) {
    u32x4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
    *reinterpret_cast<u32x4_t*>(p) = r;
  }
  static __device__ __forceinline__ float sigmoid(float z) { return sigmoidf_(z); }
};
template <> struct Row8<float> {
  static __device__ __forceinline__ void store(float* p, const float (&x)[8]) {
    *reinterpret_cast<f32x4_t*>(p) = f32x4_t{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{x[4], x[5], x[6], x[7]};
  }
  static __device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
};

template <int GROUP>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int off = GROUP / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// a row's octets by GROUP lanes, NV each; lanes without one hold zeros
template <typename TX, int NV, int GROUP>
struct NormRow {
  float s[NV][8], rstd;
  __device__ __forceinline__ void load(const TX* x, const float (&pre)[NV][8], int gl, int nvec, float inv_c, float eps) {
    Raw8<TX> raw[NV];
    float sum = 0.f, sq = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      raw[i].zero();
      if (gl + GROUP * i < nvec) raw[i].load(x + 8 * (gl + GROUP * i));
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      raw[i].unpack(s[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[i][j] += pre[i][j], sum += s[i][j];
    }
    const float mean = group_sum<GROUP>(sum) * inv_c;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) s[i][j] = gl + GROUP * i < nvec ? s[i][j] - mean : 0.f, sq = __builtin_fmaf(s[i][j], s[i][j], sq);
    rstd = 1.0f / sqrtf(group_sum<GROUP>(sq) * inv_c + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) s[i][j] *= rstd;  // the normalised row
  }
};
template <int NV, int GROUP>
__device__ __forceinline__ void load_params(const float* p, float (&x)[NV][8], int gl, int nvec) {
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    Raw8<float> raw;
    raw.zero();
    if (p && gl + GROUP * i < nvec) raw.load(p + 8 * (gl + GROUP * i));
    raw.unpack(x[i]);
  }
}

template <typename TX, typename TY, int NV, int GROUP>
__global__ __launch_bounds__(256) void stem_norm_kernel(const TX* __restrict__ x, const float* __restrict__ pre_bias,
                                                        const float* __restrict__ weight, const float* __restrict__ bias, TY* __restrict__ y,
                                                        int rows, int C, float eps, int silu) {
  const int gl = threadIdx.x % GROUP, nvec = C >> 3, row = blockIdx.x * (256 / GROUP) + threadIdx.x / GROUP;
  float pre[NV][8], w[NV][8], b[NV][8];
  load_params<NV, GROUP>(pre_bias, pre, gl, nvec);
  load_params<NV, GROUP>(weight, w, gl, nvec);
  load_params<NV, GROUP>(bias, b, gl, nvec);
  NormRow<TX, NV, GROUP> r;
  r.load(x + (size_t)min(row, rows - 1) * C, pre, gl, nvec, 1.0f / (float)C, eps);
  if (row >= rows) return;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (gl + GROUP * i >= nvec) continue;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o[j] = __builtin_fmaf(r.s[i][j], w[i][j], b[i][j]);
      if (silu) o[j] = o[j] * Row8<TY>::sigmoid(o[j]);
    }
    Row8<TY>::store(y + (size_t)row * C + 8 * (gl + GROUP * i), o);
  }
}

// Workgroups walk the rows a grid apart and keep their shares of the three parameters' gradients in registers; the waves of a workgroup combine
// through LDS, one parameter after the other, into one row of partials [grid, 3 C], which a column sum finishes (no atomics).
constexpr int kStemThreads = 512, kStemBlocks = 512;  // two workgroups a CU
static_assert(kStemBlocks * (kStemThreads / 16) <= 0x7fffffffLL - VIG_STEM_NORM_ROWS, "a walk's step behind the last row is still an int");
template <typename TX, typename TY, int NV, int GROUP>
__global__ __launch_bounds__(kStemThreads, NV == 1 ? 4 : 2) void stem_norm_bwd_kernel(const TX* __restrict__ x, const float* __restrict__ pre_bias,
                                                                       const float* __restrict__ weight, const float* __restrict__ bias,
                                                                       const TY* __restrict__ dy, TX* __restrict__ dx,
                                                                       float* __restrict__ partials, int rows, int C, float eps, int silu) {
  extern __shared__ __align__(16) float red[];  // [waves][C]
  const int gl = threadIdx.x % GROUP, nvec = C >> 3, wave = threadIdx.x >> 6;
  constexpr int kRows = kStemThreads / GROUP;
  const float inv_c = 1.0f / (float)C;
  float pre[NV][8], w[NV][8], b[NV][8], sums[3][NV][8] = {};
  load_params<NV, GROUP>(pre_bias, pre, gl, nvec);
  load_params<NV, GROUP>(weight, w, gl, nvec);
  load_params<NV, GROUP>(bias, b, gl, nvec);
  for (int row0 = blockIdx.x * kRows; row0 < rows; row0 += gridDim.x * kRows) {
    const int row = row0 + threadIdx.x / GROUP;
    const size_t base = (size_t)min(row, rows - 1) * C;
    const bool ok = row < rows;
    Raw8<TY> graw[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      graw[i].zero();
      if (ok && gl + GROUP * i < nvec) graw[i].load(dy + base + 8 * (gl + GROUP * i));
    }
    NormRow<TX, NV, GROUP> r;
    r.load(x + base, pre, gl, nvec, inv_c, eps);
    float g[NV][8], m1 = 0.f, m2 = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      graw[i].unpack(g[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (silu) {
          const float z = __builtin_fmaf(r.s[i][j], w[i][j], b[i][j]), q = Row8<TY>::sigmoid(z);
          g[i][j] *= q * __builtin_fmaf(z, 1.0f - q, 1.0f);
        }
        sums[0][i][j] = __builtin_fmaf(g[i][j], r.s[i][j], sums[0][i][j]);
        sums[1][i][j] += g[i][j];
        g[i][j] *= w[i][j];
        m1 += g[i][j], m2 = __builtin_fmaf(g[i][j], r.s[i][j], m2);
      }
    }
    m1 = group_sum<GROUP>(m1) * inv_c, m2 = group_sum<GROUP>(m2) * inv_c;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const bool has = ok && gl + GROUP * i < nvec;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        g[i][j] = r.rstd * (g[i][j] - m1 - r.s[i][j] * m2);
        if (has) sums[2][i][j] += g[i][j];
      }
      if (has && dx) Row8<TX>::store(dx + base + 8 * (gl + GROUP * i), g[i]);
    }
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    if (p) __syncthreads();  // the parameter before has been read
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v = sums[p][i][j];
#pragma unroll
        for (int d = 32; d >= GROUP; d >>= 1) v += __shfl_xor(v, d, 64);
        sums[p][i][j] = v;
      }
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if ((threadIdx.x & 63) < GROUP && gl + GROUP * i < nvec) Row8<float>::store(red + wave * C + 8 * (gl + GROUP * i), sums[p][i]);
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += kStemThreads) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < kStemThreads / 64; ++k) acc += red[k * C + c];
      partials[((size_t)blockIdx.x * 3 + p) * C + c] = acc;
    }
  }
}

int stem_grid(long long rows) { return (int)std::min<long long>(kStemBlocks, (rows + 7) / 8); }

}  // namespace

int launch_column_sum(const float* partials, float* out, int n, int C, hipStream_t stream);

bool stem_norm_supported(long long rows, int C, int x_dtype, int y_dtype) {
  return C % 8 == 0 && C > 0 && C <= 1024 && rows > 0 && rows <= VIG_STEM_NORM_ROWS && (x_dtype == 1 || (x_dtype == 0 && y_dtype == 0));
}
size_t stem_norm_bwd_workspace(long long rows, int C) { return (size_t)stem_grid(rows) * 3 * C * sizeof(float); }

#define VIG_STEM_GROUP(LAUNCH)      \
  if (C <= 128) LAUNCH(1, 16);      \
  else if (C <= 256) LAUNCH(1, 32); \
  else if (C <= 512) LAUNCH(1, 64); \
  else LAUNCH(2, 64)

template <typename TX, typename TY>
static int fwd(const void* x, const float* pre, const float* w, const float* b, void* y, int rows, int C, float eps, int silu, hipStream_t stream) {
#define VIG_STEM_CASE(NV, GROUP)                                                                                               \
  hipLaunchKernelGGL((stem_norm_kernel<TX, TY, NV, GROUP>), dim3((rows + 256 / GROUP - 1) / (256 / GROUP)), dim3(256), 0, stream, \
                     (const TX*)x, pre, w, b, (TY*)y, rows, C, eps, silu)
  VIG_STEM_GROUP(VIG_STEM_CASE);
#undef VIG_STEM_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}
template <typename TX, typename TY>
static int bwd(const void* x, const float* pre, const float* w, const float* b, const void* dy, void* dx, float* partials, int rows, int C,
               float eps, int silu, hipStream_t stream) {
#define VIG_STEM_CASE(NV, GROUP)                                                                                                       \
  hipLaunchKernelGGL((stem_norm_bwd_kernel<TX, TY, NV, GROUP>), dim3(stem_grid(rows)), dim3(kStemThreads), kStemThreads / 64 * C * sizeof(float), \
                     stream, (const TX*)x, pre, w, b, (const TY*)dy, (TX*)dx, partials, rows, C, eps, silu)
  VIG_STEM_GROUP(VIG_STEM_CASE);
#undef VIG_STEM_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_stem_norm(const void* x, const float* pre, const float* w, const float* b, void* y, long long rows, int C, float eps, int silu,
                     int x_dtype, int y_dtype, hipStream_t stream) {
  if (!stem_norm_supported(rows, C, x_dtype, y_dtype)) return -95;
  const auto fn = x_dtype == 0 ? fwd<float, float> : y_dtype == 0 ? fwd<uint16_t, float> : fwd<uint16_t, uint16_t>;
  return fn(x, pre, w, b, y, (int)rows, C, eps, silu, stream);
}
int launch_stem_norm_bwd(const void* x, const float* pre, const float* w, const float* b, const void* dy, void* dx, float* dparams, void* workspace,
                         long long rows, int C, float eps, int silu, int x_dtype, int y_dtype, hipStream_t stream) {
  if (!stem_norm_supported(rows, C, x_dtype, y_dtype)) return -95;
  const auto fn = x_dtype == 0 ? bwd<float, float> : y_dtype == 0 ? bwd<uint16_t, float> : bwd<uint16_t, uint16_t>;
  if (const int rc = fn(x, pre, w, b, dy, dx, (float*)workspace, (int)rows, C, eps, silu, stream)) return rc;
  return launch_column_sum((const float*)workspace, dparams, stem_grid(rows), 3 * C, stream);
}

}  // namespace vig
