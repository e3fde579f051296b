// Few images: the front of a block in one kernel.  Residual add, RMS norm, depthwise 3x3 convolution (+ SiLU) and the stacked
// projection behind it (classification/models/vig.py:291-294,364-369,598-606).
//
// One image is a chain of launches, each as long as its own chain of loads: a kernel here lives 3 to 5 us, about 1 us lies between
// two, and the work in them is far below that.  So a workgroup makes for itself what its tile of the projection reads: tokens come in
// patches of 2 x 8 grid cells, whose sums and norms are 4 x 10 cells whatever the grid's width, and the convolution of the patch's
// 16 tokens is every row of the contraction.  Every column tile makes them again, out of the L2; the first one stores the sums and the
// convolution's result, which the block's epilogue reads.
// What bounds it is the chain itself: loads, norms and convolution of a workgroup's patch on one CU (5 us on an empty chip too).  us,
// the two or three kernels it stands for / this: C 192, N 640: 8 x 8 6.3 / 5.0, 14 x 14 6.9 / 5.0, three 14 x 14 7.5 / 5.3; C 384, N 1280: 8 x 8
// 7.0 / 6.7, 14 x 14 8.5 / 6.9.  Patches of 4 x 8 cells and 64 columns, the contraction split over the waves: 6.0 and 9.7 us at 14 x 14 (twice
// the norms and the convolution on a CU); weights waited for in front of the convolution, eight waves at C 384: 8.1.
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

constexpr int kPatchH = 2, kPatchW = 8, kCells = (kPatchH + 2) * (kPatchW + 2), kTokens = kPatchH * kPatchW, kColumns = 128;

struct ConvLinearArgs {
  const uint16_t *x, *residual;        // [B, h*w, C]; no residual: null
  const float *norm, *taps, *conv_bias;  // [C], [C, 9], [C] or null
  const uint16_t *w, *bias;            // [N, C], [N] or null
  uint16_t *sum, *conv, *y;            // [B, h*w, C] (or null), [B, h*w, C], [B, h*w, N]
  int h, w_cells, N, down, across, silu;  // down, across: patches of an image
  float eps;
};

template <int C>
struct ConvLinearLds {
  static constexpr int kStages = C / 32;
  static constexpr int kTaps = (C * 9 * 4 + 1023) / 1024 * 1024;  // whole wave loads
  static constexpr int kTapsAt = kCells * C * 2, kWeightsAt = kTapsAt + kTaps, kRowsAt = kWeightsAt + kColumns * C * 2;
  static constexpr int kBytes = kRowsAt + kTokens * C * 2;
};

// Norms: C / 24 lanes a cell.  Convolution: a thread takes four channels of one column of the patch and walks down its four rows of
// cells.  Product: each of the first eight waves has 16 columns and the whole contraction, in stages of 32 (1 KB of either operand: 16
// rows of four 16-byte units, swapped as in gemm.hip).
template <int C>
__global__ __launch_bounds__(C == 192 ? 512 : 1024) void conv_linear_kernel(ConvLinearArgs a) {
  using Lds = ConvLinearLds<C>;
  constexpr int kThreads = C == 192 ? 512 : 1024, NV = 3, kLanes = C / 24, kStages = Lds::kStages, kUnits = C / 4;
  static_assert(kCells * kLanes <= kThreads && kUnits * kPatchW <= kThreads, "one pass of each");
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 15, quarter = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n0 = blockIdx.x * kColumns;
  const int img = blockIdx.y / (a.down * a.across), patch = blockIdx.y - img * (a.down * a.across);
  const int y0 = patch / a.across * kPatchH, x0 = (patch - patch / a.across * a.across) * kPatchW;
  const size_t image = (size_t)img * a.h * a.w_cells;
  const uint32_t lds0 = lds_offset(smem);
  // ---- under way: the taps straight to LDS, the cells' rows, what the norm and the sums start from ----
  for (int i = wave; i < Lds::kTaps / 1024; i += kThreads / 64)
    load_to_lds16(a.taps + min(256 * i + 4 * lane, C * 9 - 4), lds0 + Lds::kTapsAt + 1024 * i);
  const int sub = threadIdx.x % kLanes, cell = threadIdx.x / kLanes, cy = cell / (kPatchW + 2), cx = cell - cy * (kPatchW + 2);
  const bool in = cell < kCells && y0 - 1 + cy >= 0 && y0 - 1 + cy < a.h && x0 - 1 + cx >= 0 && x0 - 1 + cx < a.w_cells;
  const size_t at = in ? (image + (size_t)(y0 - 1 + cy) * a.w_cells + x0 - 1 + cx) * C + 8 * sub : 0;
  Raw8<uint16_t> x[NV], res[NV];
  f32x4_t norm[NV][2];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    x[i].zero(), res[i].zero();
    if (in) x[i].load(a.x + at + 8 * kLanes * i);
    if (in && a.residual) res[i].load(a.residual + at + 8 * kLanes * i);
    norm[i][0] = *reinterpret_cast<const f32x4_t*>(a.norm + 8 * (sub + kLanes * i));
    norm[i][1] = *reinterpret_cast<const f32x4_t*>(a.norm + 8 * (sub + kLanes * i) + 4);
  }
  const int unit = threadIdx.x % kUnits, col = threadIdx.x / kUnits, ch = 4 * unit;
  const f32x4_t start = a.conv_bias ? *reinterpret_cast<const f32x4_t*>(a.conv_bias + ch) : f32x4_t{0.f};
  const int n = n0 + 16 * (wave & 7) + 4 * quarter;
  const u32x2_t bias = a.bias ? *reinterpret_cast<const u32x2_t*>(a.bias + n) : u32x2_t{0u, 0u};
  // ---- sums and norms of the cells ----
  float s[NV][8], sq[NV] = {};
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float b[8];
    x[i].unpack(s[i]);
    res[i].unpack(b);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[i].a[j] = pack_bf16x2(s[i][2 * j] + b[2 * j], s[i][2 * j + 1] + b[2 * j + 1]);  // the rounded sum
    x[i].unpack(s[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) sq[i] = __builtin_fmaf(s[i][j], s[i][j], sq[i]);
  }
  float ss = (sq[0] + sq[2]) + sq[1];  // the order of rmsnorm_kernel's wave, so its bits
  // the weights, which only the product waits for: issued once the rows are here, since the compiler's waits do not count them
  asm volatile("" : "+v"(ss));
  wait_vmem<0>();
  const uint32_t weights = (uint32_t)(Lds::kWeightsAt + (wave & 7) * (kStages * 1024));
  if (wave < 8) {
    const uint16_t* const w = a.w + (size_t)(n0 + 16 * wave + (lane >> 2)) * C + 8 * ((lane & 3) ^ ((lane >> 4) & 3));
#pragma unroll
    for (int k = 0; k < kStages; ++k) load_to_lds16(w + 32 * k, lds0 + weights + 1024 * k);
  }
#pragma unroll
  for (int d = kLanes / 2; d > 0; d >>= 1) ss += __shfl_xor(ss, d);
  const float rstd = 1.0f / sqrtf(ss / (float)C + a.eps);
  if (cell < kCells) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      u32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = in ? pack_bf16x2(s[i][2 * j] * rstd * norm[i][j >> 1][2 * (j & 1)], s[i][2 * j + 1] * rstd * norm[i][j >> 1][2 * (j & 1) + 1]) : 0u;
      *reinterpret_cast<u32x4_t*>(smem + 2 * (cell * C + 8 * (sub + kLanes * i))) = v;
    }
  }
  lds_barrier();
  // ---- the convolution ----
  u32x2_t conv[kPatchH];
  if (col < kPatchW) {
    float taps[36], acc[kPatchH][4];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      const f32x4_t t = *reinterpret_cast<const f32x4_t*>(smem + Lds::kTapsAt + 36 * ch + 16 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) taps[4 * i + j] = t[j];
    }
#pragma unroll
    for (int o = 0; o < kPatchH; ++o)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[o][c] = start[c];
#pragma unroll
    for (int i = 0; i < kPatchH + 2; ++i)
#pragma unroll
      for (int dj = 0; dj < 3; ++dj) {
        const u32x2_t v = *reinterpret_cast<const u32x2_t*>(smem + 2 * ((i * (kPatchW + 2) + col + dj) * C + ch));
#pragma unroll
        for (int o = 0; o < kPatchH; ++o) {
          if (i - o < 0 || i - o > 2) continue;
#pragma unroll
          for (int c = 0; c < 4; ++c)
            acc[o][c] = __builtin_fmaf(c & 1 ? bf16hi_to_f32(v[c / 2]) : bf16lo_to_f32(v[c / 2]), taps[9 * c + (i - o) * 3 + dj], acc[o][c]);
        }
      }
#pragma unroll
    for (int o = 0; o < kPatchH; ++o) {
      if (a.silu) {
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[o][c] = acc[o][c] * sigmoidf_(acc[o][c]);
      }
      conv[o] = u32x2_t{pack_bf16x2(acc[o][0], acc[o][1]), pack_bf16x2(acc[o][2], acc[o][3])};
      const int row = kPatchW * o + col, oct = unit >> 1;
      *reinterpret_cast<u32x2_t*>(smem + Lds::kRowsAt + (oct >> 2) * 1024 + row * 64 + 16 * ((oct & 3) ^ ((row >> 2) & 3)) + 8 * (unit & 1)) = conv[o];
    }
  }
  wait_vmem<0>();
  lds_barrier();
  // ---- the product ----
  if (wave < 8) {
    f32x4_t part[4];  // (every fourth stage a sum of its own: gemm_few_kernel's order, so its bits)
#pragma unroll
    for (int k = 0; k < 4; ++k) part[k] = f32x4_t{0.f};
#pragma unroll
    for (int k = 0; k < kStages; ++k) {
      const int off = 1024 * k + 64 * r + 16 * (quarter ^ ((r >> 2) & 3));
      part[k & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(smem + weights + off),
                                                            *reinterpret_cast<const bf16x8_t*>(smem + Lds::kRowsAt + off), part[k & 3], 0, 0, 0);
    }
    f32x4_t sum = ((part[0] + part[1]) + part[2]) + part[3];
    // register m of lane (r, quarter) is channel 4 quarter + m of token r
    const int gy = y0 + r / kPatchW, gx = x0 + r % kPatchW;
    if (gy < a.h && gx < a.w_cells) {
      sum[0] += bf16lo_to_f32(bias[0]), sum[1] += bf16hi_to_f32(bias[0]), sum[2] += bf16lo_to_f32(bias[1]), sum[3] += bf16hi_to_f32(bias[1]);
      *reinterpret_cast<u32x2_t*>(a.y + (image + (size_t)gy * a.w_cells + gx) * a.N + n) =
          u32x2_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
    }
  }
  // the other outputs, from the first column tile; at the end, since a wait for loads behind them would wait for them too
  if (blockIdx.x != 0) return;
  if (a.sum && in && cy >= 1 && cy <= kPatchH && cx >= 1 && cx <= kPatchW)
#pragma unroll
    for (int i = 0; i < NV; ++i) x[i].store(a.sum + at + 8 * kLanes * i);
  if (col < kPatchW && x0 + col < a.w_cells)
#pragma unroll
    for (int o = 0; o < kPatchH; ++o)
      if (y0 + o < a.h) *reinterpret_cast<u32x2_t*>(a.conv + (image + (size_t)(y0 + o) * a.w_cells + x0 + col) * C + ch) = conv[o];
}

template <int C>
int launch(const ConvLinearArgs& a, int B, hipStream_t stream) {
  static bool done[64] = {};
  if (!allow_lds((const void*)conv_linear_kernel<C>, ConvLinearLds<C>::kBytes, done)) return -5;
  hipLaunchKernelGGL(conv_linear_kernel<C>, dim3(a.N / kColumns, (unsigned)(B * a.down * a.across)), dim3(C == 192 ? 512 : 1024), ConvLinearLds<C>::kBytes, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace

static long long patches(int B, int h, int w) { return (long long)B * ((h + kPatchH - 1) / kPatchH) * ((w + kPatchW - 1) / kPatchW); }

// While the chip takes the workgroups at once (by LDS two to a CU at C 192, one at C 384).  us, separate kernels / this: C 192, N 640 280
// workgroups 7.7 / 6.9, 320 8.7 / 7.0, 420 8.1 / 7.3, 560 8.3 / 9.9; C 384, N 1280 140 8.5 / 6.9, 280 9.7 / 12.0, 420 9.7 / 12.8.
bool norm_conv_linear_supported(int B, int h, int w, int C, int N) {
  return (C == 192 || C == 384) && h <= 1024 && w <= 1024 && N % kColumns == 0 && patches(B, h, w) * (N / kColumns) <= (C == 192 ? 512 : 256);
}
int launch_norm_conv_linear(const void* x, const void* residual, const float* norm, const float* taps, const float* conv_bias, const void* w,
                            const void* bias, void* sum, void* conv, void* y, int B, int h, int width, int C, int N, float eps, int silu,
                            hipStream_t stream) {
  if (!norm_conv_linear_supported(B, h, width, C, N)) return -95;
  const ConvLinearArgs a{(const uint16_t*)x, (const uint16_t*)residual, norm, taps, conv_bias, (const uint16_t*)w, (const uint16_t*)bias,
                         (uint16_t*)sum, (uint16_t*)conv, (uint16_t*)y, h, width, N, (h + kPatchH - 1) / kPatchH, (width + kPatchW - 1) / kPatchW,
                         silu, eps};
  return C == 192 ? launch<192>(a, B, stream) : launch<384>(a, B, stream);
}

}  // namespace vig
