// y = x . W^T (+ bias) for bf16 rows, fp32 accumulation: the projections of a block, the classifier, and the patch
// embedding's 3x3 stride-2 convolution (its nine taps are nine row matrices: the contraction runs over (tap, channel) and a
// row's address depends on the tap).
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

struct GemmArgs {
  const uint16_t *x, *w, *bias;
  uint16_t* y;
  long long ldx, ldy;
  int M, N, K;
  int gh, gw, oh, ow, cin;  // convolution: input and output grid, input channels
};
enum FewForm { kRows, kTaps, kPair };  // row matrix; convolution; SwiGLU of the products with rows n and N + n of w

__device__ const u32x4_t kZeroRow = {0u, 0u, 0u, 0u};  // what a tap outside the grid reads

// Matrix row i of a weight tile holds this channel of its 32: accumulator register 4g+m of lane (r, h) is matrix row 8g+4h+m, so
// the lane ends with channels 16h .. 16h+15 of token r, 32 contiguous bytes.
__device__ __forceinline__ int channel_of_row(int r) { return 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3); }

// The row of input pixels behind output row m, and whether tap t of it lies inside the grid.
struct Pixel {
  int base, y, x;  // element offset of the image, input coordinates of tap (0, 0)
};
__device__ __forceinline__ Pixel pixel_of(const GemmArgs& a, int m) {
  const int per = a.oh * a.ow, b = m / per, p = m - b * per, oy = p / a.ow;
  return {b * a.gh * a.gw, 2 * oy - 1, 2 * (p - oy * a.ow) - 1};
}
__device__ __forceinline__ const uint16_t* tap_row(const GemmArgs& a, const Pixel& p, int tap) {
  const int ky = tap / 3, y = p.y + ky, x = p.x + tap - 3 * ky;
  const bool in = y >= 0 && y < a.gh && x >= 0 && x < a.gw;
  return in ? a.x + (size_t)(p.base + y * a.gw + x) * a.cin : nullptr;
}

constexpr int kStageK = 32;  // contraction elements per LDS stage: 64-byte row pieces

// ---------------------------------------------------------------------------
// Few rows: one workgroup per 32 x 32 tile of y, its waves splitting the contraction.  With a few hundred rows the chip
// is nearly empty and a product lasts as long as its longest chain of loads and matrix instructions: each wave streams its
// own stages through its own ring of LDS buffers (no barrier until the tiles are added), three in flight.  The stages go
// through LDS because a wave's operand fragment is 32 rows of 32 bytes: fetched straight into registers that is 32 separate
// requests an instruction (M 196, N 768, K 2048: 9.5 us).
// ---------------------------------------------------------------------------
constexpr int kFewBufs = 4;

template <int NW, FewForm FORM>
__global__ __launch_bounds__(64 * NW) void gemm_few_kernel(GemmArgs a) {
  constexpr bool TAPS = FORM == kTaps;
  constexpr int kMats = FORM == kPair ? 2 : 1, kLoads = 2 + 2 * kMats, kBuf = 1024 * kLoads;
  extern __shared__ __align__(16) char smem[];  // [wave][buffer][2 KB each: x rows, w rows, second w rows], then the waves' tiles
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  const int stages = a.K / kStageK, mine = (stages - wave + NW - 1) / NW;  // wave w takes stages w, w + NW, ..
  const int lrow = lane >> 2, place = lane & 3;
  const uint16_t *xp[2], *wp[2];
  Pixel px[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 16 * i + lrow, unit = place ^ ((row >> 2) & 3);
    const int m = min(m0 + row, a.M - 1), n = min(n0 + row, a.N - 1);
    if constexpr (TAPS) px[i] = pixel_of(a, m);
    xp[i] = a.x + (TAPS ? 0 : (size_t)m * a.ldx) + 8 * unit;
    wp[i] = a.w + (size_t)n * a.K + 8 * unit;
  }
  const size_t second = (size_t)a.N * a.K;
  char* const ring = smem + wave * (kFewBufs * kBuf);
  const uint32_t ring0 = lds_offset(smem) + wave * (kFewBufs * kBuf);
  const int tap_stages = TAPS ? a.cin / kStageK : 1;
  const auto fetch = [&](int at) {
    const int s = wave + NW * at;
    const uint32_t buf = ring0 + (at % kFewBufs) * kBuf;
    const int tap = TAPS ? s / tap_stages : 0, c = TAPS ? (s - tap * tap_stages) * kStageK : s * kStageK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint16_t* p = xp[i] + c;
      if constexpr (TAPS) {
        const uint16_t* row = tap_row(a, px[i], tap);
        p = row ? row + (xp[i] - a.x) + c : (const uint16_t*)&kZeroRow;
      }
      load_to_lds16(p, buf + 1024 * i);
      load_to_lds16(wp[i] + s * kStageK, buf + 2048 + 1024 * i);
      if constexpr (FORM == kPair) load_to_lds16(wp[i] + second + s * kStageK, buf + 4096 + 1024 * i);
    }
  };
  f32x16_t acc[kMats];
#pragma unroll
  for (int j = 0; j < kMats; ++j) acc[j] = f32x16_t{0.f};
#pragma unroll
  for (int s = 0; s < kFewBufs - 1; ++s)
    if (s < mine) fetch(s);
  for (int s = 0; s < mine; ++s) {
    const int ahead = min(mine - 1 - s, kFewBufs - 2);
    if (ahead >= 2) wait_vmem<2 * kLoads>();
    else if (ahead == 1) wait_vmem<kLoads>();
    else wait_vmem<0>();
    const char* buf = ring + (s % kFewBufs) * kBuf;
    bf16x8_t xf[2], wf[kMats][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int off = r * 64 + 16 * ((2 * k + h) ^ ((r >> 2) & 3));
      xf[k] = *reinterpret_cast<const bf16x8_t*>(buf + off);
#pragma unroll
      for (int j = 0; j < kMats; ++j) wf[j][k] = *reinterpret_cast<const bf16x8_t*>(buf + 2048 * (j + 1) + off);
    }
    // the buffer read in the step before is refilled: its reads have been waited for by the products that used them
    if (s + kFewBufs - 1 < mine) fetch(s + kFewBufs - 1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int j = 0; j < kMats; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j][k], xf[k], acc[j], 0, 0, 0);
  }
  // accumulator register 4g+m of lane (r, h) is channel 8g+4h+m of token r
  __syncthreads();
  float(*part)[kMats][32][36] = reinterpret_cast<float(*)[kMats][32][36]>(smem);
#pragma unroll
  for (int j = 0; j < kMats; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4_t*>(&part[wave][j][r][8 * g + 4 * h]) =
          f32x4_t{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += 64 * NW) {
    const int row = i >> 3, c = (i & 7) * 4;
    f32x4_t sum[kMats];
#pragma unroll
    for (int m = 0; m < kMats; ++m) {
      sum[m] = *reinterpret_cast<const f32x4_t*>(&part[0][m][row][c]);
#pragma unroll
      for (int k = 1; k < NW; ++k) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&part[k][m][row][c]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[m][j] += v[j];
      }
    }
    if (m0 + row < a.M && n0 + c < a.N) {  // N is a multiple of 8
      if (a.bias) {
        const u32x2_t b = *reinterpret_cast<const u32x2_t*>(a.bias + n0 + c);
        sum[0][0] += bf16lo_to_f32(b[0]), sum[0][1] += bf16hi_to_f32(b[0]), sum[0][2] += bf16lo_to_f32(b[1]), sum[0][3] += bf16hi_to_f32(b[1]);
      }
      if constexpr (FORM == kPair) {  // on the values the separate layer would have stored
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float g = bf16_to_f32(f32_to_bf16(sum[0][j])), u = bf16_to_f32(f32_to_bf16(sum[1][j]));
          sum[0][j] = g * u * sigmoidf_(g);
        }
      }
      *reinterpret_cast<u32x2_t*>(a.y + (size_t)(m0 + row) * a.ldy + n0 + c) =
          u32x2_t{pack_bf16x2(sum[0][0], sum[0][1]), pack_bf16x2(sum[0][2], sum[0][3])};
    }
  }
}

// ---------------------------------------------------------------------------
// Few rows: residual add, RMS norm and the SwiGLU layer behind it in one kernel, K = 48 NW.  A workgroup's 32 rows are whole rows of the
// contraction, so it makes their sums and norms itself (2 NW lanes a row; every column tile again, out of the L2, the first one
// stores the sums) while its weights arrive; a launch costs more than that.  us, norm and layer / this, rows x K -> I:
// 1 x 192 -> 512 4.5 / 3.2, 196 x 192 -> 512 5.0 / 3.4, 392 x 192 -> 512 5.1 / 3.6, 1 x 384 -> 1024 4.7 / 3.7, 256 x 384 -> 1024
// 5.7 / 4.4 (four waves 5.3: six octets of a row to a lane); other widths, and more rows than 256 workgroups take, keep the two.
// ---------------------------------------------------------------------------
struct NormPairArgs {
  const uint16_t *x, *residual, *w;  // rows [M, K], [M, K]; weights [2 N, K], gate rows first
  const float* norm;
  uint16_t *sum, *y;  // [M, K], [M, N]
  int M, N;
  float eps;
};
template <int NW>
__global__ __launch_bounds__(64 * NW) void gemm_norm_pair_kernel(NormPairArgs a) {
  constexpr int K = 48 * NW, NV = 3, kLanes = 2 * NW, kStages = K / kStageK, kX = 2048 * kStages;
  constexpr int kMats = NW == 4 ? 2 : 1, kMine = (kStages + 3) / 4, kMat = kMats * 2048;  // eight waves: four for the gate rows, four for the others
  __shared__ __align__(16) char smem[kX + NW * kMine * kMat > 36864 ? kX + NW * kMine * kMat : 36864];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  const int part0 = wave & 3, mat0 = wave >> 2;
  // ---- the weights of this wave's stages (part0, part0 + 4, ..), all of them under way at once ----
  const uint32_t w0 = lds_offset(smem) + kX + wave * (kMine * kMat);
#pragma unroll
  for (int at = 0; at < kMine; ++at) {
    const int s = part0 + 4 * at;
    if (s < kStages) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * i + (lane >> 2), unit = (lane & 3) ^ ((row >> 2) & 3);
        const uint16_t* wp = a.w + (size_t)(min(n0 + row, a.N - 1) + mat0 * a.N) * K + 8 * unit + s * kStageK;
        load_to_lds16(wp, w0 + at * kMat + 1024 * i);
        if constexpr (kMats == 2) load_to_lds16(wp + (size_t)a.N * K, w0 + at * kMat + 2048 + 1024 * i);
      }
    }
  }
  // ---- sums and norms, 8 or 4 rows a wave ----
  {
    const int row = threadIdx.x / kLanes, sub = threadIdx.x % kLanes, m = min(m0 + row, a.M - 1);
    const size_t base = (size_t)m * K;
    Raw8<uint16_t> x[NV], res[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) x[i].load(a.x + base + 8 * (sub + kLanes * i)), res[i].load(a.residual + base + 8 * (sub + kLanes * i));
    float s[NV][8], sq[NV] = {};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float b[8];
      x[i].unpack(s[i]);
      res[i].unpack(b);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[i][j] += b[j], sq[i] = __builtin_fmaf(s[i][j], s[i][j], sq[i]);
    }
    float ss = (sq[0] + sq[2]) + sq[1];  // the order of rmsnorm_kernel's wave, so its bits
#pragma unroll
    for (int d = kLanes / 2; d > 0; d >>= 1) ss += __shfl_xor(ss, d);
    const float rstd = 1.0f / sqrtf(ss / (float)K + a.eps);
    const bool keep = blockIdx.x == 0 && m0 + row < a.M;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int o = sub + kLanes * i;
      const f32x4_t wa = *reinterpret_cast<const f32x4_t*>(a.norm + 8 * o), wb = *reinterpret_cast<const f32x4_t*>(a.norm + 8 * o + 4);
      u32x4_t y, sum;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p = j < 2 ? wa[2 * j] : wb[2 * j - 4], q = j < 2 ? wa[2 * j + 1] : wb[2 * j - 3];
        y[j] = pack_bf16x2(s[i][2 * j] * rstd * p, s[i][2 * j + 1] * rstd * q);
        sum[j] = pack_bf16x2(s[i][2 * j], s[i][2 * j + 1]);
      }
      *reinterpret_cast<u32x4_t*>(smem + (o >> 2) * 2048 + row * 64 + 16 * ((o & 3) ^ ((row >> 2) & 3))) = y;
      if (keep) *reinterpret_cast<u32x4_t*>(a.sum + base + 8 * o) = sum;
    }
  }
  wait_vmem<0>();
  __syncthreads();
  f32x16_t acc[kMats];
#pragma unroll
  for (int j = 0; j < kMats; ++j) acc[j] = f32x16_t{0.f};
#pragma unroll
  for (int at = 0; at < kMine; ++at) {
    const int s = part0 + 4 * at;
    if (s < kStages) {
      const char* wbuf = smem + kX + wave * (kMine * kMat) + at * kMat;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int off = r * 64 + 16 * ((2 * k + h) ^ ((r >> 2) & 3));
        const bf16x8_t xf = *reinterpret_cast<const bf16x8_t*>(smem + s * 2048 + off);
#pragma unroll
        for (int j = 0; j < kMats; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(wbuf + 2048 * j + off), xf, acc[j], 0, 0, 0);
      }
    }
  }
  // accumulator register 4g+m of lane (r, h) is channel 8g+4h+m of token r
  __syncthreads();
  float(*part)[2][32][36] = reinterpret_cast<float(*)[2][32][36]>(smem);
#pragma unroll
  for (int j = 0; j < kMats; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4_t*>(&part[part0][mat0 + j][r][8 * g + 4 * h]) = f32x4_t{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
  __syncthreads();
  if (threadIdx.x >= 256) return;
  const int row = threadIdx.x >> 3, c = (threadIdx.x & 7) * 4;
  f32x4_t sum[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    sum[m] = *reinterpret_cast<const f32x4_t*>(&part[0][m][row][c]);
#pragma unroll
    for (int k = 1; k < 4; ++k) sum[m] += *reinterpret_cast<const f32x4_t*>(&part[k][m][row][c]);
  }
  if (m0 + row < a.M && n0 + c < a.N) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // on the values the separate layer would have stored
      const float g = bf16_to_f32(f32_to_bf16(sum[0][j])), u = bf16_to_f32(f32_to_bf16(sum[1][j]));
      sum[0][j] = g * u * sigmoidf_(g);
    }
    *reinterpret_cast<u32x2_t*>(a.y + (size_t)(m0 + row) * a.N + n0 + c) = u32x2_t{pack_bf16x2(sum[0][0], sum[0][1]), pack_bf16x2(sum[0][2], sum[0][3])};
  }
}

// ---------------------------------------------------------------------------
// Few rows: the mixer's epilogue (both head norms, the sigmoid blend, as in blend_linear_kernel) and o_proj in one kernel, K = N = 48 NW.
// One workgroup per 32 x 32 tile of the result: for a few hundred tokens the kernel that makes whole rows fills a handful of CUs, each
// with all the weights to fetch; here a CU has a sixth or a twelfth of them, and the blend is made once a column tile.
// ---------------------------------------------------------------------------
struct BlendFewArgs {
  const uint16_t *o, *loc, *glin;  // [B, H, L, 64]; [M, K]; rows of pitch ldg
  const float *wg, *wl;            // 64 each
  const uint16_t* w;               // [K, K]
  uint16_t *y, *kept;              // [M, K]; kept: the blended rows for a backward, or null
  long long ldg;
  int M, L, silu_out;
  float eps;
};
template <int NW>
__global__ __launch_bounds__(64 * NW) void gemm_blend_kernel(BlendFewArgs a) {
  constexpr int K = 48 * NW, NV = 3, H = K / 64, kLanes = 2 * NW, kStages = K / kStageK, kMine = (kStages + NW - 1) / NW, kX = 2048 * kStages;
  constexpr int kLds = kX + NW * kMine * 2048, kPart = NW * 32 * 36 * 4;
  __shared__ __align__(16) char smem[kLds > kPart ? kLds : kPart];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  // ---- the weights of this wave's stages (wave, wave + NW, ..), all of them under way at once ----
  const uint32_t w0 = lds_offset(smem) + kX + wave * (kMine * 2048);
#pragma unroll
  for (int at = 0; at < kMine; ++at) {
    const int s = wave + NW * at;
    if (s < kStages) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * i + (lane >> 2), unit = (lane & 3) ^ ((row >> 2) & 3);
        load_to_lds16(a.w + (size_t)(n0 + row) * K + 8 * unit + s * kStageK, w0 + at * 2048 + 1024 * i);
      }
    }
  }
  // ---- the blend, 8 or 4 rows a wave: a head is eight lanes' ----
  {
    const int row = threadIdx.x / kLanes, oct0 = threadIdx.x % kLanes, sub = lane & 7, m = min(m0 + row, a.M - 1);
    const unsigned b = (unsigned)m / (unsigned)a.L, l = (unsigned)m - b * (unsigned)a.L;
    const uint16_t* const o = a.o + ((size_t)b * H * a.L + l) * 64 + 8 * sub;
    Raw8<uint16_t> ro8[NV], rl8[NV], rg8[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int oct = oct0 + kLanes * i;
      ro8[i].load(o + (size_t)(oct >> 3) * a.L * 64);
      rl8[i].load(a.loc + (size_t)m * K + 8 * oct);
      rg8[i].load(a.glin + (size_t)m * a.ldg + 8 * oct);
    }
    float wg[8], wl[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) wg[j] = a.wg[8 * sub + j], wl[j] = a.wl[8 * sub + j];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float fo[8], fl[8], fg[8], e[8], so = 0.f, sl = 0.f;
      ro8[i].unpack(fo);
      rl8[i].unpack(fl);
      rg8[i].unpack(fg);
#pragma unroll
      for (int j = 0; j < 8; ++j) so += fo[j] * fo[j], sl += fl[j] * fl[j];
#pragma unroll
      for (int d = 1; d < 8; d <<= 1) so += __shfl_xor(so, d), sl += __shfl_xor(sl, d);
      const float ro = rsqrtf(so * (1.0f / 64.0f) + a.eps), rl = rsqrtf(sl * (1.0f / 64.0f) + a.eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sg = sigmoidf_(fg[j]);
        e[j] = fo[j] * ro * wg[j] * sg + fl[j] * rl * wl[j] * (1.f - sg);
      }
      if (a.silu_out) {
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = e[j] * sigmoidf_(e[j]);
      }
      u32x4_t y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = pack_bf16x2(e[2 * j], e[2 * j + 1]);
      const int oct = oct0 + kLanes * i;
      *reinterpret_cast<u32x4_t*>(smem + (oct >> 2) * 2048 + row * 64 + 16 * ((oct & 3) ^ ((row >> 2) & 3))) = y;
      if (a.kept && blockIdx.x == 0 && m0 + row < a.M) *reinterpret_cast<u32x4_t*>(a.kept + (size_t)m * K + 8 * oct) = y;
    }
  }
  wait_vmem<0>();
  __syncthreads();
  f32x16_t acc = f32x16_t{0.f};
#pragma unroll
  for (int at = 0; at < kMine; ++at) {
    const int s = wave + NW * at;
    if (s < kStages) {
      const char* wbuf = smem + kX + wave * (kMine * 2048) + at * 2048;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int off = r * 64 + 16 * ((2 * k + h) ^ ((r >> 2) & 3));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(wbuf + off),
                                                      *reinterpret_cast<const bf16x8_t*>(smem + s * 2048 + off), acc, 0, 0, 0);
      }
    }
  }
  // accumulator register 4g+m of lane (r, h) is channel 8g+4h+m of token r
  __syncthreads();
  float(*part)[32][36] = reinterpret_cast<float(*)[32][36]>(smem);
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<f32x4_t*>(&part[wave][r][8 * g + 4 * h]) = f32x4_t{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  if (threadIdx.x >= 256) return;
  const int row = threadIdx.x >> 3, c = (threadIdx.x & 7) * 4;
  f32x4_t sum = *reinterpret_cast<const f32x4_t*>(&part[0][row][c]);
#pragma unroll
  for (int k = 1; k < NW; ++k) sum += *reinterpret_cast<const f32x4_t*>(&part[k][row][c]);
  if (m0 + row < a.M)
    *reinterpret_cast<u32x2_t*>(a.y + (size_t)(m0 + row) * K + n0 + c) = u32x2_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
}

// ---------------------------------------------------------------------------
// Many rows: tiles of 64 MI x 64 NI by four waves of 32 MI x 32 NI each, operands through kBuffers LDS stages of 32
// contraction elements (64-byte row pieces, loaded directly to LDS; the 16-byte units of a piece are swapped by a quarter of the row
// number: the sixteen lanes served together read four rows that start in each bank quarter, and their units differ).
// ---------------------------------------------------------------------------
template <int MI, int NI, int BUFS, bool TAPS>
__global__ __launch_bounds__(256, (64 * (MI + NI) * 64 * BUFS <= 80 * 1024 ? 2 : 1)) void gemm_many_kernel(GemmArgs a, int tn, int tiles) {
  constexpr int TM = 64 * MI, TN = 64 * NI, kStage = (TM + TN) * 64;  // bytes
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // each XCD gets a run of consecutive tiles (all column tiles of a row block before the next one), so that its L2 serves the rows
  const int run = (tiles + 7) >> 3, at = ((int)blockIdx.x & 7) * run + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= run || at >= tiles) return;
  const int m0 = at / tn * TM, n0 = (at - at / tn * tn) * TN;
  const int nstage = a.K / kStageK;
  const uint32_t lds0 = lds_offset(smem);
  // a load covers 16 rows of 64 bytes; unit u of row w lies at place u ^ key
  const int lrow = lane >> 2, place = lane & 3;
  const uint16_t* xp[MI];
  Pixel px[MI];
  const uint16_t* wp[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = 16 * (wave * MI + i) + lrow, m = min(m0 + row, a.M - 1);
    const int unit = place ^ ((row >> 2) & 3);
    if constexpr (TAPS) px[i] = pixel_of(a, m);
    xp[i] = a.x + (TAPS ? 0 : (size_t)m * a.ldx) + 8 * unit;
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = 16 * (wave * NI + i) + lrow;  // matrix row: its channel is permuted inside its 32
    const int n = min(n0 + (row & ~31) + channel_of_row(row & 31), a.N - 1);
    wp[i] = a.w + (size_t)n * a.K + 8 * (place ^ ((row >> 2) & 3));
  }
  const int tap_stages = TAPS ? a.cin / kStageK : 1;
  const auto fetch = [&](int s) {
    const uint32_t buf = lds0 + (s % BUFS) * kStage;
    const int tap = TAPS ? s / tap_stages : 0, c = TAPS ? (s - tap * tap_stages) * kStageK : s * kStageK;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const uint16_t* p = xp[i] + c;
      if constexpr (TAPS) {
        const uint16_t* row = tap_row(a, px[i], tap);
        p = row ? row + (xp[i] - a.x) + c : (const uint16_t*)&kZeroRow;
      }
      load_to_lds16(p, buf + (wave * MI + i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) load_to_lds16(wp[i] + s * kStageK, buf + TM * 64 + (wave * NI + i) * 1024);
  };
  const int wm = (wave & 1) * 32 * MI, wn = (wave >> 1) * 32 * NI;
  int xoff[2], woff[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int unit = (2 * k + h) ^ ((r >> 2) & 3);
    xoff[k] = (wm + r) * 64 + 16 * unit;
    woff[k] = TM * 64 + (wn + r) * 64 + 16 * unit;
  }
  f32x16_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x16_t{0.f};
#pragma unroll
  for (int s = 0; s < BUFS - 1; ++s)
    if (s < nstage) fetch(s);
  for (int s = 0; s < nstage; ++s) {
    const int ahead = min(nstage - 1 - s, BUFS - 2);
    if (ahead >= 2) wait_vmem<2 * (MI + NI)>();
    else if (ahead == 1) wait_vmem<MI + NI>();
    else wait_vmem<0>();
    lds_barrier();
    if (s + BUFS - 1 < nstage) fetch(s + BUFS - 1);
    const char* buf = smem + (s % BUFS) * kStage;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      bf16x8_t xf[MI], wf[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) xf[i] = *reinterpret_cast<const bf16x8_t*>(buf + xoff[k] + 2048 * i);
#pragma unroll
      for (int j = 0; j < NI; ++j) wf[j] = *reinterpret_cast<const bf16x8_t*>(buf + woff[k] + 2048 * j);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], xf[i], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int c = n0 + wn + 32 * j + 16 * h;
    float bias[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) bias[e] = 0.f;
    if (a.bias) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
        if (c + 8 * p < a.N) {
          const u32x4_t b = *reinterpret_cast<const u32x4_t*>(a.bias + c + 8 * p);
#pragma unroll
          for (int e = 0; e < 4; ++e) bias[8 * p + 2 * e] = bf16lo_to_f32(b[e]), bias[8 * p + 2 * e + 1] = bf16hi_to_f32(b[e]);
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = m0 + wm + 32 * i + r;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        u32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(acc[i][j][8 * p + 2 * e] + bias[8 * p + 2 * e], acc[i][j][8 * p + 2 * e + 1] + bias[8 * p + 2 * e + 1]);
        if (m < a.M && c + 8 * p < a.N) *reinterpret_cast<u32x4_t*>(a.y + (size_t)m * a.ldy + c + 8 * p) = o;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// A layer of 192 columns followed by the residual add and the RMS norm behind it (a block's down projection and the next
// block's first norm): y = norm(sum), sum = residual + x . W^T, the product and the sum rounded to bf16 as the separate kernels
// store them.  A workgroup of eight waves makes 128 whole rows, 32 x 96 a wave, operands through three LDS stages of 64
// contraction elements (whole 128-byte lines); the finished rows lie in LDS, and a wave adds the residual (fetched before the
// barrier) and normalises sixteen of them with whole-row loads and stores.  So the product is not written and read again: 32768
// rows, K 512, 17 us where the library's product and the norm took 27 (100352 rows 55 / 70).  Bound by its waits: half of the
// waves' time goes to the stages' arrival and barriers (matrix pipe and LDS 14 % busy each).  (384 columns, K 1024: 63 to 67 us
// against 72 at 50176 rows, nothing gained in a model.)
// ---------------------------------------------------------------------------
struct NormArgs {
  const uint16_t *x, *w, *residual;
  const float* norm;
  uint16_t *y, *sum;
  int M, K;
  float eps;
};

constexpr int kNormStageK = 64;  // 128-byte row pieces

constexpr int kNormCols = 192, kNormRows = 128, kNormBufs = 3, kNormStage = (kNormRows + kNormCols) * 128;

__global__ __launch_bounds__(512, 2) void gemm_norm_kernel(NormArgs a) {
  constexpr int N = kNormCols, TM = kNormRows, BUFS = kNormBufs, kStage = kNormStage;
  constexpr int kX = TM / 64, kW = N / 64, kLoads = kX + kW, kPitch = 2 * N + 16;
  static_assert(TM * kPitch <= BUFS * kStage, "the rows fit");
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m0 = blockIdx.x * TM, nstage = a.K / kNormStageK;
  const uint32_t lds0 = lds_offset(smem);
  // a load covers eight rows; unit u of row w lies at place u ^ (w / 2 mod 8)
  const int lrow = lane >> 3, place = lane & 7;
  const uint16_t *xp[kX], *wp[kW];
#pragma unroll
  for (int i = 0; i < kX; ++i) {
    const int row = 8 * (wave * kX + i) + lrow;
    xp[i] = a.x + (size_t)min(m0 + row, a.M - 1) * a.K + 8 * (place ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    const int row = 8 * (wave * kW + i) + lrow;
    wp[i] = a.w + (size_t)((row & ~31) + channel_of_row(row & 31)) * a.K + 8 * (place ^ ((row >> 1) & 7));
  }
  const auto fetch = [&](int s) {
    const uint32_t buf = lds0 + (s % BUFS) * kStage;
#pragma unroll
    for (int i = 0; i < kX; ++i) load_to_lds16(xp[i] + s * kNormStageK, buf + (wave * kX + i) * 1024);
#pragma unroll
    for (int i = 0; i < kW; ++i) load_to_lds16(wp[i] + s * kNormStageK, buf + TM * 128 + (wave * kW + i) * 1024);
  };
  const int wm = (wave & 3) * 32, wn = (wave >> 2) * 96;
  f32x16_t acc[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) acc[j] = f32x16_t{0.f};
#pragma unroll
  for (int s = 0; s < BUFS - 1; ++s)
    if (s < nstage) fetch(s);
  for (int s = 0; s < nstage; ++s) {
    const int ahead = min(nstage - 1 - s, BUFS - 2);
    if (ahead >= 2) wait_vmem<2 * kLoads>();
    else if (ahead == 1) wait_vmem<kLoads>();
    else wait_vmem<0>();
    lds_barrier();
    if (s + BUFS - 1 < nstage) fetch(s + BUFS - 1);
    const char* buf = smem + (s % BUFS) * kStage;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const char* at = buf + r * 128 + 16 * ((2 * k + h) ^ ((r >> 1) & 7));
      const bf16x8_t xf = *reinterpret_cast<const bf16x8_t*>(at + wm * 128);
      bf16x8_t wf[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) wf[j] = *reinterpret_cast<const bf16x8_t*>(at + (TM + wn + 32 * j) * 128);
#pragma unroll
      for (int j = 0; j < 3; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], xf, acc[j], 0, 0, 0);
    }
  }
  const int oct = lane & 31, first = 16 * wave + h;  // half a wave takes a row
  const bool has = oct < N / 8;
  float weight[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) weight[j] = a.norm[8 * (has ? oct : 0) + j];
  u32x4_t res[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
    res[t] = *reinterpret_cast<const u32x4_t*>(a.residual + (size_t)min(m0 + first + 2 * t, a.M - 1) * N + 8 * (has ? oct : 0));
  lds_barrier();  // every wave is past the stages: their place becomes the rows'
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      u32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(acc[j][8 * p + 2 * e], acc[j][8 * p + 2 * e + 1]);
      *reinterpret_cast<u32x4_t*>(smem + (wm + r) * kPitch + 2 * (wn + 32 * j + 16 * h) + 16 * p) = o;
    }
  lds_barrier();
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int row = first + 2 * t;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(smem + row * kPitch + 16 * (has ? oct : 0));
    float sum[8], ss = 0.f;
    u32x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[j] = pack_bf16x2(bf16lo_to_f32(v[j]) + bf16lo_to_f32(res[t][j]), bf16hi_to_f32(v[j]) + bf16hi_to_f32(res[t][j]));
      sum[2 * j] = bf16lo_to_f32(o[j]), sum[2 * j + 1] = bf16hi_to_f32(o[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(sum[j], sum[j], ss);
    if (!has) ss = 0.f;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float rstd = 1.0f / sqrtf(ss / (float)N + a.eps);
    if (has && m0 + row < a.M) {
      const size_t at = (size_t)(m0 + row) * N + 8 * oct;
      *reinterpret_cast<u32x4_t*>(a.sum + at) = o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(sum[2 * j] * rstd * weight[2 * j], sum[2 * j + 1] * rstd * weight[2 * j + 1]);
      *reinterpret_cast<u32x4_t*>(a.y + at) = o;
    }
  }
}

int launch_norm(const NormArgs& a, hipStream_t stream) {
  constexpr int lds = kNormBufs * kNormStage;
  static bool done[64] = {};
  if (!allow_lds((const void*)gemm_norm_kernel, lds, done)) return -5;
  hipLaunchKernelGGL(gemm_norm_kernel, dim3((a.M + kNormRows - 1) / kNormRows), dim3(512), lds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

template <int MI, int NI, int BUFS, bool TAPS>
int launch_many(const GemmArgs& a, hipStream_t stream) {
  constexpr size_t lds = (size_t)(64 * MI + 64 * NI) * 64 * BUFS;
  static bool done[64] = {};
  if (!allow_lds((const void*)gemm_many_kernel<MI, NI, BUFS, TAPS>, lds, done)) return -5;
  const int tn = (a.N + 64 * NI - 1) / (64 * NI), tm = (a.M + 64 * MI - 1) / (64 * MI), tiles = tn * tm;
  hipLaunchKernelGGL((gemm_many_kernel<MI, NI, BUFS, TAPS>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), lds, stream, a, tn, tiles);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

template <int NW, FewForm FORM>
int launch_few(const GemmArgs& a, hipStream_t stream) {
  constexpr size_t lds = (size_t)NW * kFewBufs * (FORM == kPair ? 6144 : 4096);
  static bool done[64] = {};
  if (!allow_lds((const void*)gemm_few_kernel<NW, FORM>, lds, done)) return -5;
  hipLaunchKernelGGL((gemm_few_kernel<NW, FORM>), dim3((a.N + 31) / 32, (a.M + 31) / 32), dim3(64 * NW), lds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace

static long long tiles_of(const GemmArgs& a, int tm, int tn) { return (long long)((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn); }

// Where these kernels are the better choice (graph-captured runs on one MI355X; library times beside them):
//   up to 640 tiles of 32 x 32: gemm_few_kernel  (M 196: N 192 K 512 3.1 us against 17.2, N 1280 K 384 3.5 / 5.2,
//                               N 768 K 2048 4.7 / 6.9; past the line its operand traffic grows with the tile count)
//   up to 9 GFLOP:              64 x 64 tiles    (M 1568 N 1280 K 384 6.1 / 6.9; M 2500 N 384 K 1024 8.0 / 8.0)
//                               or, past 512 of them, 128 x 128 tiles  (M 3136 N 1280 K 384 8.3 / 9.1, with 64 x 64 tiles 10.3; M 9216 17.6 /
//                               21.8, 22.9; M 4000 N 768 K 768 11.1 / 10.1, 13.3; M 1000 N 4096 K 768 13.4 / 11.2, 19.7)
//                               (between 2 and 9 GFLOP the device alone takes 0.41 to 1.35 of the library's time, 0.93 in the mean of 80 drawn
//                               sizes; the worst where a second tile comes to some CUs only, M 5725 N 768 K 768 16.6 / 12.2, and at
//                               M 409 N 4096 K 768 11.3 / 8.7.  But the library's front end takes 22 us of host time a call, this one 4, and models
//                               of such products wait for the host.  Whole forward, ms, library past 2 GFLOP / this, and as captured graphs: ViG-B,
//                               images of 224 px, 2 1.30 / 1.00, 0.78 / 0.78; 6 1.72 / 1.10, 1.02 / 1.08; 12 1.93 / 1.39, 1.45 / 1.42; 20 1.94 / 1.88, 1.87 /
//                               1.87; 29 2.66 / 2.68, 2.63 / 2.66; ViG-S 16 0.83 / 0.80, 0.82 / 0.80; 40 1.20 / 1.18, 1.19 / 1.18)
//   K 384 or 192, N % 64 == 0, 16384 rows and fewer for some N (regs_rows): weights in registers (linear.hip)
//   K <= 256 with 512 tiles:    256 x 128 tiles  (M 65536 N 520 K 192: other column counts)
// Beyond that the library's products win (M 50176 N 1280 K 512 and longer contractions).
constexpr int kFewTiles = 640, kSmallTiles = 512;
// Rows from which the form with its weights in registers is the better one; the table for 16384 rows and up is beside
// launch_linear_regs.  Below, the library's time goes up and down with its choice of tiles, by up to two between neighbouring
// sizes (us, library / registers): K 192, N 640: 8192 rows 10.9 / 8.3, 9408 9.2 / 9.3, 14112 18.2 / 11.5; N 704 15.5 / 9.2 at 9408;
// N 512 and 768 2 % apart at worst; N 1024 13.5 / 14.1 at 12544.  K 384, N 2048: 8192 rows 19.3 / 20.5, 9216 29 / 23, 12544 43 / 28;
// N 1536: 10192 18.9 / 20.0, 10976 38 / 22, 14112 34 / 25; but N 1280: 12544 19.0 / 21.1, N 384 10.9 / 12.0.  The lines
// lie where no measured size loses more than 2 %.
static long long regs_rows(int N, int K) {
  if (K == 192) return N >= 512 && N <= 768 ? 8192 : 16384;
  return N >= 1536 ? 10752 : 16384;
}
static bool regs_preferred(long long M, int N, int K) { return linear_regs_supported(K, N) && M >= regs_rows(N, K); }
static bool short_k_many(const GemmArgs& a) { return a.K <= 256 && tiles_of(a, 256, 128) >= 512; }

bool linear_preferred(long long M, int N, int K) {
  if (M <= 0 || M > 0x7fffffffLL - 256 || N <= 0 || K <= 0 || N % 8 || K % kStageK) return false;
  GemmArgs a{};
  a.M = (int)M, a.N = N, a.K = K;
  return regs_preferred(M, N, K) || tiles_of(a, 32, 32) <= kFewTiles || 2.0 * M * N * K <= 9e9 || short_k_many(a);
}

int launch_linear(const void* x, long long ldx, const void* w, const void* bias, void* y, long long ldy, long long M, int N, int K,
                  hipStream_t stream) {
  if (M > 0x7fffffffLL - 256 || N % 8 || K % kStageK) return -95;
  const GemmArgs a{(const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, (uint16_t*)y, ldx, ldy, (int)M, N, K, 0, 0, 0, 0, 0};
  if (tiles_of(a, 64, 64) > 0x7fffffffLL - 8) return -95;
  if (regs_preferred(M, N, K) && ldx == K && ldy == N) return launch_linear_regs(x, w, bias, y, M, N, K, stream);
  if (tiles_of(a, 32, 32) <= kFewTiles) return launch_few<4, kRows>(a, stream);
  if (short_k_many(a)) return launch_many<4, 2, 3, false>(a, stream);
  if (tiles_of(a, 64, 64) > kSmallTiles) return launch_many<2, 2, 3, false>(a, stream);
  return launch_many<1, 1, 4, false>(a, stream);
}

// SwiGLU of a linear layer with the gate rows first, tiles of 32 x 32 results, while there is at most one for a CU.  Past that
// the form with its weights in registers (linear.hip) is the better one: 196 rows, K 192, I 512 3.1 us against 4.5; 392 rows
// 3.1 / 4.0, 588 4.5 / 4.1; K 384, I 1024: 196 rows 3.5 / 5.4, 392 5.3 / 5.3.
bool few_swiglu(long long T, int K, int I) {
  if (T <= 0 || T > 0x7fffffffLL - 256 || K <= 0 || K % kStageK || I <= 0 || I % 32) return false;
  return (T + 31) / 32 * (I / 32) <= 256;
}
int launch_few_swiglu(const void* x, const void* w, void* y, long long T, int K, int I, hipStream_t stream) {
  if (!few_swiglu(T, K, I)) return -95;
  const GemmArgs a{(const uint16_t*)x, (const uint16_t*)w, nullptr, (uint16_t*)y, K, I, (int)T, I, K, 0, 0, 0, 0, 0};
  return launch_few<4, kPair>(a, stream);
}

// The same with the residual add and the RMS norm in front.
bool norm_swiglu_supported(long long T, int K, int I) { return (K == 192 || K == 384) && few_swiglu(T, K, I); }
int launch_norm_swiglu(const void* x, const void* residual, const float* norm, const void* w, void* sum, void* y, long long T, int K, int I,
                       float eps, hipStream_t stream) {
  if (!norm_swiglu_supported(T, K, I)) return -95;
  const NormPairArgs a{(const uint16_t*)x, (const uint16_t*)residual, (const uint16_t*)w, norm, (uint16_t*)sum, (uint16_t*)y, (int)T, I, eps};
  const dim3 grid(I / 32, (unsigned)((T + 31) / 32));
  if (K == 192) hipLaunchKernelGGL(gemm_norm_pair_kernel<4>, grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(gemm_norm_pair_kernel<8>, grid, dim3(512), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// The mixer's epilogue and o_proj of few rows (checked by launch_blend_linear), while there is a tile for a CU.  us, whole rows a
// workgroup / this: C 192 196 rows 4.65 / 3.47, 1176 4.72 / 3.66, 1568 (294 tiles) 4.73 / 4.40, 2548 4.79 / 4.72; C 384 196 rows
// 7.44 / 4.73 (four waves 5.17), 588 7.51 / 4.92, 784 (300 tiles, four waves) 7.48 / 7.09, 1176 7.54 / 7.41.
bool few_blend_linear(long long T, int C) { return (C == 192 || C == 384) && (T + 31) / 32 * (C / 32) <= 256; }
int launch_few_blend_linear(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l, const void* W, void* out,
                            void* kept, long long T, int L, int C, long long ldg, float eps, int silu_out, hipStream_t stream) {
  const BlendFewArgs a{(const uint16_t*)o, (const uint16_t*)loc, (const uint16_t*)glin, w_g, w_l, (const uint16_t*)W, (uint16_t*)out,
                       (uint16_t*)kept, ldg, (int)T, L, silu_out, eps};
  const dim3 grid(C / 32, (unsigned)((T + 31) / 32));
  if (C == 192) hipLaunchKernelGGL(gemm_blend_kernel<4>, grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(gemm_blend_kernel<8>, grid, dim3(512), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// The convolution library took 12 to 138 us where these take 4.3 to 96: B 1, 28 x 28 x 96 -> 192 4.3 / 12.3; B 32, 192 -> 384
// 26 / 54; B 256 96 / 137.  Long contractions (27 to 108 stages) want eight waves a tile while tiles are fewer than CUs.
// Past 640 tiles of 32 x 32 the tile of least estimated time: what it takes alone on its CU a stage, two of them on one CU `pair`
// times that (64 x 64: five fit, half a tile's time each from the third on).  28 x 28 inputs, us, "64 x 64 tiles, 128 x 192 once there is one
// for every CU" / this: 192 -> 384 32 images 26.5 / 23.8, 64 42.4 / 31.4, 96 46.8 / 39.4; 384 -> 768 24 61.6 / 54, 32 81.8 / 55.6, 40 93 / 65, 48
// 85.8 / 72.8, 96 152 / 143; 96 -> 192 96 20.1 / 18.2, 128 24.1 / 19.2; the rest as before.
struct TapsTile {
  int tm, tn;
  float stage, pair;
};
constexpr TapsTile kTapsTiles[] = {{64, 64, 0.26f, 1.23f}, {64, 192, 0.37f, 1.35f}, {128, 128, 0.47f, 1.3f}, {128, 192, 0.535f, 1.42f}};
static int taps_tile(const GemmArgs& a) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < 4; ++i) {
    const TapsTile& t = kTapsTiles[i];
    const long long deep = (tiles_of(a, t.tm, t.tn) + 255) / 256;
    const float rounds = i == 0 && deep > 2 ? 0.5f * deep : (deep >> 1) * t.pair + (deep & 1);
    if (i == 0 || t.stage * rounds < least) least = t.stage * rounds, best = i;
  }
  return best;
}
int launch_conv3x3s2(const void* x, const void* w, void* y, int B, int H, int W, int Cin, int Cout, hipStream_t stream) {
  const int oh = (H + 1) / 2, ow = (W + 1) / 2;
  const long long M = (long long)B * oh * ow;
  if (Cin % kStageK || Cout % 8 || M > 0x7fffffffLL - 256 || (long long)B * H * W > 0x7fffffffLL) return -95;
  const GemmArgs a{(const uint16_t*)x, (const uint16_t*)w, nullptr, (uint16_t*)y, 0, Cout, (int)M, Cout, 9 * Cin, H, W, oh, ow, Cin};
  if (tiles_of(a, 64, 64) > 0x7fffffffLL - 8) return -95;
  if (tiles_of(a, 32, 32) <= 256) return launch_few<8, kTaps>(a, stream);
  if (tiles_of(a, 32, 32) <= kFewTiles) return launch_few<4, kTaps>(a, stream);
  switch (taps_tile(a)) {
    case 1: return launch_many<1, 3, 4, true>(a, stream);
    case 2: return launch_many<2, 2, 4, true>(a, stream);
    case 3: return launch_many<2, 3, 4, true>(a, stream);
  }
  return launch_many<1, 1, 4, true>(a, stream);
}

bool linear_norm_supported(long long M, int N, int K) {
  return N == kNormCols && M > 0 && M <= 0x7fffffffLL - 256 && K > 0 && K % kNormStageK == 0;
}
int launch_linear_norm(const void* x, const void* w, const void* residual, const float* norm, void* y, void* sum, long long M, int N,
                       int K, float eps, hipStream_t stream) {
  if (!linear_norm_supported(M, N, K)) return -95;
  return launch_norm({(const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)residual, norm, (uint16_t*)y, (uint16_t*)sum, (int)M, K, eps},
                     stream);
}

}  // namespace vig
