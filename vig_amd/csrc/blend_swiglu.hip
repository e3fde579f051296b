// Few rows of 192 channels: the middle of a block in one kernel.  Both head norms and the sigmoid blend, o_proj, residual add, RMS norm
// and the SwiGLU layer behind it (classification/models/vig.py:447-461,606-608,492-497).
//
// The norm wants whole rows of o_proj, the layer behind it many columns: a workgroup has 16 rows and 64 of the SwiGLU's columns, and makes
// the blend, all of o_proj (72 MFMAs of 16 x 16 x 32) and the norm of its rows itself, out of the L2; the first column tile stores the
// sums.  Everything it reads is under way from the first instruction, straight to LDS, in the order in which it is waited for (rows, o_proj's
// weights, the layer's); what bounds it is that chain: 160 KB of LDS filled at a CU's rate, then five short steps with a barrier each.
// Every product is four sums over every fourth stage, added up in the order of the kernels it stands for (gemm_blend_kernel, gemm_norm_pair_kernel),
// so their bits.  us, those two / this, I 512: 1 row 7.0 / 5.4, 49 7.4 / 5.5, 196 7.6 / 5.6, 392 7.7 / 5.8, 512 (256 workgroups) 7.9 / 6.1.
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

constexpr int kC = 192, kRows = 16, kCols = 64, kSteps = kC / 32, kUnit = 1024;  // a unit: 16 rows of 64 bytes
constexpr int kOct = kC / 8, kItems = kRows * kOct;                               // channel octets of a row, of the tile

struct BlendSwigluArgs {
  const uint16_t *o, *loc, *glin;  // [B, H, L, 64]; [M, C]; rows of pitch ldg
  const float *wg, *wl;            // 64 each
  const uint16_t *wo, *residual;   // [C, C]; [M, C]
  const float* norm;               // [C]
  const uint16_t* w;               // [2 N, C], gate rows first
  uint16_t *sum, *y;               // [M, C], [M, N]
  long long ldg;
  int M, N, L, silu_out;
  float eps, norm_eps;
};

// byte offsets in LDS
constexpr int kWo = 0, kW = kWo + kC * kC * 2, kIn = kW + 2 * kCols * kC * 2, kSmall = kIn + 4 * kItems * 16, kX = kSmall + 2048,
              kA = kX + kRows * kC * 2, kMidLds = kA + kRows * kC * 2;
static_assert(kMidLds <= 160 * 1024, "one workgroup to a CU");

// place of octet o of row r in a tile of units (unit o / 4), 16-byte places swapped as in gemm.hip
__device__ __forceinline__ int place(int r, int o) { return (o >> 2) * kUnit + r * 64 + 16 * ((o & 3) ^ ((r >> 2) & 3)); }

__global__ __launch_bounds__(512) void blend_swiglu_kernel(BlendSwigluArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 15, quarter = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m0 = blockIdx.y * kRows, n0 = blockIdx.x * kCols;
  const uint32_t lds0 = lds_offset(smem);
  // ---- everything under way: rows (waves 0 to 5, a thread an octet), small weights (6, 7); weights, 9 and 6 units a wave ----
  const int row = (int)threadIdx.x / kOct, oct = (int)threadIdx.x - row * kOct;
  if (wave < kItems / 64) {
    const int m = min(m0 + row, a.M - 1);
    const unsigned b = (unsigned)m / (unsigned)a.L, l = (unsigned)m - b * (unsigned)a.L;
    const uint32_t in = lds0 + kIn + 1024 * wave;
    load_to_lds16(a.o + (((size_t)b * (kC / 64) + (oct >> 3)) * a.L + l) * 64 + 8 * (oct & 7), in);
    load_to_lds16(a.loc + (size_t)m * kC + 8 * oct, in + 16 * kItems);
    load_to_lds16(a.glin + (size_t)m * a.ldg + 8 * oct, in + 32 * kItems);
    load_to_lds16(a.residual + (size_t)m * kC + 8 * oct, in + 48 * kItems);
  } else if (wave == 6) {  // both head norms' weights, 256 bytes each, and again
    load_to_lds16((lane & 16 ? a.wl : a.wg) + 4 * (lane & 15), lds0 + kSmall);
  } else {  // the norm's, 768 bytes
    load_to_lds16(a.norm + 4 * min(lane, 47), lds0 + kSmall + 1024);
  }
  const int wrow = lane >> 2, wunit = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
  for (int i = 0; i < 9; ++i) {  // unit u: rows 16 (u / 6) .. of o_proj's weights, stage u % 6
    const int u = 9 * wave + i, t = u / kSteps, s = u - t * kSteps;
    load_to_lds16(a.wo + (size_t)(16 * t + wrow) * kC + 8 * wunit + 32 * s, lds0 + kWo + kUnit * u);
  }
#pragma unroll
  for (int i = 0; i < kSteps; ++i)  // waves 0 to 3: gate rows of column tile `wave`, 4 to 7: the others
    load_to_lds16(a.w + (size_t)((wave >> 2) * a.N + n0 + 16 * (wave & 3) + wrow) * kC + 8 * wunit + 32 * i, lds0 + kW + kUnit * (kSteps * wave + i));
  wait_vmem<15>();
  lds_barrier();
  // ---- the blend: a head is eight lanes' ----
  if (wave < kItems / 64) {
    const char* in = smem + kIn + 16 * threadIdx.x;
    Raw8<uint16_t> ro8, rl8, rg8;
    ro8.a = *reinterpret_cast<const u32x4_t*>(in);
    rl8.a = *reinterpret_cast<const u32x4_t*>(in + 16 * kItems);
    rg8.a = *reinterpret_cast<const u32x4_t*>(in + 32 * kItems);
    const float* wg = reinterpret_cast<const float*>(smem + kSmall) + 8 * (oct & 7);
    float fo[8], fl[8], fg[8], e[8], so = 0.f, sl = 0.f;
    ro8.unpack(fo), rl8.unpack(fl), rg8.unpack(fg);
#pragma unroll
    for (int j = 0; j < 8; ++j) so += fo[j] * fo[j], sl += fl[j] * fl[j];
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) so += __shfl_xor(so, d), sl += __shfl_xor(sl, d);
    const float ro = rsqrtf(so * (1.0f / 64.0f) + a.eps), rl = rsqrtf(sl * (1.0f / 64.0f) + a.eps);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float sg = sigmoidf_(fg[j]);
      e[j] = fo[j] * ro * wg[j] * sg + fl[j] * rl * wg[64 + j] * (1.f - sg);
    }
    if (a.silu_out) {
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = e[j] * sigmoidf_(e[j]);
    }
    u32x4_t v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = pack_bf16x2(e[2 * j], e[2 * j + 1]);
    *reinterpret_cast<u32x4_t*>(smem + kX + place(row, oct)) = v;
  }
  wait_vmem<6>();
  lds_barrier();
  // ---- o_proj: column tiles `wave` and, for the first four waves, 8 + wave ----
  for (int t = wave; t < kC / 16; t += 8) {
    f32x4_t part[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) part[k] = f32x4_t{0.f};
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int off = 64 * r + 16 * (quarter ^ ((r >> 2) & 3));
      part[s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(smem + kWo + kUnit * (kSteps * t + s) + off),
                                                            *reinterpret_cast<const bf16x8_t*>(smem + kX + kUnit * s + off), part[s & 3], 0, 0, 0);
    }
    const f32x4_t acc = ((part[0] + part[1]) + part[2]) + part[3];
    // register m of lane (r, quarter) is channel 4 quarter + m of row r
    *reinterpret_cast<u32x2_t*>(smem + kA + 2 * (kC * r + 16 * t + 4 * quarter)) = u32x2_t{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
  }
  lds_barrier();
  // ---- sums and norms: eight lanes a row, three octets each ----
  u32x4_t kept[3];
  const int nrow = threadIdx.x >> 3, sub = threadIdx.x & 7;
  if (wave < kRows / 8) {
    float s[3][8], sq[3] = {};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int at = kOct * nrow + sub + 8 * i;
      Raw8<uint16_t> x, res;
      x.a = *reinterpret_cast<const u32x4_t*>(smem + kA + 16 * at);
      res.a = *reinterpret_cast<const u32x4_t*>(smem + kIn + 48 * kItems + 16 * at);
      float b[8];
      x.unpack(s[i]), res.unpack(b);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[i][j] += b[j], sq[i] = __builtin_fmaf(s[i][j], s[i][j], sq[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j) kept[i][j] = pack_bf16x2(s[i][2 * j], s[i][2 * j + 1]);
    }
    float ss = (sq[0] + sq[2]) + sq[1];  // the order of rmsnorm_kernel's wave, so its bits
#pragma unroll
    for (int d = 4; d > 0; d >>= 1) ss += __shfl_xor(ss, d);
    const float rstd = 1.0f / sqrtf(ss / (float)kC + a.norm_eps);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int o = sub + 8 * i;
      const float* weight = reinterpret_cast<const float*>(smem + kSmall + 1024) + 8 * o;
      u32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = pack_bf16x2(s[i][2 * j] * rstd * weight[2 * j], s[i][2 * j + 1] * rstd * weight[2 * j + 1]);
      *reinterpret_cast<u32x4_t*>(smem + kX + place(nrow, o)) = v;
    }
  }
  wait_vmem<0>();
  lds_barrier();
  // ---- gate and up products of 16 columns a wave ----
  if (wave < kCols / 16) {
    f32x4_t gates[4], ups[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) gates[k] = ups[k] = f32x4_t{0.f};
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int off = 64 * r + 16 * (quarter ^ ((r >> 2) & 3));
      const bf16x8_t xf = *reinterpret_cast<const bf16x8_t*>(smem + kX + kUnit * s + off);
      gates[s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(smem + kW + kUnit * (kSteps * wave + s) + off), xf, gates[s & 3], 0, 0, 0);
      ups[s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(smem + kW + kUnit * (kSteps * (wave + 4) + s) + off), xf, ups[s & 3], 0, 0, 0);
    }
    const f32x4_t gate = ((gates[0] + gates[1]) + gates[2]) + gates[3], up = ((ups[0] + ups[1]) + ups[2]) + ups[3];
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // on the values the separate layer would have stored
      const float g = bf16_to_f32(f32_to_bf16(gate[j])), u = bf16_to_f32(f32_to_bf16(up[j]));
      v[j] = g * u * sigmoidf_(g);
    }
    if (m0 + r < a.M)
      *reinterpret_cast<u32x2_t*>(a.y + (size_t)(m0 + r) * a.N + n0 + 16 * wave + 4 * quarter) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
  if (blockIdx.x == 0 && wave < kRows / 8 && m0 + nrow < a.M) {
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4_t*>(a.sum + (size_t)(m0 + nrow) * kC + 8 * (sub + 8 * i)) = kept[i];
  }
}

}  // namespace

bool blend_swiglu_supported(long long T, int C, int N) {
  return C == kC && N > 0 && N % kCols == 0 && T > 0 && T <= 0x7fffffffLL - 256 && (T + kRows - 1) / kRows * (N / kCols) <= 256;
}
int launch_blend_swiglu(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l, const void* w_out,
                        const void* residual, const float* norm, const void* w, void* sum, void* y, long long T, int L, int C, int N,
                        long long ldg, float eps, int silu_out, float norm_eps, hipStream_t stream) {
  if (!blend_swiglu_supported(T, C, N)) return -95;
  static bool done[64] = {};
  if (!allow_lds((const void*)blend_swiglu_kernel, kMidLds, done)) return -5;
  const BlendSwigluArgs a{(const uint16_t*)o, (const uint16_t*)loc, (const uint16_t*)glin, w_g, w_l, (const uint16_t*)w_out, (const uint16_t*)residual,
                          norm, (const uint16_t*)w, (uint16_t*)sum, (uint16_t*)y, ldg, (int)T, N, L, silu_out, eps, norm_eps};
  hipLaunchKernelGGL(blend_swiglu_kernel, dim3(N / kCols, (unsigned)((T + kRows - 1) / kRows)), dim3(512), kMidLds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace vig
