// Elementwise / stencil neighbours of the GLA op: direction-wise gate preparation,
// the 3x3 depthwise stencil on the token grid, the sigmoid locality gate and the
// RMS-norm blend epilogue.  All are HBM-bound: each element is read once with
// 16-byte (bf16 x8) or 16-byte (f32 x4) accesses along the channel dimension and
// written once; stencil neighbours come from L1/L2.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace vig {

// ---------------------------------------------------------------------------
// vector-of-8 channel access (one 16-byte transaction for bf16, two for f32)
// ---------------------------------------------------------------------------
template <typename T> struct Vec8;
template <> struct Vec8<uint16_t> {
  static __device__ __forceinline__ void load(const uint16_t* p, float (&x)[8]) {
    const u32x4_t r = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = bf16lo_to_f32(r[i]);
      x[2 * i + 1] = bf16hi_to_f32(r[i]);
    }
  }
  static __device__ __forceinline__ void store(uint16_t* p, const float (&x)[8]) {
    u32x4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
    *reinterpret_cast<u32x4_t*>(p) = r;
  }
};
template <> struct Vec8<float> {
  static __device__ __forceinline__ void load(const float* p, float (&x)[8]) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p);
    const f32x4_t b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a[i];
      x[4 + i] = b[i];
    }
  }
  static __device__ __forceinline__ void store(float* p, const float (&x)[8]) {
    f32x4_t a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = x[i];
      b[i] = x[4 + i];
    }
    *reinterpret_cast<f32x4_t*>(p) = a;
    *reinterpret_cast<f32x4_t*>(p + 4) = b;
  }
};

// ---------------------------------------------------------------------------
// direction-wise gate preparation
//   in  [B, L, 2*H*Dk]  ->  out [2, B, H, L, Dk],  logsigmoid(x) * inv_norm, clamp
// HBM-bound.  A thread takes N octets of the rows, their loads under way together.  Measured (us, before: a workgroup for 32 tokens
// of an image, a wave for every fourth): fp32 400 x 768 channels 8.9, now 2.6; 4704 x 768 11.2, now 6.1; 25088 x 384 14.4, now 13.8.
// ---------------------------------------------------------------------------
template <typename TI, typename TO, int N>
__global__ __launch_bounds__(256) void dirgate_kernel(const TI* __restrict__ in, TO* __restrict__ out, int B, int L,
                                                       int H, int Dk, float inv_norm, float clamp_min, int use_clamp, int tokens) {
  const int nv = 2 * H * Dk / 8;         // channel octets per token row
  const int dk8 = Dk >> 3;
  const OctetRows rows(B, L, nv, tokens);
  const TI* src = in + (size_t)blockIdx.x * tokens * nv * 8;
  for (int x0 = threadIdx.x; x0 < rows.n; x0 += 256 * N) {
    Raw8<TI> raw[N];
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (x0 + 256 * u < rows.n) raw[u].load(src + (size_t)(x0 + 256 * u) * 8);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (x0 + 256 * u >= rows.n) break;
      const Octet at(rows, x0 + 256 * u, nv, L);
      const int head = at.cv / dk8, d8 = at.cv - head * dk8, dir = head >= H, hh = head - dir * H;
      float x[8];
      raw[u].unpack(x);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // logsigmoid(x) = min(x,0) - log(1 + exp(-|x|)); hardware exp/log are accurate to ~1e-7 absolute here
        float yv = logsigmoidf_(x[j]);
        yv *= inv_norm;
        if (use_clamp) yv = fmaxf(yv, clamp_min);
        x[j] = yv;
      }
      Vec8<TO>::store(out + ((((size_t)dir * B + at.b) * H + hh) * L + at.l) * (size_t)Dk + (size_t)d8 * 8, x);
    }
  }
}

// Backward of the gate preparation: d_in[b, l, c] = d_out[dir, b, h, l, d] * inv_norm * sigmoid(-x), zero where the
// forward clamped (x = in[b, l, c]; d/dx logsigmoid(x) = sigmoid(-x)).
template <typename TI, typename TO, int N>
__global__ __launch_bounds__(256) void dirgate_bwd_kernel(const TI* __restrict__ in, const TO* __restrict__ d_out,
                                                           TI* __restrict__ d_in, int B, int L, int H, int Dk,
                                                           float inv_norm, float clamp_min, int use_clamp, int tokens) {
  const int nv = 2 * H * Dk / 8;
  const int dk8 = Dk >> 3;
  const OctetRows rows(B, L, nv, tokens);
  const size_t first = (size_t)blockIdx.x * tokens * nv * 8;
  for (int x0 = threadIdx.x; x0 < rows.n; x0 += 256 * N) {
    Raw8<TI> raw[N];
    Raw8<TO> grad[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (x0 + 256 * u >= rows.n) break;
      const Octet at(rows, x0 + 256 * u, nv, L);
      const int head = at.cv / dk8, d8 = at.cv - head * dk8, dir = head >= H, hh = head - dir * H;
      raw[u].load(in + first + (size_t)(x0 + 256 * u) * 8);
      grad[u].load(d_out + ((((size_t)dir * B + at.b) * H + hh) * L + at.l) * (size_t)Dk + (size_t)d8 * 8);
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (x0 + 256 * u >= rows.n) break;
      float x[8], g[8];
      raw[u].unpack(x);
      grad[u].unpack(g);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool clamped = use_clamp && logsigmoidf_(x[j]) * inv_norm < clamp_min;
        x[j] = clamped ? 0.f : g[j] * inv_norm * sigmoidf_(-x[j]);
      }
      Vec8<TI>::store(d_in + first + (size_t)(x0 + 256 * u) * 8, x);
    }
  }
}

int launch_dirgate_bwd(const void* in, const void* d_out, void* d_in, int B, int L, int H, int Dk, float inv_norm,
                       float clamp_min, int in_dtype, int out_dtype, hipStream_t stream) {
  const int use_clamp = clamp_min == clamp_min;  // NaN disables
  if (B > 65535 || !octet_rows_ok(B, L)) return -22;
  const int nv = 2 * H * Dk / 8, each = octets_each((long long)B * L, nv);
  int tokens = octet_tokens(nv, each);
  const dim3 grid(octet_grid((long long)B * L, tokens)), block(256);
#define VIG_DGB_CASE(TI, TO)                                                                                                   \
  hipLaunchKernelGGL((each == 4 ? dirgate_bwd_kernel<TI, TO, 4> : dirgate_bwd_kernel<TI, TO, 1>), grid, block, 0, stream,     \
                     (const TI*)in, (const TO*)d_out, (TI*)d_in, B, L, H, Dk, inv_norm, clamp_min, use_clamp, tokens)
  if (in_dtype == 0 && out_dtype == 0) VIG_DGB_CASE(float, float);
  else if (in_dtype == 0 && out_dtype == 1) VIG_DGB_CASE(float, uint16_t);
  else if (in_dtype == 1 && out_dtype == 0) VIG_DGB_CASE(uint16_t, float);
  else VIG_DGB_CASE(uint16_t, uint16_t);
#undef VIG_DGB_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

template <typename TI, typename TO>
static int launch_dirgate_t(const void* in, void* out, int B, int L, int H, int Dk, float inv_norm,
                            float clamp_min, hipStream_t stream) {
  const int use_clamp = clamp_min == clamp_min;  // NaN disables
  if (B > 65535 || !octet_rows_ok(B, L)) return -22;
  const int nv = 2 * H * Dk / 8, each = octets_each((long long)B * L, nv);
  int tokens = octet_tokens(nv, each);
  const dim3 grid(octet_grid((long long)B * L, tokens)), block(256);
  hipLaunchKernelGGL((each == 4 ? dirgate_kernel<TI, TO, 4> : dirgate_kernel<TI, TO, 1>), grid, block, 0, stream, (const TI*)in, (TO*)out, B, L, H, Dk, inv_norm, clamp_min, use_clamp, tokens);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_dirgate(const void* in, void* out, int B, int L, int H, int Dk, float inv_norm, float clamp_min,
                   int in_dtype, int out_dtype, hipStream_t stream) {
  if (in_dtype == 0 && out_dtype == 0) return launch_dirgate_t<float, float>(in, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  if (in_dtype == 0 && out_dtype == 1) return launch_dirgate_t<float, uint16_t>(in, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  if (in_dtype == 1 && out_dtype == 0) return launch_dirgate_t<uint16_t, float>(in, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  return launch_dirgate_t<uint16_t, uint16_t>(in, out, B, L, H, Dk, inv_norm, clamp_min, stream);
}

// ---------------------------------------------------------------------------
// direction-wise gate preparation with the second (rank -> 2*H*Dk) layer of the gate projection inside:
//   low [B, L, 16] (rows ld elements apart), w1 [2*H*Dk, 16], b1 [2*H*Dk]
//   x = low . w1^T + b1, rounded to the storage type of `low` (what the separate layer would have stored),
//   out [2, B, H, L, Dk] = logsigmoid(x) * inv_norm, clamp
// The rank-16 product is 16 multiply-adds per output, far below what the output write costs, so the [B, L, 2*H*Dk]
// intermediate never goes to memory.  One workgroup owns 32 consecutive tokens of one batch element; their low-rank
// rows sit in LDS as f32; a thread keeps the 8x16 weights of one channel octet in registers for all its tokens.
// ---------------------------------------------------------------------------
constexpr int kGateRank = 16;

template <typename T> struct Stored;  // value after a round trip through the storage type
template <> struct Stored<float> { static __device__ __forceinline__ float of(float x) { return x; } };
template <> struct Stored<uint16_t> {
  static __device__ __forceinline__ float of(float x) { return bf16_to_f32(f32_to_bf16(x)); }
};

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void dirgate_lowrank_kernel(const TI* __restrict__ low, long long ld,
                                                               const TI* __restrict__ w1, const TI* __restrict__ b1,
                                                               TO* __restrict__ out, int B, int L, int H, int Dk,
                                                               float inv_norm, float clamp_min, int use_clamp) {
  constexpr int R = kGateRank, TOK = 32;
  __shared__ float lowf[TOK][R];
  const int nv = 2 * H * Dk / 8;  // channel octets per token row
  const int dk8 = Dk >> 3;
  const int b = blockIdx.y;
  const int l0 = blockIdx.x * TOK;
  if (threadIdx.x < TOK * (R / 8)) {
    const int t = threadIdx.x / (R / 8), part = threadIdx.x % (R / 8);
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (l0 + t < L) Vec8<TI>::load(low + ((size_t)b * L + l0 + t) * (size_t)ld + part * 8, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) lowf[t][part * 8 + j] = x[j];
  }
  __syncthreads();
  const int per = nv < 256 ? nv : 256;  // threads side by side on one token
  const int groups = 256 / per;         // tokens in flight
  const int oc = threadIdx.x % per, tg = threadIdx.x / per;
  if (tg >= groups) return;
  for (int cv = oc; cv < nv; cv += per) {
    float w[8][R], bias[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int p = 0; p < R / 8; ++p) {
        float x[8];
        Vec8<TI>::load(w1 + ((size_t)cv * 8 + j) * R + p * 8, x);
#pragma unroll
        for (int i = 0; i < 8; ++i) w[j][p * 8 + i] = x[i];
      }
    Vec8<TI>::load(b1 + (size_t)cv * 8, bias);
    const int d8 = cv % dk8, hh = (cv / dk8) % H, dir = cv / (dk8 * H);
    TO* dst = out + ((((size_t)dir * B + b) * H + hh) * L) * (size_t)Dk + (size_t)d8 * 8;
    for (int t = tg; t < TOK; t += groups) {
      const int l = l0 + t;
      if (l >= L) break;
      float acc[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float xr = lowf[t][r];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = __builtin_fmaf(xr, w[j][r], acc[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = Stored<TI>::of(acc[j] + bias[j]);
        float yv = logsigmoidf_(x);
        yv *= inv_norm;
        yv = fmaxf(yv, clamp_min);  // (no clamp: clamp_min is NaN and fmaxf returns the other operand)
        acc[j] = yv;
      }
      Vec8<TO>::store(dst + (size_t)l * Dk, acc);
    }
  }
}

// The same for bf16 inputs on the matrix cores: one v_mfma_f32_32x32x16_bf16 is the whole rank-16 product of 32
// channels x 32 tokens.  Operand A holds weight rows, operand B the tokens' low-rank rows, both read straight from
// memory as one 16-byte load per lane (lane = (row r, contraction half h) supplies elements 8h..8h+7 of its row).
// Accumulator register 4g+m of lane (r, h) holds matrix row 8g+4h+m of column r; matrix row i is given channel
// 16*((i>>2)&1) + 4*(i>>3) + (i&3) of the tile, so that lane (r, h) ends up with channels 16h..16h+15 of token r:
// 32 contiguous bytes of the head-major output.  Tokens are numbered over B*L; a workgroup owns NTG groups of 32 and
// its four waves take the channel tiles in turn, each weight tile serving all the groups (gridDim.y workgroups share a group's tiles).  Needs Dk % 16 == 0 (a 16-channel run stays inside one head).
template <typename TO, int NTG>
__global__ __launch_bounds__(256) void dirgate_lowrank_mfma_kernel(const uint16_t* __restrict__ low, long long ld,
                                                                    const uint16_t* __restrict__ w1,
                                                                    const uint16_t* __restrict__ b1,
                                                                    TO* __restrict__ out, long long ntok, int B, int L,
                                                                    int H, int Dk, float inv_norm, float clamp_min,
                                                                    int use_clamp) {
  constexpr int R = kGateRank;
  (void)use_clamp;  // (a NaN clamp_min already means "no clamp" to fmaxf)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  // NTG groups of 32 tokens per workgroup: their low-rank rows are fetched first, a weight tile serves all of them
  u32x4_t xb[NTG];
  bool tok_ok[NTG];
  size_t row_off[NTG];  // (b*H*L + l) * Dk of the token: head hh adds hh*L*Dk
#pragma unroll
  for (int g = 0; g < NTG; ++g) {
    const unsigned tok = (blockIdx.x * NTG + g) * 32u + r;  // the launch keeps B*L below 2^31
    tok_ok[g] = tok < (unsigned)ntok;
    const unsigned tokc = tok_ok[g] ? tok : (unsigned)ntok - 1;
    xb[g] = *reinterpret_cast<const u32x4_t*>(low + (size_t)tokc * (size_t)ld + 8 * h);
    const unsigned b = tokc / (unsigned)L, l = tokc - b * (unsigned)L;
    row_off[g] = ((size_t)b * H * L + l) * (size_t)Dk;
  }
  const int chan_of_row = 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
  const int ntiles = 2 * H * Dk / 32;
  const size_t dir_stride = (size_t)B * H * L * Dk;
  // a tile's weights and biases are requested one tile ahead (a wave walks tiles wave, wave + 4, ...)
  auto request = [&](int tile, u32x4_t& wa, u32x4_t& blo, u32x4_t& bhi) {
    const int c0 = min(tile, ntiles - 1) * 32;
    wa = *reinterpret_cast<const u32x4_t*>(w1 + (size_t)(c0 + chan_of_row) * R + 8 * h);
    blo = *reinterpret_cast<const u32x4_t*>(b1 + c0 + 16 * h);
    bhi = *reinterpret_cast<const u32x4_t*>(b1 + c0 + 16 * h + 8);
  };
  u32x4_t wa_next, blo_next, bhi_next;
  request(wave + 4 * blockIdx.y, wa_next, blo_next, bhi_next);
  const float inv_dk = 1.0f / (float)Dk, inv_h = 1.0f / (float)H;
  for (int tile = wave + 4 * blockIdx.y; tile < ntiles; tile += 4 * gridDim.y) {
    const int c0 = tile * 32;
    const u32x4_t wa = wa_next, blo = blo_next, bhi = bhi_next;
    request(tile + 4 * gridDim.y, wa_next, blo_next, bhi_next);
    float bias[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bias[2 * j] = bf16lo_to_f32(blo[j]), bias[2 * j + 1] = bf16hi_to_f32(blo[j]);
      bias[8 + 2 * j] = bf16lo_to_f32(bhi[j]), bias[8 + 2 * j + 1] = bf16hi_to_f32(bhi[j]);
    }
    const int c = c0 + 16 * h;  // first of this lane's 16 channels
    // (quotients by float reciprocals: exact for channel numbers below 2^20, a fraction of the integer division's cost)
    const int cd = (int)(((float)c + 0.5f) * inv_dk), d = c - cd * Dk;
    const int dir = (int)(((float)cd + 0.5f) * inv_h), hh = cd - dir * H;
    TO* const dst0 = out + (size_t)dir * dir_stride + (size_t)hh * L * Dk + d;
#pragma unroll
    for (int g = 0; g < NTG; ++g) {
      f32x16_t acc;
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] = 0.f;
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wa),
                                                    __builtin_bit_cast(bf16x8_t, xb[g]), acc, 0, 0, 0);
      float lo[8], hi[8];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float x = Stored<uint16_t>::of(acc[j] + bias[j]);
        float yv = logsigmoidf_(x);
        yv *= inv_norm;
        yv = fmaxf(yv, clamp_min);  // (no clamp: clamp_min is NaN and fmaxf returns the other operand)
        if (j < 8) lo[j] = yv;
        else hi[j - 8] = yv;
      }
      if (tok_ok[g]) {
        TO* dst = dst0 + row_off[g];
        Vec8<TO>::store(dst, lo);
        Vec8<TO>::store(dst + 8, hi);
      }
    }
  }
}

// Backward of the low-rank gate preparation for bf16 rows, on the matrix cores: for 32 tokens x 32 channels the product low . w1^T
// is formed as in the forward, dx = d_out * inv_norm * sigmoid(-x) (zero where the forward clamped) is rounded to bf16 and
// goes to memory (the weight gradient reads it), and the same registers are the operand of the second product
// d_low = dx . w1: a lane's sixteen channels are two runs of eight, which is what one step's operand takes, and the transposed
// weights (w1t [16][2*H*Dk]) are addressed to match.  A workgroup owns 32 tokens; its waves take the channel tiles in
// turn and add their d_low through LDS.  Bound by reading d_out and writing dx once: the separate layer's two products and
// the elementwise pass moved the [B*L, 2*H*Dk] matrix five times.
// us at 4 / 6 / 8 / 12 waves (a wave per channel tile at most): rows 784, 768 channels 12.5 / 10.7 / 9.1 / 8.4; 4704, 768 13.4 / 11.5 / 10.0 / 9.6;
// 25088, 384 17.1 / 18.1 / 15.7 / 19.3; 11760, 768 18.7 / 18.9 / 16.0 / 17.5.
// A form of its own where nothing is clamped, as in the models: whether a gate was, costs two of a value's four transcendental
// instructions, which were what bound the kernel (25088 rows, 384 15.8 -> 13.0 us; 11760, 768 16.2 -> 12.5; 784, 768 9.1 -> 7.5).
constexpr int kGateBwdWaves = 8;

template <typename TO, bool CLAMP>
__global__ __launch_bounds__(64 * kGateBwdWaves) void dirgate_lowrank_bwd_kernel(const uint16_t* __restrict__ low, long long ld,
                                                                  const uint16_t* __restrict__ w1,
                                                                  const uint16_t* __restrict__ w1t,
                                                                  const uint16_t* __restrict__ b1,
                                                                  const TO* __restrict__ d_out, uint16_t* __restrict__ dx,
                                                                  uint16_t* __restrict__ d_low, long long ldd,
                                                                  long long ntok, int B, int L, int H, int Dk,
                                                                  float inv_norm, float clamp_min) {
  constexpr int R = kGateRank;
  __shared__ f32x4_t part[kGateBwdWaves][2][64];  // [wave][rank octet][lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const unsigned tok = blockIdx.x * 32u + r;
  const bool tok_ok = tok < (unsigned)ntok;
  const unsigned tokc = tok_ok ? tok : (unsigned)ntok - 1;
  const u32x4_t xb = *reinterpret_cast<const u32x4_t*>(low + (size_t)tokc * (size_t)ld + 8 * h);
  const unsigned b = tokc / (unsigned)L, l = tokc - b * (unsigned)L;
  const size_t row_off = ((size_t)b * H * L + l) * (size_t)Dk;
  const int chan_of_row = 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
  const int width = 2 * H * Dk, ntiles = width / 32;
  const size_t dir_stride = (size_t)B * H * L * Dk;
  f32x16_t dl;
#pragma unroll
  for (int j = 0; j < 16; ++j) dl[j] = 0.f;
  for (int tile = wave; tile < ntiles; tile += waves) {
    const int c = tile * 32 + 16 * h;  // first of this lane's 16 channels
    const int cd = c / Dk, d = c - cd * Dk, dir = cd / H, hh = cd - dir * H;
    const TO* src = d_out + (size_t)dir * dir_stride + (size_t)hh * L * Dk + d + row_off;
    float g[2][8];
    Vec8<TO>::load(src, g[0]);
    Vec8<TO>::load(src + 8, g[1]);
    const u32x4_t wa = *reinterpret_cast<const u32x4_t*>(w1 + (size_t)(tile * 32 + chan_of_row) * R + 8 * h);
    u32x4_t wt[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};  // matrix rows past the rank stay zero
    float bias[2][8];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      Vec8<uint16_t>::load(b1 + c + 8 * p, bias[p]);
      if (r < R) wt[p] = *reinterpret_cast<const u32x4_t*>(w1t + (size_t)r * width + c + 8 * p);
    }
    f32x16_t acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.f;
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wa), __builtin_bit_cast(bf16x8_t, xb), acc,
                                                  0, 0, 0);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      u32x4_t o;
      float e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = Stored<uint16_t>::of(acc[8 * p + j] + bias[p][j]);
        const bool clamped = CLAMP && logsigmoidf_(x) * inv_norm < clamp_min;
        e[j] = clamped ? 0.f : g[p][j] * inv_norm * sigmoidf_(-x);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(e[2 * j], e[2 * j + 1]);
      if (tok_ok) *reinterpret_cast<u32x4_t*>(dx + (size_t)tok * width + c + 8 * p) = o;
      dl = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wt[p]), __builtin_bit_cast(bf16x8_t, o), dl,
                                                   0, 0, 0);
    }
  }
  // accumulator register 4g+m of lane (r, h) is rank 8g+4h+m of token r; ranks 0..15 are g = 0, 1
#pragma unroll
  for (int g = 0; g < 2; ++g) part[wave][g][lane] = f32x4_t{dl[4 * g], dl[4 * g + 1], dl[4 * g + 2], dl[4 * g + 3]};
  __syncthreads();
  for (int g = wave; g < 2; g += waves) {  // (a single wave where there is a single tile)
    if (!tok_ok) break;
    f32x4_t sum = part[0][g][lane];
    for (int k = 1; k < waves; ++k) sum += part[k][g][lane];
    *reinterpret_cast<u32x2_t*>(d_low + (size_t)tok * (size_t)ldd + 8 * g + 4 * h) =
        u32x2_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  }
}

int launch_dirgate_lowrank_bwd(const void* low, long long ld, const void* w1, const void* w1t, const void* b1,
                               const void* d_out, void* dx, void* d_low, long long ldd, int B, int L, int H, int Dk,
                               float inv_norm, float clamp_min, int out_dtype, hipStream_t stream) {
  const long long ntok = (long long)B * L;
  if (Dk % 16 != 0 || ntok >= 0x7fffffffLL - 64 || 2LL * H * Dk > (1 << 20)) return -95;
  const dim3 grid((unsigned)((ntok + 31) / 32)), block(64 * std::min(kGateBwdWaves, 2 * H * Dk / 32));
#define VIG_DLB_CASE(TO)                                                                                             \
  hipLaunchKernelGGL((clamp_min == clamp_min ? dirgate_lowrank_bwd_kernel<TO, true> : dirgate_lowrank_bwd_kernel<TO, false>), grid, block, 0, stream, (const uint16_t*)low, ld,             \
                     (const uint16_t*)w1, (const uint16_t*)w1t, (const uint16_t*)b1, (const TO*)d_out, (uint16_t*)dx, \
                     (uint16_t*)d_low, ldd, ntok, B, L, H, Dk, inv_norm, clamp_min)
  if (out_dtype == 1) VIG_DLB_CASE(uint16_t);
  else VIG_DLB_CASE(float);
#undef VIG_DLB_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

template <typename TI, typename TO>
static int launch_dirgate_lowrank_t(const void* low, long long ld, const void* w1, const void* b1, void* out, int B,
                                    int L, int H, int Dk, float inv_norm, float clamp_min, hipStream_t stream) {
  const int use_clamp = clamp_min == clamp_min;  // NaN disables
  if (B > 65535) return -22;
  hipLaunchKernelGGL((dirgate_lowrank_kernel<TI, TO>), dim3((L + 31) / 32, B), dim3(256), 0, stream, (const TI*)low, ld,
                     (const TI*)w1, (const TI*)b1, (TO*)out, B, L, H, Dk, inv_norm, clamp_min, use_clamp);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_dirgate_lowrank(const void* low, long long ld, const void* w1, const void* b1, void* out, int B, int L,
                           int H, int Dk, int rank, float inv_norm, float clamp_min, int in_dtype, int out_dtype,
                           hipStream_t stream) {
  if (rank != kGateRank) return -95;
  if (in_dtype == 1 && Dk % 16 == 0 && (long long)B * L < 0x7fffffffLL - 64 && 2LL * H * Dk <= (1 << 20)) {
    const int use_clamp = clamp_min == clamp_min;  // NaN disables
    const long long ntok = (long long)B * L;
    constexpr int kGroups = 1;  // token groups of 32 per workgroup (two measured no faster)
    const unsigned nb = (unsigned)((ntok + 32 * kGroups - 1) / (32 * kGroups));
    // few tokens: the channel tiles of a token group over up to 1024 workgroups in all (B 1, H 3 4.3 -> 3.3 us; B 4, H 6
    // 4.2 -> 2.9; B 16 4.6 -> 3.5), a round of four tiles at least for each
    const int rounds = (2 * H * Dk / 32 + 3) / 4;
    const dim3 grid(nb, (unsigned)max(1, min(rounds, (int)(1024 / nb)))), block(256);
    if (out_dtype == 1)
      hipLaunchKernelGGL((dirgate_lowrank_mfma_kernel<uint16_t, kGroups>), grid, block, 0, stream, (const uint16_t*)low, ld,
                         (const uint16_t*)w1, (const uint16_t*)b1, (uint16_t*)out, ntok, B, L, H, Dk, inv_norm,
                         clamp_min, use_clamp);
    else
      hipLaunchKernelGGL((dirgate_lowrank_mfma_kernel<float, kGroups>), grid, block, 0, stream, (const uint16_t*)low, ld,
                         (const uint16_t*)w1, (const uint16_t*)b1, (float*)out, ntok, B, L, H, Dk, inv_norm,
                         clamp_min, use_clamp);
    return hipGetLastError() == hipSuccess ? 0 : -5;
  }
  if (in_dtype == 0 && out_dtype == 0) return launch_dirgate_lowrank_t<float, float>(low, ld, w1, b1, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  if (in_dtype == 0 && out_dtype == 1) return launch_dirgate_lowrank_t<float, uint16_t>(low, ld, w1, b1, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  if (in_dtype == 1 && out_dtype == 0) return launch_dirgate_lowrank_t<uint16_t, float>(low, ld, w1, b1, out, B, L, H, Dk, inv_norm, clamp_min, stream);
  return launch_dirgate_lowrank_t<uint16_t, uint16_t>(low, ld, w1, b1, out, B, L, H, Dk, inv_norm, clamp_min, stream);
}

// ---------------------------------------------------------------------------
// 3x3 depthwise stencil on the token grid, channels-last.  One workgroup owns one image (or one head slab), a
// group of 64 channels and a band of grid rows: it stages the band plus a one-cell halo all around in LDS, with
// zeros where the halo leaves the grid (coalesced 16-byte loads, every input byte leaves L2 once, and no tap needs a
// bounds check or a clamped address).  Thread = (channel octet, token lane) keeps the 8x9 weights of its channels
// in registers and walks the band's tokens lane, lane+32, ...
//   GATE = false:  y = conv(x) (+bias) (SiLU optional)          x, y [N, h*w, C] with row stride `stride` elements
//   GATE = true :  y = x * sigmoid(conv(x))                      (bias / SiLU unused)
// weights [Ctot, 9] f32.
// ---------------------------------------------------------------------------
constexpr int kStencilGroup = 64;  // channels per workgroup

template <typename T, bool GATE>
__global__ __launch_bounds__(256) void stencil3x3_kernel(const T* __restrict__ x, const float* __restrict__ wt,
                                                          const float* __restrict__ bias, T* __restrict__ y,
                                                          T* __restrict__ pre, int h, int w, int stride,
                                                          int groups_per_image, int wmod, int cgroup, int band_rows,
                                                          int silu) {
  extern __shared__ __align__(16) char smem[];
  T* tile = reinterpret_cast<T*>(smem);  // [(band_rows + 2) * (w + 2)][64]
  const int oct = threadIdx.x & 7, tl = threadIdx.x >> 3;  // 8 octets x 32 token lanes
  const int img = blockIdx.x / groups_per_image, grp = blockIdx.x % groups_per_image;
  const int r0 = blockIdx.y * band_rows;  // first output row of the band
  const int r1 = min(r0 + band_rows, h);
  const int L = h * w, pw = w + 2;
  const bool ch_ok = grp * kStencilGroup + oct * 8 < cgroup;  // channel tail of the last group
  const size_t base = (size_t)img * L * stride + (size_t)grp * kStencilGroup + oct * 8;
  // ---- this thread's 8 x 9 weights: 72 consecutive floats, fetched (as 16-byte loads) ahead of the staging loop
  // so that their latency runs under it ----
  const int wch = (blockIdx.x / groups_per_image % wmod) * cgroup + grp * kStencilGroup + oct * 8;  // first weight channel
  float wreg[8][9];
  float breg[8];
  if (ch_ok) {
    float* wflat = &wreg[0][0];
#pragma unroll
    for (int i = 0; i < 18; ++i) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(wt + (size_t)wch * 9 + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) wflat[4 * i + e] = v[e];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) breg[j] = (!GATE && bias) ? bias[wch + j] : 0.f;
  }
  // ---- stage padded cells (pr, pc) <-> grid (r0 - 1 + pr, pc - 1) ----
  // kBatch cells per thread are in flight at a time: the loads of a batch are issued before the first LDS store waits
  constexpr int kBatch = sizeof(T) == 2 ? 8 : 4;
  // (A thread's cells are 32 apart: row and column are carried along.  With a division a cell, B 256, 14 x 14, C 384 took 22.8 us
  // instead of 21.4, B 8, 64 x 64, C 192 13.0 instead of 12.0.  In the output loop below, where the division runs under the LDS
  // reads, the same costs time: 25.2 us.)
  const int ncell = (r1 - r0 + 2) * pw;
  const int prows = 32 / pw, pcols = 32 - prows * pw;
  int pr = tl / pw, pc = tl - pr * pw;
  for (int t0 = tl; t0 < ncell; t0 += 32 * kBatch) {
    Raw8<T> cell[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int t = t0 + 32 * u;
      const int r = r0 - 1 + pr, c = pc - 1;
      pr += prows, pc += pcols;
      if (pc >= pw) pc -= pw, ++pr;
      cell[u].zero();
      if (t < ncell && ch_ok && r >= 0 && r < h && c >= 0 && c < w)
        cell[u].load(x + base + (size_t)(r * w + c) * stride);
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int t = t0 + 32 * u;
      if (t < ncell) cell[u].store(tile + t * kStencilGroup + oct * 8);
    }
  }
  __syncthreads();
  if (!ch_ok) return;
  const int nout = (r1 - r0) * w;
  for (int t = tl; t < nout; t += 32) {
    const int rl = t / w, c = t - rl * w;
    const T* p = tile + (rl * pw + c) * kStencilGroup + oct * 8;  // padded cell of tap (-1, -1)
    float acc[8], ctr[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = breg[j], ctr[j] = 0.f;
#pragma unroll
    for (int di = 0; di < 3; ++di) {
#pragma unroll
      for (int dj = 0; dj < 3; ++dj) {
        float xv[8];
        Vec8<T>::load(p + (di * pw + dj) * kStencilGroup, xv);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = __builtin_fmaf(xv[j], wreg[j][di * 3 + dj], acc[j]);
        if (GATE && di == 1 && dj == 1) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ctr[j] = xv[j];
        }
      }
    }
    if (GATE) {
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = ctr[j] * sigmoidf_(acc[j]);
    } else if (silu) {
      if (pre) {  // kept for the backward; the activation reads the stored value
        Vec8<T>::store(pre + base + (size_t)((r0 + rl) * w + c) * stride, acc);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = Stored<T>::of(acc[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = acc[j] * sigmoidf_(acc[j]);
    }
    Vec8<T>::store(y + base + (size_t)((r0 + rl) * w + c) * stride, acc);
  }
}

template <typename T, bool GATE>
static int launch_stencil(const void* x, const float* wt, const float* bias, void* y, void* pre, int images, int h, int w,
                          int stride, int wmod, int cgroup, int silu, hipStream_t stream) {
  // rows per band so that (band + 2) x (w + 2) padded cells x 64 channels fit 48 KB of LDS
  const int row_bytes = (w + 2) * kStencilGroup * (int)sizeof(T);
  int band = 48 * 1024 / row_bytes - 2;
  if (band < 1) return -95;
  if (band > h) band = h;
  const int groups = (cgroup + kStencilGroup - 1) / kStencilGroup;
  // Few images: shorter bands, until there are kFewBands workgroups.  One image's 3 to 24 workgroups leave the chip empty and a
  // band lasts as long as its chain of loads and taps: 14 x 14, C 192 B 1 8.1 -> 4.5 us, B 16 8.5 -> 5.6; 32 x 32, C 384 B 1
  // 10.6 -> 5.0.  (256 workgroups and more: 6.3 at B 16, the halo rows of one-row bands are read three times; 64: 6.6.)
  constexpr int kFewBands = 128;
  const int per = (kFewBands + images * groups - 1) / (images * groups);
  if (per > (h + band - 1) / band) band = max(1, h / per);
  const int nband = (h + band - 1) / band;
  const size_t lds = (size_t)(band + 2) * row_bytes;
  hipLaunchKernelGGL((stencil3x3_kernel<T, GATE>), dim3(images * groups, nband), dim3(256), lds, stream, (const T*)x, wt,
                     bias, (T*)y, (T*)pre, h, w, stride, groups, wmod, cgroup, band, silu);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// ---------------------------------------------------------------------------
// The depthwise convolution where there is not enough of it for the staged form above: a thread makes four channels of one column of a
// band of rows.  It walks down the band with the three cells of a row (its own and the two beside it, which other threads fetch too:
// the lines are in L1) and three rows of sums under way, the next three rows on their way from memory.  No cell passes LDS and no wave
// waits for another, except once for the taps' weights, which come by way of LDS (a lane's 36 floats lie 144 bytes apart).  A
// workgroup: 16 quads of channels (a line of bf16) by 16 columns, counted through bands and images.
// Sums in the staged form's order, so its bits.
// ---------------------------------------------------------------------------
template <typename T> struct Quad;  // four values of a row
template <> struct Quad<uint16_t> {
  u32x2_t a;
  __device__ __forceinline__ void zero() { a = u32x2_t{0u, 0u}; }
  __device__ __forceinline__ void load(const uint16_t* p) { a = *reinterpret_cast<const u32x2_t*>(p); }
  __device__ __forceinline__ void unpack(float (&v)[4]) const {
    v[0] = bf16lo_to_f32(a[0]), v[1] = bf16hi_to_f32(a[0]), v[2] = bf16lo_to_f32(a[1]), v[3] = bf16hi_to_f32(a[1]);
  }
  static __device__ __forceinline__ void store(uint16_t* p, const float (&v)[4]) {
    *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
};
template <> struct Quad<float> {
  f32x4_t a;
  __device__ __forceinline__ void zero() { a = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ void load(const float* p) { a = *reinterpret_cast<const f32x4_t*>(p); }
  __device__ __forceinline__ void unpack(float (&v)[4]) const { v[0] = a[0], v[1] = a[1], v[2] = a[2], v[3] = a[3]; }
  static __device__ __forceinline__ void store(float* p, const float (&v)[4]) { *reinterpret_cast<f32x4_t*>(p) = f32x4_t{v[0], v[1], v[2], v[3]}; }
};

template <typename T>
__global__ __launch_bounds__(256) void dwconv3x3_columns_kernel(const T* __restrict__ x, const float* __restrict__ wt,
                                                                const float* __restrict__ bias, T* __restrict__ y, T* __restrict__ pre,
                                                                int columns, int h, int w, int C, int bands, int band, int silu) {
  __shared__ __align__(16) float wts[kStencilGroup * 9];
  const int quad = threadIdx.x & 15, ch = blockIdx.y * kStencilGroup + 4 * quad;
  const int column = blockIdx.x * 16 + (threadIdx.x >> 4);
  const bool own = column < columns && ch < C;
  const int line = column / w, c = column - line * w;  // (image, band)
  const int img = line / bands, r0 = (line - img * bands) * band;
  const int r1 = own ? min(r0 + band, h) : r0 - 2;  // (no rows for a thread without a column)
  const size_t base = ((size_t)img * h * w + c) * C + ch, pitch = (size_t)w * C;
  Quad<T> cell[3][3];
  const auto fetch = [&](int row, Quad<T> (&to)[3]) {
    const bool in = row >= 0 && row <= r1 && row < h;
    const T* p = x + base + (in ? row * pitch : 0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      to[d].zero();
      if (in && (d == 1 || (d == 0 ? c > 0 : c < w - 1))) to[d].load(p + (d - 1) * C);
    }
  };
#pragma unroll
  for (int u = 0; u < 3; ++u) fetch(r0 - 1 + u, cell[u]);
  {
    const int n = min(kStencilGroup, C - (int)blockIdx.y * kStencilGroup) * 9;  // (a multiple of 72)
    const float* from = wt + (size_t)blockIdx.y * (kStencilGroup * 9);
    for (int i = 4 * threadIdx.x; i < n; i += 1024) *reinterpret_cast<f32x4_t*>(wts + i) = *reinterpret_cast<const f32x4_t*>(from + i);
  }
  float b[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias && own) {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(bias + ch);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = v[j];
  }
  __syncthreads();
  float k[4][9];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(wts + 36 * quad + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) k[(4 * i + e) / 9][(4 * i + e) % 9] = v[e];
  }
  float s0[4] = {0.f, 0.f, 0.f, 0.f}, s1[4] = {b[0], b[1], b[2], b[3]};  // sums of the row above the one at hand, and of its own
  for (int p0 = r0 - 1; p0 <= r1; p0 += 3) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int p = p0 + u;
      if (p > r1) break;
      float s2[4] = {b[0], b[1], b[2], b[3]};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        float v[4];
        cell[u][d].unpack(v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s0[j] = __builtin_fmaf(v[j], k[j][6 + d], s0[j]);
          s1[j] = __builtin_fmaf(v[j], k[j][3 + d], s1[j]);
          s2[j] = __builtin_fmaf(v[j], k[j][d], s2[j]);
        }
      }
      fetch(p + 3, cell[u]);
      if (p > r0) {
        const size_t at = base + (p - 1) * pitch;
        if (silu) {
          if (pre) {  // kept for the backward; the activation reads the stored value
            Quad<T>::store(pre + at, s0);
#pragma unroll
            for (int j = 0; j < 4; ++j) s0[j] = Stored<T>::of(s0[j]);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) s0[j] = s0[j] * sigmoidf_(s0[j]);
        }
        Quad<T>::store(y + at, s0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) s0[j] = s1[j], s1[j] = s2[j];
    }
  }
}

// The columns form while quads x columns of all images are no more than this.  Beyond, two bands are more threads than the chip takes at once, the
// form is bound by its vector work (a quad's row costs as much around its 36 products as in them) and the staged form's bands of a whole
// image are quicker than two of its bands (than one only where images are tall: inputs from memory, us, staged / one / two: C 192 172 k columns 14 x 14 16.7 / 15.8 / 16.7,
// 198 k 48 x 48 52.0 / 53.8 / 48.7).  us, staged / columns, bf16 unless said: C 384 32 x 14 x 14 9.8 / 8.1, 64 images 13.2 / 10.6, 90 (120 k) 15.8 / 12.2, 128
// (172 k) 17.3 / 19.5, 256 23.3 / 26.0; C 192 128 images (86 k) 11.6 / 9.0, 256 (172 k) 15.1 / 15.7, 8 x 64 x 64 12.8 / 10.3, 3 x 48 x 48 8.0 / 6.2;
// C 768 64 x 14 x 14 (172 k) 14.8 / 16.0, 10 x 32 x 32 15.2 / 11.8; fp32 C 768 8 x 32 x 32 18.2 / 13.8, C 192 8 x 48 x 48 15.6 / 10.2; one image
// 14 x 14 4.3 / 3.9.
constexpr long long kColumnThreads = 150000;
template <typename T>
static int launch_dwconv3x3_t(const void* x, const float* wt, const float* bias, void* y, void* pre, int B, int h, int w, int C, int silu,
                              hipStream_t stream) {
  const long long threads = (long long)B * w * (C / 4), cells = (long long)B * h * w;
  if (3 * (w + 2) * kStencilGroup * (int)sizeof(T) > 48 * 1024) return -95;
  // every batch element is an image of C channels; all images share the C weight channels
  if (threads > kColumnThreads || cells > (1 << 30)) return launch_stencil<T, false>(x, wt, bias, y, pre, B, h, w, C, 1, C, silu, stream);
  // Bands for two hundred thousand threads, as far as there are rows (8 x 64 x 64, C 192: for half or twice as many 11.2, 11.8 instead of 10.3), but
  // no more threads than the chip takes at once, four workgroups to a CU: a band less where the last one would begin a second round, unless that
  // leaves one long band (us, inputs from memory, staged / with that band / without; C 192: 170 x 11 x 11 10.3 / 11.7 / 9.8, 231 x 8 x 8 9.7 / 10.3 / 8.1, 255 x 11 x 11 13.1 / 14.1 / 13.1,
  // 350 x 8 x 8 13.1 / 11.8 / 10.9, 200 x 14 x 14 16.2 / 15.5 / 15.3; 116 x 24 x 24 21.3 / 20.6 / 21.7; fp32 170 x 11 x 11 12.4 / 13.1 / 10.8)
  const int fill = (int)((200000 + threads - 1) / threads), fit = (int)std::max<long long>(1, 4 * 256 * 256 / threads);
  const int want = std::min(h, fit > 1 || h <= 16 ? std::min(fill, fit) : fill), band = (h + want - 1) / want, bands = (h + band - 1) / band;
  const int columns = B * bands * w;
  hipLaunchKernelGGL(dwconv3x3_columns_kernel<T>, dim3((columns + 15) / 16, (C + kStencilGroup - 1) / kStencilGroup), dim3(256), 0, stream,
                     (const T*)x, wt, bias, (T*)y, (T*)pre, columns, h, w, C, bands, band, silu);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}
int launch_dwconv3x3(const void* x, const float* wt, const float* bias, void* y, void* pre, int B, int h, int w, int C,
                     int silu, int io_dtype, hipStream_t stream) {
  return (io_dtype == 0 ? launch_dwconv3x3_t<float> : launch_dwconv3x3_t<uint16_t>)(x, wt, bias, y, pre, B, h, w, C, silu, stream);
}

int launch_locality_gate(const void* o, const float* wt, void* y, int B, int H, int h, int w, int Dv, int io_dtype,
                         hipStream_t stream) {
  if (Dv > 64) return -95;
  // every (batch, head) slab is an "image" of Dv channels; head hd uses weight channels [hd*Dv, hd*Dv + Dv)
  if (io_dtype == 0) return launch_stencil<float, true>(o, wt, nullptr, y, nullptr, B * H, h, w, Dv, H, Dv, 0, stream);
  return launch_stencil<uint16_t, true>(o, wt, nullptr, y, nullptr, B * H, h, w, Dv, H, Dv, 0, stream);
}

// ---------------------------------------------------------------------------
// Residual add, RMS norm and the depthwise 3x3 convolution behind it in one kernel, bf16, C = 24 LANES channels.  A workgroup makes
// up to 14 columns of the grid, of one row or of a band that it walks three rows at a time (WALK): the sums and norms of these cells
// and of those around them (LANES lanes a token), staged rounded in LDS between zeros, three rows or the five that three rows of taps
// reach; then the taps.  One row is bound by latency (two launches with a chain of loads each became one; the taps' weights come by
// way of LDS: fetched by the octets of 72 that a thread needs, as above, they cost 1.8 us at C 192 and 3 at 384), the walk by
// what one workgroup a CU has under way (vector pipe 46 %): 115 registers leave C 384 no second one (80 for two spill 35: 46 -> 61 us);
// its next rows are fetched during the taps.  C 384, 256 x 14 x 14: 37.6 us = 4.1 TB/s of the two inputs and two outputs; the two kernels 46.4.
// ---------------------------------------------------------------------------
constexpr int kNormStencilCols = 14;  // with the two beside them in three rows: 48 tokens

struct NormStencilArgs {
  const uint16_t *x, *residual;  // [B, h*w, C]; no residual: null
  const float *norm, *wt, *bias; // [C], [C, 9], [C] or null
  uint16_t *sum, *y;             // [B, h*w, C]; sum may be null
  int h, w, rows, cols, silu;  // rows and columns of a workgroup
  float eps;
};
template <int LANES, bool WALK>  // three rows of tokens at a time; then four columns of channel pairs
__global__ __launch_bounds__(48 * LANES) void norm_stencil_kernel(NormStencilArgs a) {
  constexpr int NV = 3, C = 8 * NV * LANES, kThreads = 48 * LANES, kPairs = C / 2, kCols = kThreads / kPairs, kRing = WALK ? 5 : 3;
  extern __shared__ __align__(16) char smem[];
  uint16_t* tile = reinterpret_cast<uint16_t*>(smem);  // [kRing rows][columns + 2][C]
  const int bands = (a.h + a.rows - 1) / a.rows, img = blockIdx.x / bands, row0 = (blockIdx.x - img * bands) * a.rows;
  const int rows = WALK ? min(a.rows, a.h - row0) : 1, steps = WALK ? (rows + 4) / 3 : 1;
  const int c0 = blockIdx.y * a.cols, cols = min(a.cols, a.w - c0), pw = cols + 2;
  const size_t image = (size_t)img * a.h * a.w * C;
  float* wts = reinterpret_cast<float*>(smem + 2 * kRing * (kNormStencilCols + 2) * C);  // [C][9]
  const int pair = threadIdx.x % kPairs, col = threadIdx.x / kPairs;
  constexpr int kWLoads = (C * 9 / 4 + kThreads - 1) / kThreads;
  f32x4_t wraw[kWLoads];
#pragma unroll
  for (int i = 0; i < kWLoads; ++i) {
    const int at = (int)threadIdx.x + i * kThreads;
    if (at < C * 9 / 4) wraw[i] = *reinterpret_cast<const f32x4_t*>(a.wt + 4 * at);
  }
  const float b0 = a.bias ? a.bias[2 * pair] : 0.f, b1 = a.bias ? a.bias[2 * pair + 1] : 0.f;
  // padded cell (p, pc) of the band is grid cell (row0 - 1 + p, c0 + pc - 1); step k brings rows 3k .. 3k + 2
  const int sub = threadIdx.x % LANES, t = threadIdx.x / LANES, pr = t / pw, pc = t - pr * pw, c = c0 + pc - 1;
  const bool own = t < 3 * pw;
  Raw8<uint16_t> x[NV], res[NV];
  const auto inside = [&](int p) { return own && p <= rows + 1 && row0 - 1 + p >= 0 && row0 - 1 + p < a.h && c >= 0 && c < a.w; };
  const auto fetch = [&](int p) {
    const bool in = inside(p);
    const size_t at = in ? image + (size_t)((row0 - 1 + p) * a.w + c) * C : 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      x[i].zero(), res[i].zero();
      if (in) x[i].load(a.x + at + 8 * (sub + LANES * i));
      if (in && a.residual) res[i].load(a.residual + at + 8 * (sub + LANES * i));
    }
  };
  fetch(pr);
  float wreg[18];
  for (int k = 0; k < steps; ++k) {
    if (own) {
      const int p = 3 * k + pr;
      const bool in = inside(p);
      float s[NV][8], sq[NV] = {};
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        float b[8];
        x[i].unpack(s[i]);
        res[i].unpack(b);
#pragma unroll
        for (int j = 0; j < 4; ++j) res[i].a[j] = pack_bf16x2(s[i][2 * j] + b[2 * j], s[i][2 * j + 1] + b[2 * j + 1]);  // the rounded sum
        if (a.sum && in && p >= 1 && p <= rows && pc >= 1 && pc <= cols)
          res[i].store(a.sum + image + (size_t)((row0 - 1 + p) * a.w + c) * C + 8 * (sub + LANES * i));
        res[i].unpack(s[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j) sq[i] = __builtin_fmaf(s[i][j], s[i][j], sq[i]);
      }
      float ss = (sq[0] + sq[2]) + sq[1];  // the order of rmsnorm_kernel's wave, so its bits
#pragma unroll
      for (int d = LANES / 2; d > 0; d >>= 1) ss += __shfl_xor(ss, d);
      const float rstd = 1.0f / sqrtf(ss / (float)C + a.eps);
      uint16_t* const cell = tile + ((p % kRing) * pw + pc) * C;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int o = 8 * (sub + LANES * i);
        const f32x4_t wa = *reinterpret_cast<const f32x4_t*>(a.norm + o), wb = *reinterpret_cast<const f32x4_t*>(a.norm + o + 4);
        u32x4_t n;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float f = j < 2 ? wa[2 * j] : wb[2 * j - 4], g = j < 2 ? wa[2 * j + 1] : wb[2 * j - 3];
          n[j] = in ? pack_bf16x2(s[i][2 * j] * rstd * f, s[i][2 * j + 1] * rstd * g) : 0u;
        }
        *reinterpret_cast<u32x4_t*>(cell + o) = n;
      }
    }
    if (k == 0) {
#pragma unroll
      for (int i = 0; i < kWLoads; ++i) {
        const int at = (int)threadIdx.x + i * kThreads;
        if (at < C * 9 / 4) *reinterpret_cast<f32x4_t*>(wts + 4 * at) = wraw[i];
      }
    }
    if (WALK && k + 1 < steps) fetch(3 * k + 3 + pr);
    __syncthreads();
    if (k == 0) {
#pragma unroll
      for (int i = 0; i < 9; ++i) wreg[2 * i] = wts[pair * 18 + 2 * i], wreg[2 * i + 1] = wts[pair * 18 + 2 * i + 1];
    }
    // rows 3k - 2 .. 3k of the band, of the five (one of the three) rows in LDS
    constexpr int kOut = WALK ? 3 : 1;
    const int first = WALK ? 3 * k - 2 : 0;
    const uint16_t* taps[kOut + 2];
#pragma unroll
    for (int i = 0; i < kOut + 2; ++i) taps[i] = tile + ((first + kRing + i) % kRing) * pw * C + pair * 2;
    for (int cc = col; cc < cols; cc += kCols) {
      float lo[kOut], hi[kOut];
#pragma unroll
      for (int i = 0; i < kOut; ++i) lo[i] = b0, hi[i] = b1;
#pragma unroll
      for (int i = 0; i < kOut + 2; ++i)
#pragma unroll
        for (int dj = 0; dj < 3; ++dj) {
          const uint32_t v = *reinterpret_cast<const uint32_t*>(taps[i] + (cc + dj) * C);
#pragma unroll
          for (int o = 0; o < kOut; ++o) {
            if (i - o < 0 || i - o > 2) continue;
            lo[o] = __builtin_fmaf(bf16lo_to_f32(v), wreg[(i - o) * 3 + dj], lo[o]);
            hi[o] = __builtin_fmaf(bf16hi_to_f32(v), wreg[9 + (i - o) * 3 + dj], hi[o]);
          }
        }
#pragma unroll
      for (int o = 0; o < kOut; ++o) {
        if (WALK && (first + o < 0 || first + o >= rows)) continue;
        if (a.silu) lo[o] = lo[o] * sigmoidf_(lo[o]), hi[o] = hi[o] * sigmoidf_(hi[o]);
        *reinterpret_cast<uint32_t*>(a.y + image + (size_t)((row0 + first + o) * a.w + c0 + cc) * C + pair * 2) = pack_bf16x2(lo[o], hi[o]);
      }
    }
    if (WALK && k + 1 < steps) __syncthreads();
  }
}

// Rows of the grid for a workgroup, 0: the two kernels are quicker.  One row costs 3 us and 0.015 for each workgroup of 384 channels (the
// rows around are read and normed three times), a walk 5 us for every step of a round (two workgroups to a CU, one at C 384) and for
// the round's start, the two kernels 10.5 us and 0.77 for 1000 cells of 384 channels.  us, the two kernels / one row / 4 / 7 / 14 rows:
//   C 192 64 x 14 x 14 15.2 / 8.9 / 10.5 / 13.6 / 23.7, 128 images 21.9 / 17.1 / 14.5 / 14.9 / 25.0, 256 31.5 / 28.6 / 32.4 / 21.6 / 27.5,
//   512 52.4 / 51.0 / 53.5 / 45.6 / 38.6; C 384 32 x 14 x 14 14.1 / 9.0 / 12.4 / 17.1 / 30.5, 64 images 19.9 / 17.1 / 14.0 / 17.5 / 30.1,
//   128 28.5 / 29.0 / 26.9 / 20.9 / 32.0, 256 46.4 / 51.5 / 50.1 / 39.3 / 37.6, 512 91 / 97 / 100 / 82 / 79.
// Rounds that are half empty leave it to the two kernels.  Other grids, 150 drawn of 5 to 100 rows and columns, up to 600 images and 2e7
// values: 0.41 to 0.92 of the two kernels' time where this is taken, 0.66 in the mean.
static int norm_stencil_rows(int B, int h, int w, int C) {
  if ((C != 192 && C != 384) || h > 1024 || w > 1024 || (long long)B * h * w > 0x7fffffff) return 0;
  const long long columns = (long long)B * ((w - 1) / kNormStencilCols + 1), slots = C == 192 ? 512 : 256;
  const double two = 0.95 * (10.5 + 2e-6 * C * B * h * w);
  double least = 3 + 4e-5 * C * columns * h;
  int best = 1;
  for (int rows = 4; rows < h + 3; rows += 3) {
    const double us = 5.0 * ((columns * ((h + rows - 1) / rows) + slots - 1) / slots * ((std::min(rows, h) + 4) / 3 + 1));
    if (us < least) best = rows, least = us;
  }
  return least <= two ? best : 0;
}
bool norm_dwconv3x3_supported(int B, int h, int w, int C) { return norm_stencil_rows(B, h, w, C) > 0; }
int launch_norm_dwconv3x3(const void* x, const void* residual, const float* norm, const float* wt, const float* bias, void* sum, void* y,
                          int B, int h, int w, int C, float eps, int silu, hipStream_t stream) {
  const int rows = norm_stencil_rows(B, h, w, C);
  if (rows == 0) return -95;
  const int parts = (w - 1) / kNormStencilCols + 1, cols = (w + parts - 1) / parts;
  const NormStencilArgs a{(const uint16_t*)x, (const uint16_t*)residual, norm, wt, bias, (uint16_t*)sum, (uint16_t*)y, h, w, rows, cols, silu, eps};
  const bool walk = rows > 1;
  const size_t lds = (2 * (walk ? 5 : 3) * (kNormStencilCols + 2) + 36) * (size_t)C;
  const dim3 grid(B * ((h + rows - 1) / rows), (w + cols - 1) / cols);
  auto kernel = C == 192 ? (walk ? norm_stencil_kernel<8, true> : norm_stencil_kernel<8, false>)
                         : (walk ? norm_stencil_kernel<16, true> : norm_stencil_kernel<16, false>);
  if (walk && C == 384) {
    static bool done[64] = {};
    if (!allow_lds(reinterpret_cast<const void*>(kernel), lds, done)) return -5;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(2 * C), lds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// ---------------------------------------------------------------------------
// RMS-norm blend epilogue.  One group of Dv/8 lanes owns one (b, l, head) row of
// Dv values; the two mean-squares are reduced with lane shuffles inside the group.
//   y[b,l,hd*Dv+d] = rms(o[b,hd,l,:])*w_g*s + rms(local[b,l,hd,:])*w_l*(1-s)
// HBM-bound (three streams in, one out).  A thread takes N octets of the rows, their loads under way together; it keeps its octet
// of the norms' weights (256 is a multiple of a head's octets).  Measured (us, before: a workgroup for 32 tokens of
// an image, a wave for every fourth, 64 octets at a time): bf16 100 x 768 channels 16.0, now 2.9; 5670 x 768 20.5, now 7.9 (4.4 TB/s); 25088
// x 384 21.0, now 16.8.
// ---------------------------------------------------------------------------
template <typename T, int N>
__global__ __launch_bounds__(256) void locality_blend_kernel(const T* __restrict__ o, const T* __restrict__ loc,
                                                              const T* __restrict__ glin,
                                                              const float* __restrict__ wg,
                                                              const float* __restrict__ wl, T* __restrict__ y, int B,
                                                              int H, int L, int Dv, long long ldg, float eps,
                                                              int silu_out, int tokens) {
  const int d8n = Dv >> 3;  // lanes per row: 4 (Dv=32) or 8 (Dv=64); divides 64, so groups never straddle a wave
  const int nv = H * d8n;   // channel octets per token row
  const int d8 = threadIdx.x & (d8n - 1);
  const OctetRows rows(B, L, nv, tokens);
  const size_t first = (size_t)blockIdx.x * tokens * nv * 8;
  const float inv_dv = 1.0f / (float)Dv;
  float w_g[8], w_l[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) w_g[j] = wg[d8 * 8 + j], w_l[j] = wl[d8 * 8 + j];
  for (int x0 = threadIdx.x; x0 < rows.n; x0 += 256 * N) {
    Raw8<T> ro8[N], rl8[N], rg8[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (x0 + 256 * u >= rows.n) break;  // (whole groups: a row's octets are a multiple of theirs)
      const Octet at(rows, x0 + 256 * u, nv, L);
      const int hd = at.cv / d8n;
      ro8[u].load(o + (((size_t)at.b * H + hd) * L + at.l) * (size_t)Dv + d8 * 8);
      rl8[u].load(loc + first + (size_t)(x0 + 256 * u) * 8);
      rg8[u].load(glin + ((size_t)at.b * L + at.l) * (size_t)ldg + (size_t)at.cv * 8);  // g_lin rows are ldg elements apart
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (x0 + 256 * u >= rows.n) break;
      float xo[8], xl[8], xg[8];
      ro8[u].unpack(xo);
      rl8[u].unpack(xl);
      rg8[u].unpack(xg);
      float so = 0.f, sl = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) so += xo[j] * xo[j], sl += xl[j] * xl[j];
      for (int m = 1; m < d8n; m <<= 1) {
        so += __shfl_xor(so, m);
        sl += __shfl_xor(sl, m);
      }
      const float ro = rsqrtf(so * inv_dv + eps);
      const float rl = rsqrtf(sl * inv_dv + eps);
      float out[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float s = sigmoidf_(xg[j]);
        float v = xo[j] * ro * w_g[j] * s + xl[j] * rl * w_l[j] * (1.f - s);
        if (silu_out) v = v * sigmoidf_(v);
        out[j] = v;
      }
      Vec8<T>::store(y + first + (size_t)(x0 + 256 * u) * 8, out);
    }
  }
}

int launch_locality_blend(const void* o, const void* loc, const void* glin, const float* wg, const float* wl, void* y,
                          int B, int H, int L, int Dv, long long ldg, float eps, int silu_out, int io_dtype,
                          hipStream_t stream) {
  if (B > 65535 || !octet_rows_ok(B, L)) return -22;
  const int nv = H * (Dv / 8), each = octets_each((long long)B * L, nv);
  int tokens = octet_tokens(nv, each);
  const dim3 grid(octet_grid((long long)B * L, tokens)), block(256);
#define VIG_BLEND_CASE(T)                                                                                                    \
  hipLaunchKernelGGL((each == 4 ? locality_blend_kernel<T, 4> : locality_blend_kernel<T, 1>), grid, block, 0, stream,       \
                     (const T*)o, (const T*)loc, (const T*)glin, wg, wl, (T*)y, B, H, L, Dv, ldg, eps, silu_out, tokens)
  if (io_dtype == 0) VIG_BLEND_CASE(float);
  else VIG_BLEND_CASE(uint16_t);
#undef VIG_BLEND_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// ---------------------------------------------------------------------------
// Backward of the depthwise 3x3 convolution on token-major rows x, dy [B, h*w, C], input, weight and bias gradients in one
// pass (zero padding):
//   dx[q, c] = sum over taps of wt[c, t] * dy[q - t, c],  dw[c, t] = sum over b, q of dy[q - t, c] * x[q, c],  db[c] = sum dy
// Both sums run over the same nine neighbours of dy, so a workgroup stages a tile of dy with its halo in LDS (as the forward
// does: 64 channels, a band of the grid) and reads x and writes dx once: bound by those three streams.  A thread keeps four
// channels (their 36 weights and 40 sums stay in registers) and takes every sixteenth position; the sixteen positions combine
// by lane exchange and then through LDS in a fixed order, and the workgroup leaves one row of `partials`
// [workgroups, 10 * C] (columns c*9 + tap, then 9*C + c for the bias), which a column sum finishes.
// With `pre` (the stored convolution result in front of a SiLU) dy is the gradient behind the activation and is taken through
// it while the tile is staged, rounded to the storage type.
// Measured with the column sum (us, bf16; before: bands as tall as LDS allows and at most four workgroups an image and channel group, its weights
// as 36 loads of a float): 128 images of 14 x 14, C 384 27.5, now 23.8; 256 46, now 40; 24 of 28 x 28 26, now 22.5; 8 of 64 x 64, C 192 101, now 32;
// 2 of 61 x 61 54, now 13; 1 of 14 x 14 16, now 8.5.  (Two or four positions' rows of x under way instead of one: 24.1, 30 at 128 images.)
// ---------------------------------------------------------------------------
constexpr int kWgradSplit = 4, kWgradMostSplit = 32, kWgradFill = 512;  // workgroups per image and channel group, at most
constexpr int kBwdWaves = 4;

template <typename T> struct Vec4;
template <> struct Vec4<uint16_t> {
  static __device__ __forceinline__ f32x4_t load(const uint16_t* p) {
    const u32x2_t r = *reinterpret_cast<const u32x2_t*>(p);
    return f32x4_t{bf16lo_to_f32(r[0]), bf16hi_to_f32(r[0]), bf16lo_to_f32(r[1]), bf16hi_to_f32(r[1])};
  }
  static __device__ __forceinline__ void store(uint16_t* p, const f32x4_t x) {
    *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
  }
};
template <> struct Vec4<float> {
  static __device__ __forceinline__ f32x4_t load(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
  static __device__ __forceinline__ void store(float* p, const f32x4_t x) { *reinterpret_cast<f32x4_t*>(p) = x; }
};

template <typename T, bool SILU>
__global__ __launch_bounds__(64 * kBwdWaves) void dwconv3x3_bwd_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ pre, const float* __restrict__ wt,
    T* __restrict__ dx, float* __restrict__ partials, int h, int w, int C, int groups, int band_rows, int band_cols,
    int col_bands, int nbands) {
  extern __shared__ __align__(16) char smem[];
  T* tile = reinterpret_cast<T*>(smem);  // [(band_rows + 2) * (band_cols + 2)][64]
  const int img = blockIdx.x / groups, grp = blockIdx.x % groups;
  const size_t base = (size_t)img * h * w * C + (size_t)grp * kStencilGroup;
  const int oct = threadIdx.x & 7, sl = threadIdx.x >> 3;   // staging: 8 octets x 32 positions
  const int quad = threadIdx.x & 15, tl = threadIdx.x >> 4;  // sums: 16 quads x 16 positions
  const bool oct_ok = grp * kStencilGroup + oct * 8 < C;
  const int ch = grp * kStencilGroup + quad * 4;
  const bool quad_ok = ch < C;
  f32x4_t wk[9], dw[10];
#pragma unroll
  for (int i = 0; i < 9; ++i) {  // 36 consecutive floats
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
    const float* w4 = wt + (size_t)ch * 9 + 4 * i;
    if (quad_ok && dx) {
      if ((reinterpret_cast<uintptr_t>(wt) & 15) == 0) x = *reinterpret_cast<const f32x4_t*>(w4);
      else x = f32x4_t{w4[0], w4[1], w4[2], w4[3]};  // (a caller's weights may start anywhere)
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) wk[(4 * i + e) % 9][(4 * i + e) / 9] = x[e];
  }
#pragma unroll
  for (int t = 0; t < 10; ++t) dw[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int band = blockIdx.y; band < nbands; band += gridDim.y) {
    const int r0 = band / col_bands * band_rows, c0 = band % col_bands * band_cols;
    const int nr = min(band_rows, h - r0), nc = min(band_cols, w - c0);
    const int pw = nc + 2, ncell = (nr + 2) * pw;
    __syncthreads();  // the previous band's readers are done
    constexpr int kBatch = sizeof(T) == 2 && !SILU ? 8 : 4;
    for (int t0 = sl; t0 < ncell; t0 += 32 * kBatch) {
      Raw8<T> cell[kBatch], act[SILU ? kBatch : 1];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int t = t0 + 32 * u;
        const int pr = t / pw, r = r0 - 1 + pr, c = c0 - 1 + t - pr * pw;
        cell[u].zero();
        if constexpr (SILU) act[u].zero();
        if (t < ncell && oct_ok && r >= 0 && r < h && c >= 0 && c < w) {
          const size_t at = base + (size_t)(r * w + c) * C + oct * 8;
          cell[u].load(dy + at);
          if constexpr (SILU) act[u].load(pre + at);
        }
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int t = t0 + 32 * u;
        if (t < ncell) {
          T* const dst = tile + t * kStencilGroup + oct * 8;
          if constexpr (SILU) {
            float g[8], z[8];
            cell[u].unpack(g);
            act[u].unpack(z);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float sg = sigmoidf_(z[j]);
              g[j] *= sg * (1.f + z[j] * (1.f - sg));
            }
            Vec8<T>::store(dst, g);
          } else {
            cell[u].store(dst);
          }
        }
      }
    }
    __syncthreads();
    if (quad_ok) {
      const int nout = nr * nc;
      auto place = [&](int t) {  // element offset of output position t (clamped: the load ahead stays inside)
        t = min(t, nout - 1);
        const int rl = t / nc;
        return base + (size_t)((r0 + rl) * w + c0 + t - rl * nc) * C + quad * 4;
      };
      f32x4_t xn = Vec4<T>::load(x + place(tl));
      for (int t = tl; t < nout; t += 16) {
        const f32x4_t xq = xn;
        xn = Vec4<T>::load(x + place(t + 16));
        const int rl = t / nc, cl = t - rl * nc;
        const T* p = tile + (rl * pw + cl) * kStencilGroup + quad * 4;
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int di = 0; di < 3; ++di) {
#pragma unroll
          for (int dj = 0; dj < 3; ++dj) {
            const f32x4_t g = Vec4<T>::load(p + (di * pw + dj) * kStencilGroup);
            const int tap = (2 - di) * 3 + (2 - dj);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              acc[j] = __builtin_fmaf(g[j], wk[tap][j], acc[j]);
              dw[tap][j] = __builtin_fmaf(g[j], xq[j], dw[tap][j]);
              if (di == 1 && dj == 1) dw[9][j] += g[j];
            }
          }
        }
        if (dx) Vec4<T>::store(dx + place(t), acc);
      }
    }
  }
  if (!partials) return;  // uniform over the grid
  // ---- sixteen positions of a quad: four in the wave by lane exchange, four waves through LDS ----
#pragma unroll
  for (int t = 0; t < 10; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dw[t][j] += __shfl_xor(dw[t][j], 16, 64);
      dw[t][j] += __shfl_xor(dw[t][j], 32, 64);
    }
  f32x4_t* red = reinterpret_cast<f32x4_t*>(smem);  // [wave][quad][tap]
  __syncthreads();
  if ((threadIdx.x & 63) < 16) {
#pragma unroll
    for (int t = 0; t < 10; ++t) red[((threadIdx.x >> 6) * 16 + quad) * 10 + t] = dw[t];
  }
  __syncthreads();
  float* const prow = partials + ((size_t)img * gridDim.y + blockIdx.y) * ((size_t)C * 10);
  if (threadIdx.x < 160) {
    const int q = threadIdx.x / 10, t = threadIdx.x - q * 10;
    f32x4_t sum = red[q * 10 + t];
#pragma unroll
    for (int k = 1; k < kBwdWaves; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += red[(k * 16 + q) * 10 + t][j];
    const int c = grp * kStencilGroup + q * 4;
    if (c < C) {
#pragma unroll
      for (int j = 0; j < 4; ++j) prow[t < 9 ? (size_t)(c + j) * 9 + t : (size_t)C * 9 + c + j] = sum[j];
    }
  }
}

int launch_column_sum(const float* partials, float* out, int n, int C, hipStream_t stream);

// Workgroups an image's channel group may be split over: four, or as many as bring two workgroups a compute unit.
static int wgrad_split(int B, int C) {
  const long long have = (long long)B * ((C + kStencilGroup - 1) / kStencilGroup);
  return (int)std::min<long long>(kWgradMostSplit, std::max<long long>(kWgradSplit, (kWgradFill + have - 1) / have));
}
size_t dwconv3x3_wgrad_workspace(int B, int C) { return (size_t)B * wgrad_split(B, C) * C * 10 * sizeof(float); }
// (a workspace for four is enough)
size_t dwconv3x3_wgrad_least_workspace(int B, int C) { return (size_t)B * kWgradSplit * C * 10 * sizeof(float); }

template <typename T, bool SILU>
static int launch_dwconv3x3_bwd_t(const void* x, const void* dy, const void* pre, const float* wt, void* dx, float* dw_db,
                                  float* partials, int most_split, int B, int h, int w, int C, vig_sum_jobs* later, hipStream_t stream) {
  constexpr int kCells = 48 * 1024 / (kStencilGroup * (int)sizeof(T));  // three workgroups' tiles fit a CU's LDS
  const int band_cols = w < kCells / 6 - 2 ? w : kCells / 6 - 2;        // four rows at least
  const int rows = kCells / (band_cols + 2) - 2;
  const int col_bands = (w + band_cols - 1) / band_cols, groups = (C + kStencilGroup - 1) / kStencilGroup;
  int band_rows = rows < h ? rows : h;
  // Few images: shorter bands, a workgroup each, until there are two a compute unit (us at 256 / 512 / 768 / 1024: 16 images of 14 x 14,
  // C 384 11.5 / 11.2 / 12.4 / 12.5; 20 of 20 x 20 15.8 / 15.2 / 17.6 / 17.7; 9 of 47 x 47 30.5 / 23.3 / 23.9 / 27.5; 8 of 64 x 64, C 192
  // 33 / 32 / 24 / 24: a workgroup's weights, lane exchanges and partial sums cost about as much as two rows of a grid)
  const long long have = (long long)B * groups * col_bands;
  while (band_rows > 2 && have * ((h + band_rows - 1) / band_rows) < kWgradFill && (h + band_rows - 2) / (band_rows - 1) * col_bands <= most_split)
    --band_rows;
  const int nbands = (h + band_rows - 1) / band_rows * col_bands;
  const int split = nbands < most_split ? nbands : most_split;
  size_t lds = (size_t)(band_rows + 2) * (band_cols + 2) * kStencilGroup * sizeof(T);
  const size_t sums = (size_t)kBwdWaves * 16 * 10 * sizeof(f32x4_t);
  if (lds < sums) lds = sums;
  hipLaunchKernelGGL((dwconv3x3_bwd_kernel<T, SILU>), dim3((unsigned)B * groups, split), dim3(64 * kBwdWaves), lds, stream,
                     (const T*)x, (const T*)dy, (const T*)pre, wt, (T*)dx, dw_db ? partials : nullptr, h, w, C, groups,
                     band_rows, band_cols, col_bands, nbands);
  if (hipGetLastError() != hipSuccess) return -5;
  if (dw_db && later) return put_off(*later, partials, dw_db, split * B, C * 10, false) ? 0 : -22;
  return dw_db ? launch_column_sum(partials, dw_db, split * B, C * 10, stream) : 0;
}

int launch_dwconv3x3_bwd(const void* x, const void* dy, const void* pre, const float* wt, void* dx, float* dw_db,
                         void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, vig_sum_jobs* later,
                         hipStream_t stream) {
  if (B > 65535 || C % 8 != 0 || (long long)h * w > 0x7fffffffLL - 64 || (long long)C * 10 > 0x7fffffffLL ||
      (long long)B * ((C + 63) / 64) > 0x7fffffffLL)
    return -22;
  auto fn = io_dtype == 0 ? (pre ? launch_dwconv3x3_bwd_t<float, true> : launch_dwconv3x3_bwd_t<float, false>)
                          : (pre ? launch_dwconv3x3_bwd_t<uint16_t, true> : launch_dwconv3x3_bwd_t<uint16_t, false>);
  // (without weight gradients nobody's partial sums need room)
  const int most = dw_db ? (int)std::min<size_t>(wgrad_split(B, C), workspace_bytes / ((size_t)B * C * 10 * sizeof(float))) : wgrad_split(B, C);
  return fn(x, dy, pre, wt, dx, dw_db, static_cast<float*>(workspace), most, B, h, w, C, later, stream);
}

// ---------------------------------------------------------------------------
// Backward of the RMS-norm blend epilogue, threads as in the forward.  With s = sig(g_lin),
// on = rms(o) * w_g, ln = rms(local) * w_l, y0 = on * s + ln * (1 - s), y = silu_out ? y0 * sig(y0) : y0:
//   dy0 = dy * d(y)/d(y0),  d_on = dy0 * s,  d_ln = dy0 * (1 - s),  d_glin = dy0 * (on - ln) * s * (1 - s),
//   d_o = rms_backward(o, w_g, d_on),  d_local = rms_backward(local, w_l, d_ln)   (per (token, head) row of Dv),
//   dw_g[d] = sum d_on * o * r_o,  dw_l[d] = sum d_ln * local * r_l   over batch, tokens and heads.
// The weight gradients leave as one row of `partials` [workgroups, 2 * Dv] per workgroup (threads park their sums in
// LDS and 2 * Dv threads add the ones of their channel, in a fixed order), which a column sum finishes.  HBM-bound (four streams in,
// three out): a thread fetches its next octet while it works on one, and there are as many workgroups as rows of partials fit.  Measured with
// the column sum (us, before: a workgroup for 32 tokens of an image): bf16 100 x 768 channels 28, now 6.9; 5670 x 768 35, now 18; 25088 x
// 384 41, now 29 (4.7 TB/s); fp32 400 x 768 30, now 7.9.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void locality_blend_bwd_kernel(
    const T* __restrict__ o, const T* __restrict__ loc, const T* __restrict__ glin, const float* __restrict__ wg,
    const float* __restrict__ wl, const T* __restrict__ dy, T* __restrict__ d_o, T* __restrict__ d_loc,
    T* __restrict__ d_glin, float* __restrict__ partials, int B, int H, int L, int Dv, long long ldg, long long ldd, float eps,
    int silu_out, int tokens) {
  __shared__ float park[256][17];  // per thread: 8 dw_g + 8 dw_l sums of its channel octet (17: bank spread)
  const int d8n = Dv >> 3;
  const int nv = H * d8n;
  const int d8 = threadIdx.x & (d8n - 1);
  const OctetRows rows(B, L, nv, tokens);
  const size_t first = (size_t)blockIdx.x * tokens * nv * 8;
  const float inv_dv = 1.0f / (float)Dv;
  float w_g[8], w_l[8], dwg[8], dwl[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) w_g[j] = wg[d8 * 8 + j], w_l[j] = wl[d8 * 8 + j], dwg[j] = 0.f, dwl[j] = 0.f;
  struct Item {
    Raw8<T> o, l, g, dy;
    size_t head, gate;
  } next;
  const auto fetch = [&](int x, Item& it) {
    const Octet at(rows, x, nv, L);
    it.head = (((size_t)at.b * H + at.cv / d8n) * L + at.l) * (size_t)Dv + d8 * 8;
    const size_t row = (size_t)at.b * L + at.l;
    it.gate = row * (size_t)ldd + (size_t)at.cv * 8;
    it.o.load(o + it.head);
    it.l.load(loc + first + (size_t)x * 8);
    it.g.load(glin + row * (size_t)ldg + (size_t)at.cv * 8);
    it.dy.load(dy + first + (size_t)x * 8);
  };
  if ((int)threadIdx.x < rows.n) fetch(threadIdx.x, next);
  for (int x = threadIdx.x; x < rows.n; x += 256) {  // (whole groups of lanes stay or leave)
    const Item it = next;
    if (x + 256 < rows.n) fetch(x + 256, next);
    float xo[8], xl[8], xg[8], g[8];
    it.o.unpack(xo);
    it.l.unpack(xl);
    it.g.unpack(xg);
    it.dy.unpack(g);
    float so = 0.f, sl = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) so += xo[j] * xo[j], sl += xl[j] * xl[j];
    for (int m = 1; m < d8n; m <<= 1) {
      so += __shfl_xor(so, m);
      sl += __shfl_xor(sl, m);
    }
    const float ro = rsqrtf(so * inv_dv + eps);
    const float rl = rsqrtf(sl * inv_dv + eps);
    float don[8], dln[8], dgl[8];
    float mo = 0.f, ml = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = sigmoidf_(xg[j]);
      const float on = xo[j] * ro * w_g[j], ln = xl[j] * rl * w_l[j];
      float dy0 = g[j];
      if (silu_out) {
        const float y0 = on * s + ln * (1.f - s);
        const float sy = sigmoidf_(y0);
        dy0 *= sy * (1.f + y0 * (1.f - sy));
      }
      don[j] = dy0 * s;
      dln[j] = dy0 * (1.f - s);
      dgl[j] = dy0 * (on - ln) * s * (1.f - s);
      mo = __builtin_fmaf(don[j] * w_g[j], xo[j], mo);
      ml = __builtin_fmaf(dln[j] * w_l[j], xl[j], ml);
    }
    for (int m = 1; m < d8n; m <<= 1) {
      mo += __shfl_xor(mo, m);
      ml += __shfl_xor(ml, m);
    }
    const float co = ro * ro * mo * inv_dv, cl = rl * rl * ml * inv_dv;
    float eo[8], el[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      eo[j] = ro * (don[j] * w_g[j] - xo[j] * co);
      el[j] = rl * (dln[j] * w_l[j] - xl[j] * cl);
      dwg[j] = __builtin_fmaf(don[j] * ro, xo[j], dwg[j]);
      dwl[j] = __builtin_fmaf(dln[j] * rl, xl[j], dwl[j]);
    }
    Vec8<T>::store(d_o + it.head, eo);
    Vec8<T>::store(d_loc + first + (size_t)x * 8, el);
    Vec8<T>::store(d_glin + it.gate, dgl);
  }
  // thread (which, d) adds, in thread order, the parked sums of every thread whose octet holds channel d
#pragma unroll
  for (int j = 0; j < 8; ++j) park[threadIdx.x][j] = dwg[j], park[threadIdx.x][8 + j] = dwl[j];
  __syncthreads();
  if ((int)threadIdx.x < 2 * Dv) {
    const int which = threadIdx.x / Dv, d = threadIdx.x - which * Dv;
    const int want = d >> 3, slot = 8 * which + (d & 7);
    float total = 0.f;
    for (int t = want; t < 256; t += d8n) total += park[t][slot];
    partials[(size_t)blockIdx.x * (size_t)(2 * Dv) + threadIdx.x] = total;
  }
}

// Workgroups: 512, two a compute unit (both their registers and the column sum behind them).  us at 512 / 1024 / 2048: rows 5880 x 384
// bf16 13.0 / 13.4 / 14.8, fp32 16.4 / 18.9 / 20.8; 25088 x 384 28.8 / 29.4 / 31.4; 4704 x 768 16.0 / 17.7 / 17.9.
constexpr int kBlendBwdBlocks = 512;
// rows of partial sums there is room for: a workgroup for every 32 tokens of an image (what a caller has to bring), and up to
// kBlendBwdBlocks one for two tokens
static long long blend_bwd_rows(int B, int L) {
  const long long per_32 = (long long)B * ((L + 31) / 32), fine = std::min<long long>(((long long)B * L + 1) / 2, kBlendBwdBlocks);
  return std::max(fine, per_32);
}
size_t locality_blend_bwd_workspace(int B, int L, int Dv) {
  return (size_t)blend_bwd_rows(B, L) * 2 * Dv * sizeof(float);
}

// (a workspace without the rows beyond one for 32 tokens is enough)
size_t locality_blend_bwd_least_workspace(int B, int L, int Dv) { return (size_t)B * ((L + 31) / 32) * 2 * Dv * sizeof(float); }

int launch_locality_blend_bwd(const void* o, const void* loc, const void* glin, const float* wg, const float* wl,
                              const void* dy, void* d_o, void* d_loc, void* d_glin, float* dw, void* workspace, long long workspace_rows, int B,
                              int H, int L, int Dv, long long ldg, long long ldd, float eps, int silu_out, int io_dtype,
                              vig_sum_jobs* later, hipStream_t stream) {
  if (B > 65535 || !octet_rows_ok(B, L)) return -22;
  const int nv = H * (Dv / 8);
  const long long total = (long long)B * L, room = std::min<long long>(kBlendBwdBlocks, workspace_rows);
  // whole rounds of 256 octets, as few as the workgroups allow
  int rounds = (int)std::max<long long>(1, (total * nv + 256 * room - 1) / (256 * room)), tokens = octet_tokens(nv, rounds);
  while ((total + tokens - 1) / tokens > room) tokens = octet_tokens(nv, ++rounds);
  const dim3 grid((unsigned)((total + tokens - 1) / tokens)), block(256);
  float* partials = static_cast<float*>(workspace);
  if (io_dtype == 0)
    hipLaunchKernelGGL((locality_blend_bwd_kernel<float>), grid, block, 0, stream, (const float*)o, (const float*)loc,
                       (const float*)glin, wg, wl, (const float*)dy, (float*)d_o, (float*)d_loc, (float*)d_glin,
                       partials, B, H, L, Dv, ldg, ldd, eps, silu_out, tokens);
  else
    hipLaunchKernelGGL((locality_blend_bwd_kernel<uint16_t>), grid, block, 0, stream, (const uint16_t*)o,
                       (const uint16_t*)loc, (const uint16_t*)glin, wg, wl, (const uint16_t*)dy, (uint16_t*)d_o,
                       (uint16_t*)d_loc, (uint16_t*)d_glin, partials, B, H, L, Dv, ldg, ldd, eps, silu_out, tokens);
  if (hipGetLastError() != hipSuccess) return -5;
  if (later) return put_off(*later, partials, dw, (int)grid.x, 2 * Dv, false) ? 0 : -22;
  return launch_column_sum(partials, dw, (int)grid.x, 2 * Dv, stream);
}

}  // namespace vig
