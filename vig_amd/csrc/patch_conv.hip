// First convolution of ViG's v2 patch embedding (classification/models/vig.py:651: kernel 9, stride 8, padding 1,
// 3 input channels) as an implicit GEMM on the matrix cores, reading the images in the [B, C, H, W] layout they
// arrive in and writing channels-last rows [B, OH, OW, Cout] -- what the LayerNorm kernel behind it consumes.
//
// One workgroup produces up to 32 pixels of one output row (b, oy), all Cout channels.  Its input is the slab of
// Cin * KH image rows (27 for 3 channels x 9 kernel rows), 256 columns of them; each goes to LDS shifted by one element, so
// that input column ix of the piece sits at element ix + 1 and element 0 is the column in front (the left padding): pixel ox then finds its first eight kernel
// columns at elements 8*ox .. 8*ox+7, and the rest of 16 (9 real ones, the weights of the others are zero) in a second copy of the row, eight elements on: two aligned
// 16-byte reads.  Either copy has zeros for the columns that the kernel does not have, as the weights do: they belong to the next window, and a pixel that is not
// finite stays out of a window it is not in.  us, one row without zeros / this / masks at the reads, 256 images of 224 px: 96 channels 37.3 / 38.2 / 39.3, with the norm
// 54.6 / 57.9 / 58.1 (55.0 with its sums' present pitch); 192 57.9 / 59.5 / 58.5, 94.7 / 97.5 / 102.9; 384 81.1 / 82.3 / 89.5.  The
// contraction runs over (channel, kernel row) steps of 16 kernel columns: one v_mfma_f32_32x32x16_bf16 per step with
// the weights (matrix rows = output channels) in registers for the life of the workgroup and the pixels as columns.
// Matrix rows are assigned channels so that a lane ends with 16 consecutive channels of one pixel (32 contiguous
// bytes).  The one-element shift costs no unaligned access: a lane takes the last element of its left neighbour's
// 16-byte chunk (a lane shuffle) and funnel-shifts its own chunk behind it.
// Rows wider than 248 columns are cut into pieces of 256 (a wide row went through a layout copy and the convolution library:
// 101 us at 8 x 1024 x 1024, 27 us in pieces).
#include "common.h"
#include "launch.h"

namespace vig {

namespace {

constexpr int kPcStride = 8;       // convolution stride = elements per pixel step in a staged row
constexpr int kPcRowElems = 512;   // staged row: 32 chunks of 8 elements, and the 32 behind each
constexpr int kPcKW = 16;          // kernel columns per contraction step (weights beyond the real width are zero)

// The layer norm behind it (NORM), as layernorm_kernel gives it for the stored rows, bit for bit: + pre_bias (rounded), norm, SiLU.
struct PcNorm {
  const float *weight, *bias, *pre_bias;  // [Cout]; pre_bias may be null
  float eps;
  int silu;
};
// the sum that layernorm_kernel's lanes, one to an octet, come to by exchange
template <int N>
__device__ __forceinline__ float octet_tree(const float* row) {
  constexpr int G = 32;
  static_assert(N <= G, "one octet to a lane of the kernel behind");
  float a[G];
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(row + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) a[i + j] = v[j];
  }
#pragma unroll
  for (int i = N; i < G; ++i) a[i] = 0.f;
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < off; ++i) a[i] += a[i + off];
  return a[0];
}

// NORM: the workgroup has whole rows of channels, so their norm needs two exchanges of octet sums through LDS (a barrier each, one of
// which takes the place of the one in front of the next staging) instead of a pass over memory.  us, two kernels / this: 96 channels, one image of
// 224 px 8.5 / 6.7, 8 9.5 / 6.9, 256 76 / 55, 8 of 1024 px 50 / 35; 192, 1 9.4 / 7.7, 32 24 / 19, 256 100 / 97, 224, 256 103 / 95, 256, 256 110 / 95 (one workgroup to a CU: its 190
// registers brought down to 168 for a second one spill 13 to 18, 124).  At 384 channels the 48 octets spill (60 images 55 / 73): two kernels.
template <int KS, int NW, bool NORM>  // KS = Cin * KH contraction steps, NW = Cout / 32 waves
__global__ __launch_bounds__(NW > 8 ? 64 * NW : 512) void patch_conv_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wp,
                                                         uint16_t* __restrict__ y, int Cin, int H, int W, int KH, int KW,
                                                         int OH, int OW, int Cout, int pieces, int nitems, PcNorm norm) {
  // floats between two pixels' octet sums: an odd number of fours, so that 16 pixels meet every bank once (seven waves, 32 floats, all pixels in the same four
  // banks: 224 channels, 256 images of 224 px, 133 us for 95)
  constexpr int kPitch = 4 * (NW | 1);
  static_assert(kPitch >= 4 * NW && kPitch % 8 == 4, "pixels spread over the banks");
  extern __shared__ __align__(16) char smem[];
  uint16_t* slab = reinterpret_cast<uint16_t*>(smem);  // [KS][kPcRowElems]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int nwaves = NW;
  const int r = lane & 31, h = lane >> 5;
  float* const stats = reinterpret_cast<float*>(smem + KS * kPcRowElems * 2);  // [sums, squares][32 pixels][octets]
  float* const params = stats + 2 * 32 * kPitch;                              // weight, bias, pre_bias [32 NW]
  if constexpr (NORM) {
    for (int i = threadIdx.x; i < 32 * NW; i += blockDim.x)
      params[i] = norm.weight[i], params[32 * NW + i] = norm.bias[i], params[64 * NW + i] = norm.pre_bias ? norm.pre_bias[i] : 0.f;
  }
  // this wave's 32 output channels: matrix row i holds channel 16*((i>>2)&1) + 4*(i>>3) + (i&3) of the tile, which
  // leaves lane (r, h) with channels 16h .. 16h+15 of pixel r in its accumulator registers
  const int chan_of_row = 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
  u32x4_t wf[KS];
#pragma unroll
  for (int t = 0; t < KS; ++t)
    wf[t] = *reinterpret_cast<const u32x4_t*>(wp + ((size_t)(32 * wave + chan_of_row) * KS + t) * kPcKW + 8 * h);
  // the kernel's columns among the first eight and the second
  u32x4_t first, second;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n0 = KW - 2 * j, n1 = n0 - 8;
    first[j] = n0 >= 2 ? ~0u : n0 == 1 ? 0xFFFFu : 0u;
    second[j] = n1 >= 2 ? ~0u : n1 == 1 ? 0xFFFFu : 0u;
  }
  // image rows of the slab a thread fetches: half-wave (wave, h) takes slab rows 2*p + h, p = wave, wave + nwaves, ..;
  // the chunks of the next output row are in flight while the current one is multiplied
  constexpr int kMaxP = ((KS + 1) / 2 + NW - 1) / NW;  // row pairs per wave
  auto fetch = [&](int item, u32x4_t (&v)[kMaxP], uint32_t (&front)[kMaxP]) {
    const int row = item / pieces, c0 = (item - row * pieces) * 256;
    const int b = row / OH, oy = row - b * OH;
#pragma unroll
    for (int i = 0; i < kMaxP; ++i) {
      const int t = 2 * (wave + i * nwaves) + h;
      const int c = t / KH, ky = t - c * KH;
      const int iy = oy * kPcStride - 1 + ky;
      v[i] = u32x4_t{0u, 0u, 0u, 0u};
      front[i] = 0u;
      if (item < nitems && t < KS && iy >= 0 && iy < H) {
        const uint16_t* p = x + (((size_t)b * Cin + c) * H + iy) * (size_t)W + c0;
        if (c0 + r * 8 < W) v[i] = *reinterpret_cast<const u32x4_t*>(p + r * 8);
        if (c0 > 0 && r == 0) front[i] = *reinterpret_cast<const uint32_t*>(p - 2);
      }
    }
  };
  u32x4_t v[kMaxP];
  uint32_t front[kMaxP];
  fetch(blockIdx.x, v, front);
  for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
    // ---- stage the slab: lane r = 16-byte chunk r of its image row, shifted by one element ----
#pragma unroll
    for (int i = 0; i < kMaxP; ++i) {
      const int t = 2 * (wave + i * nwaves) + h;
      uint32_t prev = __shfl(v[i][3], (r + 31) & 31, 32);  // the left neighbour's last pair; chunk 0 has the column in front there
      const uint32_t last = prev >> 16;                    // (chunk 0: the last chunk's)
      if (r == 0) prev = front[i];
      u32x4_t o;
      o[0] = __builtin_amdgcn_alignbit(v[i][0], prev, 16);
      o[1] = __builtin_amdgcn_alignbit(v[i][1], v[i][0], 16);
      o[2] = __builtin_amdgcn_alignbit(v[i][2], v[i][1], 16);
      o[3] = __builtin_amdgcn_alignbit(v[i][3], v[i][2], 16);
      if (t < KS) {
        *reinterpret_cast<u32x4_t*>(slab + t * kPcRowElems + r * 8) = o & first;
        // chunk r is what follows chunk r - 1; behind the last one there is its pixel's ninth column
        if (r == 0) o = u32x4_t{last, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(slab + t * kPcRowElems + 256 + 8 * ((r + 31) & 31)) = o & second;
      }
    }
    __syncthreads();
    fetch(item + gridDim.x, v, front);
    // ---- pixels x channels: KS contraction steps ----
    f32x16_t acc;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.f;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      const u32x4_t px = *reinterpret_cast<const u32x4_t*>(slab + t * kPcRowElems + r * kPcStride + 256 * h);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf[t]),
                                                    __builtin_bit_cast(bf16x8_t, px), acc, 0, 0, 0);
    }
    u32x4_t lo, hi;
    const auto pack = [&](const auto& v) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo[j] = pack_bf16x2(v[2 * j], v[2 * j + 1]);
        hi[j] = pack_bf16x2(v[8 + 2 * j], v[8 + 2 * j + 1]);
      }
    };
    pack(acc);
    if constexpr (NORM) {
      float s[16];
      const auto unpack = [&] {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s[2 * j] = bf16lo_to_f32(lo[j]), s[2 * j + 1] = bf16hi_to_f32(lo[j]);
          s[8 + 2 * j] = bf16lo_to_f32(hi[j]), s[9 + 2 * j] = bf16hi_to_f32(hi[j]);
        }
      };
      const float* const mine = params + 32 * wave + 16 * h;
      unpack();
      if (norm.pre_bias) {
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] += mine[64 * NW + j];
        pack(s);
        unpack();
      }
      float* const place = stats + r * kPitch + 4 * wave + 2 * h;
      float sum[2] = {0.f, 0.f}, sq[2] = {0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 16; ++j) sum[j >> 3] += s[j];
      *reinterpret_cast<u32x2_t*>(place) = u32x2_t{__float_as_uint(sum[0]), __float_as_uint(sum[1])};
      __syncthreads();  // (and nobody reads the slab any more)
      const float mean = octet_tree<4 * NW>(stats + r * kPitch) / (float)(32 * NW);
#pragma unroll
      for (int j = 0; j < 16; ++j) s[j] -= mean, sq[j >> 3] = __builtin_fmaf(s[j], s[j], sq[j >> 3]);
      *reinterpret_cast<u32x2_t*>(place + 32 * kPitch) = u32x2_t{__float_as_uint(sq[0]), __float_as_uint(sq[1])};
      __syncthreads();
      const float rstd = 1.0f / sqrtf(octet_tree<4 * NW>(stats + (32 + r) * kPitch) / (float)(32 * NW) + norm.eps);
#pragma unroll
      for (int j = 0; j < 16; ++j) s[j] = __builtin_fmaf(s[j] * rstd, mine[j], mine[32 * NW + j]);
      pack(s);
      if (norm.silu) {
        unpack();
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = s[j] * sigmoidf_(s[j]);
        pack(s);
      }
    }
    const int row = item / pieces, ox = (item - row * pieces) * 32 + r;
    if (ox < OW) {
      uint16_t* dst = y + ((size_t)row * OW + ox) * (size_t)Cout + 32 * wave + 16 * h;
      *reinterpret_cast<u32x4_t*>(dst) = lo;
      *reinterpret_cast<u32x4_t*>(dst + 8) = hi;
    }
    if (!NORM) __syncthreads();  // the next step's staging overwrites the slab
  }
}

}  // namespace

bool patch_conv_supported(int Cin, int H, int W, int KH, int KW, int stride, int padding, int Cout) {
  if (stride != kPcStride || padding != 1 || KW < 1 || KW > kPcKW || Cin * KH != 27) return false;
  if (W % 8 != 0 || H < 1 || (W > 248 && KW > 9)) return false;  // (a piece holds nine columns of its last pixel)
  const int OW = (W + 2 - KW) / stride + 1;
  // (twelve waves, one workgroup a CU: 384 channels, 224 px, 1 image 12.4 us, 40 21.3, where the library took 39.7 for 32 and 21 beside it)
  return OW >= 1 && Cout % 32 == 0 && ((Cout >= 64 && Cout <= 256) || Cout == 384);
}

static int launch(const void* x, const void* w_packed, void* y, int B, int Cin, int H, int W, int KH, int KW, int Cout, const PcNorm* norm,
                  hipStream_t stream) {
  if (!patch_conv_supported(Cin, H, W, KH, KW, kPcStride, 1, Cout)) return -95;
  const int OH = (H + 2 - KH) / kPcStride + 1, OW = (W + 2 - KW) / kPcStride + 1;
  const int pieces = (OW + 31) / 32;
  if (OH < 1 || (long long)B * OH * pieces > 0x7fffffffLL - 4096 || Cout / 32 < 2) return -95;
  const int nitems = B * OH * pieces;
  // Two workgroups to a CU of up to four waves, one of more; each walks pieces grid apart.  Of more waves one has enough under way, and a second one a CU, whether it
  // fits beside the first (up to 192 channels without the norm: 168 registers) or not, only fetches the weights again, 3 us a launch at any size: us, two to a CU / one, 16
  // and 256 images of 224 px: 160 channels 11.4 / 8.6, 61.4 / 58.4, with the norm 14.3 / 11.4, 98.8 / 95.5; 192 12.1 / 8.9, 62.4 / 59.0, 15.1 / 11.6, 100.6 / 97.0; 224 12.2 /
  // 8.9, 62.4 / 58.5; 256 13.1 / 9.5, 65.6 / 62.2, 16.4 / 12.3, 99.5 / 94.9; 384, 16 18.9 / 13.4, 128 50.8 / 42.5.
  const int most = Cout > 128 ? 256 : 512, grid = nitems < most ? nitems : most;
  const size_t lds = (size_t)27 * kPcRowElems * sizeof(uint16_t) + (norm ? 4 * (2 * 32 * 4 * (Cout / 32 | 1) + 3 * Cout) : 0);
#define VIG_PC_CASE(NW)                                                                                            \
  case NW:                                                                                                         \
    hipLaunchKernelGGL((norm ? patch_conv_kernel<27, NW, (NW <= 8)> : patch_conv_kernel<27, NW, false>), dim3(grid), dim3(64 * NW), lds, stream, \
                       (const uint16_t*)x, (const uint16_t*)w_packed, (uint16_t*)y, Cin, H, W, KH, KW, OH, OW, Cout, pieces, nitems,          \
                       norm ? *norm : PcNorm{});                                                                                        \
    break
  switch (Cout / 32) {
    VIG_PC_CASE(2);
    VIG_PC_CASE(3);
    VIG_PC_CASE(4);
    VIG_PC_CASE(5);
    VIG_PC_CASE(6);
    VIG_PC_CASE(7);
    VIG_PC_CASE(8);
    VIG_PC_CASE(12);
    default:
      return -95;
  }
#undef VIG_PC_CASE
  return hipGetLastError() == hipSuccess ? 0 : -5;
}
int launch_patch_conv(const void* x, const void* w_packed, void* y, int B, int Cin, int H, int W, int KH, int KW, int Cout, hipStream_t stream) {
  return launch(x, w_packed, y, B, Cin, H, W, KH, KW, Cout, nullptr, stream);
}
int launch_patch_conv_norm(const void* x, const void* w_packed, const float* weight, const float* bias, const float* pre_bias, void* y, int B,
                           int Cin, int H, int W, int KH, int KW, int Cout, float eps, int silu, hipStream_t stream) {
  if (Cout > 256) return -95;
  const PcNorm norm{weight, bias, pre_bias, eps, silu};
  return launch(x, w_packed, y, B, Cin, H, W, KH, KW, Cout, &norm, stream);
}

}  // namespace vig
