// Weight and bias gradients of a linear layer over bf16 rows:  dW[n, k] = sum_t dY[t, n] X[t, k],  db[n] = sum_t dY[t, n],
// fp32 accumulation and fp32 results, in a fixed order (a training step is reproducible bit for bit).
//
// The output is small (a ViG-S layer's widths: 16 to 2048 by 16 to 1024) and the contraction long (25 088 tokens at a batch
// of 128), so the tokens are split over workgroups: 128 x 128 tiles of dW times as many token ranges as give about two
// workgroups per CU, partial tiles in a workspace, a second kernel that adds them.  (The library's GEMM for this shape runs
// 24 to 100 workgroups: 100 to 135 us per layer and weight at B128, 8.3 of the 23.9 ms of a ViG-S training step.)
//
// A workgroup streams 32 tokens of both operands at a time through four LDS buffers, direct-to-LDS loads of whole
// 256-byte row pieces, three stages in flight (16 KB each: what the L2's latency asks for).  The contraction runs over
// tokens, so an operand fragment needs 8 tokens of one channel: ds_read_b64_tr_b16 hands every lane of a group of sixteen
// four tokens of its channel out of a 4 x 16 block.  The 32-byte units of a row are swapped among themselves by the row
// number (the loads fetch them that way), so that the four rows of such a block lie in different banks.
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

constexpr int kWgTile = 128;    // channels of either operand per workgroup
constexpr int kWgStage = 32;    // tokens per stage
constexpr int kWgBuffers = 4;
constexpr int kWgHalf = kWgStage * kWgTile * 2;  // bytes of one operand's stage
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_t;

struct WgradArgs {
  const uint16_t *dy, *x;
  long long ldy, ldx;
  float* part;   // [splits][N][K] (or the result itself for one split)
  float* bpart;  // [splits][N] or null
  int T, N, K, per;  // tokens per split, a multiple of the stage
  int tn, tiles, splits;  // tiles along N, tiles of dW, token ranges
};

template <bool BIAS>
__global__ __launch_bounds__(256, 2) void linear_wgrad_kernel(WgradArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // workgroups go to the XCDs in turn: each XCD gets a run of consecutive (range, tile) pairs, so that its L2 serves a
  // range's rows to that range's tiles (dealt out one by one, every XCD fetched every row: 54 -> 36 us at N 1280, K 384)
  const int total = a.splits * a.tiles, run = (total + 7) >> 3;
  const int at = ((int)blockIdx.x & 7) * run + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= run || at >= total) return;
  const int split = at / a.tiles, tile = at - split * a.tiles;
  const int tk = tile / a.tn;
  const int n0 = (tile - tk * a.tn) * kWgTile, k0 = tk * kWgTile;
  const int t0 = split * a.per, t1 = min(a.T, t0 + a.per);
  const int nstage = (t1 - t0 + kWgStage - 1) / kWgStage;
  const int wn = 64 * (wave & 1), wk = 64 * (wave >> 1);  // this wave's 64 x 64 of the tile

  // a wave's share of a stage: rows 8*wave .. +8 of both operands, four rows (1 KB) per load.  Rows and channels past the
  // end are read from the last row and from channel 0 (every load is issued: the waits below count them); such rows are
  // cleared, such channels' results are not stored.
  const int lrow = 8 * wave + (lane >> 4), piece = lane & 15;
  int coln[2], colk[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int col = 16 * ((piece >> 1) ^ ((lrow + 4 * i) & 7)) + 8 * (piece & 1);  // channel the 16 bytes at this place hold
    coln[i] = n0 + col < a.N ? n0 + col : 0;
    colk[i] = k0 + col < a.K ? k0 + col : 0;
  }
  const uint32_t lds0 = lds_offset(smem);
  const auto fetch = [&](int stage) {
    const uint32_t buf = lds0 + (stage % kWgBuffers) * (2 * kWgHalf);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = min(t0 + stage * kWgStage + lrow + 4 * i, t1 - 1);
      const uint32_t dst = buf + (8 * wave + 4 * i) * 256;
      load_to_lds16(a.dy + (size_t)t * a.ldy + coln[i], dst);
      load_to_lds16(a.x + (size_t)t * a.ldx + colk[i], dst + kWgHalf);
    }
  };
  // rows past the last token of the range contribute nothing: both operands' are zeroed (one of them might hold a NaN)
  const auto clear_tail = [&](int stage) {
    char* buf = smem + (stage % kWgBuffers) * (2 * kWgHalf);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = lrow + 4 * i;
      if (t0 + stage * kWgStage + row >= t1) {
        *reinterpret_cast<u32x4_t*>(buf + row * 256 + 16 * piece) = u32x4_t{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(buf + kWgHalf + row * 256 + 16 * piece) = u32x4_t{0u, 0u, 0u, 0u};
      }
    }
  };
  // byte offsets, inside an operand's stage, of this lane's part of the fragment of channel block b (32 channels), tokens
  // 8h + 4q .. +4 of a k-step: source lane = (token (l>>2)&3, channels 4*(l&3) of the group's sixteen)
  int offn[2][2], offk[2][2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int tok = 8 * h + 4 * q + ((lane >> 2) & 3), half = (lane >> 4) & 1;
      offn[b][q] = tok * 256 + 32 * (((wn >> 4) + 2 * b + half) ^ (tok & 7)) + 8 * (lane & 3);
      offk[b][q] = kWgHalf + tok * 256 + 32 * (((wk >> 4) + 2 * b + half) ^ (tok & 7)) + 8 * (lane & 3);
    }
  f32x16_t acc[2][2], accb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accb[i] = f32x16_t{0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{0.f};
  }
  const bool with_bias = BIAS && k0 == 0 && wk == 0;
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  const auto frag = [&](char* buf, int off) {
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(buf + off));
    return lo;
  };
  for (int s = 0; s < kWgBuffers - 1; ++s)
    if (s < nstage) fetch(s);
  for (int s = 0; s < nstage; ++s) {
    // this wave's share of stage s has landed: the (up to two) later stages' four loads each may still be out
    const int later = min(nstage - 1 - s, kWgBuffers - 2);
    if (later == 2) wait_vmem<8>();
    else if (later == 1) wait_vmem<4>();
    else wait_vmem<0>();
    if (t0 + (s + 1) * kWgStage > t1) {
      clear_tail(s);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    asm volatile("s_barrier" ::: "memory");
    if (s + kWgBuffers - 1 < nstage) fetch(s + kWgBuffers - 1);  // (the buffer read in stage s - 1: everyone is past it)
    char* buf = smem + (s % kWgBuffers) * (2 * kWgHalf);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4_t fn[2], fk[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const s16x4_t n_lo = frag(buf, offn[b][0] + ks * 4096), n_hi = frag(buf, offn[b][1] + ks * 4096);
        const s16x4_t k_lo = frag(buf, offk[b][0] + ks * 4096), k_hi = frag(buf, offk[b][1] + ks * 4096);
        fn[b] = __builtin_bit_cast(u32x4_t, __builtin_shufflevector(n_lo, n_hi, 0, 1, 2, 3, 4, 5, 6, 7));
        fk[b] = __builtin_bit_cast(u32x4_t, __builtin_shufflevector(k_lo, k_hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(fn[i], fk[j], acc[i][j]);
      if (with_bias) {
#pragma unroll
        for (int i = 0; i < 2; ++i) accb[i] = mfma(fn[i], ones, accb[i]);
      }
    }
  }
  float* part = a.part + (size_t)split * a.N * a.K;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + wk + 32 * j + r;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const int n = n0 + wn + 32 * i + 8 * (c >> 2) + 4 * h + (c & 3);
        if (n < a.N && k < a.K) part[(size_t)n * a.K + k] = acc[i][j][c];
      }
    }
  if (with_bias && r == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const int n = n0 + wn + 32 * i + 8 * (c >> 2) + 4 * h + (c & 3);
        if (n < a.N) a.bpart[(size_t)split * a.N + n] = accb[i][c];
      }
  }
}

// sums of the splits' partial results: 32 columns of four values by eight groups of splits per block, the groups' sums
// added in LDS in order; the last blocks do the bias (one value a column)
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const float* __restrict__ part, float* __restrict__ dw, long long n4,
                                                        const float* __restrict__ bpart, float* __restrict__ db, int N,
                                                        int splits) {
  __shared__ f32x4_t sums[8][32];
  const int col = threadIdx.x & 31, grp = threadIdx.x >> 5;
  const long long i = (long long)blockIdx.x * 32 + col;
  const bool bias = i >= n4;
  const long long j = i - n4;
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (!bias) {
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(part) + i;
#pragma unroll 4
    for (int k = grp; k < splits; k += 8) s += p[(long long)k * n4];
  } else if (db && j < N) {
    for (int k = grp; k < splits; k += 8) s[0] += bpart[(long long)k * N + j];
  }
  sums[grp][col] = s;
  __syncthreads();
  if (grp != 0) return;
#pragma unroll
  for (int k = 1; k < 8; ++k) s += sums[k][col];
  if (!bias) reinterpret_cast<f32x4_t*>(dw)[i] = s;
  else if (db && j < N) db[j] = s[0];
}

int wgrad_splits(long long T, int N, int K) {
  const long long tiles = (long long)((N + kWgTile - 1) / kWgTile) * ((K + kWgTile - 1) / kWgTile);
  long long s = 512 / tiles;                       // two workgroups per CU
  const long long most = (T + 255) / 256;          // at least eight stages each
  if (s > most) s = most;
  if (s > 128) s = 128;
  if (s > 8) s = s / 8 * 8;                        // a range's tiles stay on one XCD
  return s < 1 ? 1 : (int)s;
}

}  // namespace

bool linear_wgrad_supported(long long T, int N, int K) {
  return T > 0 && T < 0x7fffffffLL - 4096 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 && N <= (1 << 20) && K <= (1 << 20);
}
size_t linear_wgrad_workspace(long long T, int N, int K) {
  return (size_t)wgrad_splits(T, N, K) * ((size_t)N * K + N) * sizeof(float);
}

int launch_linear_wgrad(const void* dy, long long ldy, const void* x, long long ldx, long long T, int N, int K, float* dw,
                        float* db, void* workspace, hipStream_t stream) {
  static bool attr_done[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -5;
  constexpr int lds = kWgBuffers * 2 * kWgHalf;
  if (!attr_done[dev]) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(linear_wgrad_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
        hipFuncSetAttribute(reinterpret_cast<const void*>(linear_wgrad_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return -5;
    attr_done[dev] = true;
  }
  const int want = wgrad_splits(T, N, K);
  WgradArgs a{};
  a.dy = (const uint16_t*)dy, a.x = (const uint16_t*)x, a.ldy = ldy, a.ldx = ldx;
  a.T = (int)T, a.N = N, a.K = K;
  a.per = (int)(((T + want - 1) / want + kWgStage - 1) / kWgStage * kWgStage);
  const int splits = (int)((T + a.per - 1) / a.per);
  float* ws = (float*)workspace;
  a.part = splits > 1 ? ws : dw;
  a.bpart = db ? (splits > 1 ? ws + (size_t)splits * N * K : db) : nullptr;
  a.tn = (N + kWgTile - 1) / kWgTile, a.tiles = a.tn * ((K + kWgTile - 1) / kWgTile), a.splits = splits;
  const dim3 grid(8 * ((splits * a.tiles + 7) / 8));
  if (db) hipLaunchKernelGGL(linear_wgrad_kernel<true>, grid, dim3(256), lds, stream, a);
  else hipLaunchKernelGGL(linear_wgrad_kernel<false>, grid, dim3(256), lds, stream, a);
  if (splits > 1) {
    const long long n4 = (long long)N * K / 4, all = n4 + (db ? N : 0);
    hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)((all + 31) / 32)), dim3(256), 0, stream, a.part, dw, n4, a.bpart, db, N, splits);
  }
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace vig
