// fp32 matrix products on the bf16 matrix cores (gfx950): out = A B^T (+ bias) (+ add), every operand in three bf16 pieces and six
// products each (f32_tiles.h: no larger error than fp32 fused multiply-adds).  The products of an fp32 training step: a layer
// (both operands with the contraction contiguous), its input gradient (the weight read across), its weight gradient (both read
// across; the column sums of the gradient, the bias gradient, on the way).
//
// Why not the BLAS library: its front end takes 22 us of host time a call, 183 calls a step, and a small model's step waits for
// the host (ViG-T, 9 images of 240 px: 9.1 ms, with this 6.3); and its error is three times as large (2.5e-7 against 8e-8 of the
// largest output at 2048 columns and a contraction of 384).
//
// A workgroup of four waves makes a 64 x 64 tile, a wave 32 x 32 of it, 32 contraction steps at a time through two LDS buffers: a
// thread fetches eight steps of one row of either operand two stages ahead, cuts them up and writes them as matrix-core operands,
// while the matrix instructions of the stage before run (twelve of 32 clocks a wave; the cutting up and the addresses take as many
// clocks of the vector unit).  Long contractions over few tiles (weight gradients) are split over workgroups, whose partial tiles a
// second kernel adds in a fixed order.  8100 rows, 2048 columns, contraction 384: 117 us (109 TFLOP/s in fp32; matrix cores busy 23 %, vector
// unit 33 %, LDS 24 %: two waves a SIMD that meet at a barrier a stage leave the rest; further waves do not fit the registers).
#include "f32_tiles.h"

namespace vig {

namespace {

constexpr int kMmTile = 64, kMmStep = 32;
constexpr int kMmOperand = 2 * 2 * 3 * 1024;  // bytes of one operand's stage: row halves x 16-step pieces x bf16 pieces
constexpr int kMmMaxSplit = 32;
constexpr int kMmAhead = 2;  // stages fetched ahead of the one being staged; a workgroup's stages are a multiple of it

struct MatmulArgs {
  const float *a, *b, *bias, *add;
  float *out, *partial, *sums;  // partial: [split][M][N] (null: straight to out); sums of A's rows: [split][M] (null: not wanted)
  long long lda, ldb, ldadd, ldo;
  int M, N, K, steps_per_split;
  unsigned a_bytes, b_bytes;
};

// eight contraction steps k0 .. k0 + 7 of row `row` (nothing beyond the matrix)
template <bool ACROSS>
__device__ __forceinline__ f32x8_t fetch8(rsrc_t r, int row, int rows, int k0, int K, unsigned ld) {
  f32x8_t x;
  if (ACROSS) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const unsigned off = row < rows && k0 + e < K ? ((unsigned)(k0 + e) * ld + (unsigned)row) * 4u : kOutOfRange;
      x[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    }
  } else {
    const unsigned off = row < rows && k0 < K ? ((unsigned)row * ld + (unsigned)k0) * 4u : kOutOfRange;
    const f32x4_t a = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    const f32x4_t b = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 16, 0));
    x = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  return x;
}
// row and octet of steps that a thread fetches: neighbouring lanes take neighbouring rows, so that the LDS writes of sixteen lanes
// are consecutive; four (16 rows) or one (64 rows) octets of a row in one instruction
template <bool ACROSS>
__device__ __forceinline__ void item_of(int tid, int& row, int& oct) {
  if (ACROSS) row = tid & 63, oct = tid >> 6;
  else row = (tid & 15) | ((tid >> 6) << 4), oct = (tid >> 4) & 3;
}
__device__ __forceinline__ void stage8(char* operand, int row, int oct, f32x8_t x) {
  const P3 p = split8(x);
  char* u = operand + ((row >> 5) * 2 + (oct >> 1)) * 3072;
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4_t*>(unit_ptr(u, i, (row & 31) + 32 * (oct & 1))) = p.p[i];
}

}  // namespace

template <bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void matmul_f32_kernel(MatmulArgs g) {
  __shared__ __align__(16) char lds[2][2][kMmOperand];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w >> 1, wn = w & 1;
  const int m0 = blockIdx.y * kMmTile, n0 = blockIdx.x * kMmTile;
  const rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.a), 0, g.a_bytes, 0x00020000);
  const rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.b), 0, g.b_bytes, 0x00020000);
  int arow, aoct, brow, boct;
  item_of<TA>(tid, arow, aoct);
  item_of<TB>(tid, brow, boct);
  // (steps_per_split is a multiple of kMmAhead; steps beyond the contraction are zeros)
  const int first = blockIdx.z * g.steps_per_split, steps = min(g.steps_per_split, (g.K + kMmStep - 1) / kMmStep - first);
  const unsigned lda = (unsigned)g.lda, ldb = (unsigned)g.ldb;
  f32x8_t xa[kMmAhead], xb[kMmAhead];
  const auto fetch = [&](int s, int slot) {
    xa[slot] = fetch8<TA>(ra, m0 + arow, g.M, (first + s) * kMmStep + 8 * aoct, g.K, lda);
    xb[slot] = fetch8<TB>(rb, n0 + brow, g.N, (first + s) * kMmStep + 8 * boct, g.K, ldb);
  };
  float sum = 0.f;  // of the fetched steps of A's row
  const auto stage = [&](int slot, int buf, bool own) {
    const f32x8_t x = xa[slot];
    if (TA) sum += own ? ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])) : 0.f;
    stage8(lds[buf][0], arow, aoct, x);
    stage8(lds[buf][1], brow, boct, xb[slot]);
  };
  f32x16_t big = {0.f}, small = {0.f};
#pragma unroll
  for (int j = 0; j < kMmAhead; ++j) fetch(j, j);
  stage(0, 0, true);
  fetch(kMmAhead, 0);
  lds_barrier();
  for (int s0 = 0; s0 < steps; s0 += kMmAhead) {
    // (no branch in here: the waits for what is under way would have to assume that it was not taken)
#pragma unroll
    for (int j = 0; j < kMmAhead; ++j) {
      const int s = s0 + j, slot = (j + 1) % kMmAhead;
      char* ta = lds[s & 1][0] + wm * 6144;
      char* tb = lds[s & 1][1] + wn * 6144;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) mfma6(load_p3(ta, ks, lane), load_p3(tb, ks, lane), big, small);
      stage(slot, (s + 1) & 1, s + 1 < steps);
      fetch(s + 1 + kMmAhead, slot);
      lds_barrier();
    }
  }
  big += small;
  const int n = n0 + 32 * wn + r;
  unsigned at[16];  // rows (none beyond the matrix)
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const int m = m0 + 32 * wm + 8 * (c >> 2) + 4 * h + (c & 3);
    at[c] = m < g.M && n < g.N ? (unsigned)m : kOutOfRange;
  }
  // An infinity has no pieces (it less itself is no number), and a leading product can overflow where the whole does not: elements
  // that did not come out finite are made again from plain multiply-adds.
  bool finite = true;
#pragma unroll
  for (int c = 0; c < 16; ++c) finite = finite && __builtin_fabsf(big[c]) < __builtin_inff();
  if (__builtin_expect(__any(!finite), 0)) {
    f32x16_t plain = {0.f};
    const int last = min(g.K, (first + steps) * kMmStep);
    for (int k = first * kMmStep; k < last; ++k) {
      const float y = n < g.N ? g.b[TB ? (size_t)k * g.ldb + n : (size_t)n * g.ldb + k] : 0.f;
#pragma unroll
      for (int c = 0; c < 16; ++c)
        plain[c] = fmaf(at[c] != kOutOfRange ? g.a[TA ? (size_t)k * g.lda + at[c] : (size_t)at[c] * g.lda + k] : 0.f, y, plain[c]);
    }
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (!(__builtin_fabsf(big[c]) < __builtin_inff())) big[c] = plain[c];
  }
  if (g.partial) {
    float* part = g.partial + (size_t)blockIdx.z * g.M * g.N;
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (at[c] != kOutOfRange) part[(size_t)at[c] * g.N + n] = big[c];
  } else {
    if (g.bias && n < g.N) big += g.bias[n];
    if (g.add) {
      float add[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) add[c] = at[c] != kOutOfRange ? g.add[(size_t)at[c] * g.ldadd + n] : 0.f;
#pragma unroll
      for (int c = 0; c < 16; ++c) big[c] += add[c];
    }
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (at[c] != kOutOfRange) g.out[(size_t)at[c] * g.ldo + n] = big[c];
  }
  if (TA && g.sums && blockIdx.x == 0) {
    float* red = reinterpret_cast<float*>(lds);  // (everybody is through with the stages)
    red[tid] = sum;
    __syncthreads();
    if (tid < 64 && m0 + tid < g.M)
      g.sums[(size_t)blockIdx.z * g.M + m0 + tid] = (red[tid] + red[64 + tid]) + (red[128 + tid] + red[192 + tid]);
  }
}

// adds the partial tiles of a split contraction, four columns a thread, and the partial sums of A's rows behind them
__global__ __launch_bounds__(256) void matmul_f32_sum_kernel(MatmulArgs g, float* __restrict__ sums_out, int split) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4, total = (long long)g.M * g.N;
  if (i < total) {
    const int m = (int)(i / g.N), n = (int)(i - (long long)m * g.N);
    f32x4_t y = *reinterpret_cast<const f32x4_t*>(g.partial + i);
    for (int s = 1; s < split; ++s) y += *reinterpret_cast<const f32x4_t*>(g.partial + (size_t)s * total + i);
    if (g.bias) y += f32x4_t{g.bias[n], g.bias[n + 1], g.bias[n + 2], g.bias[n + 3]};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (g.add) y[e] += g.add[(size_t)m * g.ldadd + n + e];
      g.out[(size_t)m * g.ldo + n + e] = y[e];
    }
  }
  const long long m = i / 4 - (total + 3) / 4;
  if (sums_out && m >= 0 && m < g.M) {
    float y = g.sums[m];
    for (int s = 1; s < split; ++s) y += g.sums[(size_t)s * g.M + m];
    sums_out[m] = y;
  }
}

// Workgroups that one contraction is split over, so that two workgroups a compute unit have at least eight stages each (at least
// four: the same times within 1 % at 400 and 1960 rows).
static int matmul_split(long long M, int N, long long K) {
  if (N % 4 != 0) return 1;
  const long long tiles = ((M + kMmTile - 1) / kMmTile) * ((N + kMmTile - 1) / kMmTile), steps = (K + kMmStep - 1) / kMmStep;
  long long s = 512 / tiles;
  if (s > steps / 8) s = steps / 8;
  if (s > kMmMaxSplit) s = kMmMaxSplit;
  return s < 2 ? 1 : (int)s;
}

size_t matmul_f32_workspace(long long M, int N, long long K) {
  const int s = matmul_split(M, N, K);
  return s == 1 ? 0 : ((size_t)s * M * N + (size_t)s * M) * sizeof(float);
}

// 32-bit offsets, whole octets of steps where the contraction is contiguous, and one grid
bool matmul_f32_supported(long long lda, bool ta, long long ldb, bool tb, long long M, int N, long long K) {
  const long long limit = 1LL << 29;  // elements: 2 GiB
  const auto extent = [](long long rows, long long ld, bool across, long long K) { return across ? (K - 1) * ld + rows : (rows - 1) * ld + K; };
  return M > 0 && N > 0 && K > 0 && M < limit && K < limit && extent(M, lda, ta, K) < limit / 2 && extent(N, ldb, tb, K) < limit / 2 &&
         (ta || (K % 8 == 0 && lda % 4 == 0)) && (tb || (K % 8 == 0 && ldb % 4 == 0)) && (M + kMmTile - 1) / kMmTile <= 65535 && !(ta && !tb);
}

int launch_matmul_f32(const float* a, long long lda, bool ta, const float* b, long long ldb, bool tb, const float* bias, const float* add,
                      long long ldadd, float* out, long long ldo, float* a_sums, long long M, int N, long long K, void* workspace,
                      hipStream_t stream) {
  const auto bytes = [](long long rows, long long ld, bool across, long long K) {
    return (unsigned)(4 * (across ? (K - 1) * ld + rows : (rows - 1) * ld + K));
  };
  const int split = matmul_split(M, N, K), steps = (int)((K + kMmStep - 1) / kMmStep);
  const int per_split = ((steps + split - 1) / split + kMmAhead - 1) / kMmAhead * kMmAhead;
  MatmulArgs g{a, b, bias, add, out, nullptr, a_sums, lda, ldb, ldadd, ldo, (int)M, N, (int)K, per_split, bytes(M, lda, ta, K),
               bytes(N, ldb, tb, K)};
  const int parts = (steps + g.steps_per_split - 1) / g.steps_per_split;
  if (split > 1) {
    g.partial = (float*)workspace;
    g.sums = a_sums ? g.partial + (size_t)split * M * N : nullptr;
  }
  const dim3 grid((N + kMmTile - 1) / kMmTile, (unsigned)((M + kMmTile - 1) / kMmTile), parts);
  if (ta) hipLaunchKernelGGL((matmul_f32_kernel<true, true>), grid, dim3(256), 0, stream, g);
  else if (tb) hipLaunchKernelGGL((matmul_f32_kernel<false, true>), grid, dim3(256), 0, stream, g);
  else hipLaunchKernelGGL((matmul_f32_kernel<false, false>), grid, dim3(256), 0, stream, g);
  if (split > 1) {
    const long long threads = (long long)M * N / 4 + (a_sums ? M : 0);
    hipLaunchKernelGGL(matmul_f32_sum_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, g, a_sums, parts);
  }
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace vig
