// Weight and bias gradients of a linear layer over bf16 rows:  dW[n, k] = sum_t dY[t, n] X[t, k],  db[n] = sum_t dY[t, n],
// fp32 accumulation and fp32 results, in a fixed order (a training step is reproducible bit for bit).
//
// The outputs are small (a ViG-S layer's widths: 16 to 2048 by 16 to 1024) and the contraction long (25 088 tokens at a batch
// of 128), so the tokens are split over workgroups: 128 x 128 tiles of dW times as many token ranges as give about two
// workgroups per CU, partial tiles in a workspace, a second kernel that adds them.  Several layers over the same tokens go out
// together, up to four: their tiles share the chip, and the start of a launch (11 us until the pipes run full), the partial
// tiles (a 128 x 128 one per workgroup, however few layers there are to work on) and the adding launch are paid once.
// T 25088, us, two launches a layer against two in all: 2048 x 384 and 384 x 1024 105 -> 86, 384 x 384, 1168 x 384 and 384 x 16 87 -> 59;
// T 1568, the latter 34 -> 20.
//
// A workgroup streams 32 tokens of both operands at a time through four LDS buffers, direct-to-LDS loads of whole
// 256-byte row pieces, three stages in flight (16 KB each: what the L2's latency asks for).  The contraction runs over
// tokens, so an operand fragment needs 8 tokens of one channel: ds_read_b64_tr_b16 hands every lane of a group of sixteen
// four tokens of its channel out of a 4 x 16 block.  The 32-byte units of a row are swapped among themselves by the row
// number (the loads fetch them that way), so that the four rows and two units that 32 lanes read lie in different banks.
// What bounds it, at one layer of 2048 x 384 over 25088 rows (63 us): 31 us the loop (1.27 PFLOP/s, what a large product of the library
// reaches), 11 until the pipes run full, 4 to 7 writing and 7 to 9 adding the partial tiles.  Fragments read a k-step ahead of their
// products gave 3 %; 128 x 192 and 256 x 192 tiles, which ask the L2 for 0.8 and 0.6 of the operands, 57 to 60 us there and no better where
// a node's layers share the launch; lines touched 4 to 20 stages ahead by a fifth wave were no faster.
#include <math.h>

#include <algorithm>

#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

constexpr int kWgTile = 128;    // channels of either operand per workgroup
constexpr int kWgStage = 32;    // tokens per stage
constexpr int kWgBuffers = 4;
constexpr int kWgRow = kWgTile * 2;              // bytes of an operand's row in LDS
constexpr int kWgHalf = kWgStage * kWgRow;       // bytes of one operand's stage
constexpr int kWgLoads = 4;                      // 1 KB loads of a wave and stage
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_t;

struct WgradLayer {
  const uint16_t *dy, *x;
  long long ldy, ldx;
  float* part;   // [splits][N][K] (or the result itself for one split)
  float* bpart;  // [splits][N] or null
  int N, K;
  int tn, first;  // tiles along N, the layer's first tile
};
struct WgradArgs {
  WgradLayer layer[kWgradLayers];
  int T, per;  // tokens, tokens per split (a multiple of the stage)
  int layers, tiles, splits;
};

// how the 32-byte units of a row of an operand's stage are swapped
__device__ __forceinline__ int unit_swap(int row) { return 2 * (row & 3); }

__global__ __launch_bounds__(256, 2) void linear_wgrad_kernel(WgradArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // workgroups go to the XCDs in turn: each XCD gets a run of consecutive (range, tile) pairs, so that its L2 serves a
  // range's rows to that range's tiles (dealt out one by one, every XCD fetched every row: 54 -> 36 us at N 1280, K 384)
  const int total = a.splits * a.tiles, run = (total + 7) >> 3;
  const int at = ((int)blockIdx.x & 7) * run + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= run || at >= total) return;
  const int split = at / a.tiles, all_tile = at - split * a.tiles;
  int which = 0;
  for (int i = 1; i < a.layers; ++i) which = all_tile >= a.layer[i].first ? i : which;
  const WgradLayer& y = a.layer[which];
  const int N = y.N, K = y.K, tile = all_tile - y.first;
  const uint16_t *const dy = y.dy, *const x = y.x;
  const long long ldy = y.ldy, ldx = y.ldx;
  const int tk = tile / y.tn;
  const int n0 = (tile - tk * y.tn) * kWgTile, k0 = tk * kWgTile;
  const int t0 = split * a.per, t1 = min(a.T, t0 + a.per);
  const int nstage = (t1 - t0 + kWgStage - 1) / kWgStage;
  const int wn = 64 * (wave & 1), wk = 64 * (wave >> 1);  // this wave's 64 x 64 of the tile
  const int flip = wave >> 1;  // block of 32 channels of dY that comes first: the one whose bias is this wave's

  // a wave's share of a stage: rows 8*wave .. +8 of both operands, four rows (1 KB) per load.  Rows and channels past the
  // end are read from the last row and from channel 0 (every load is issued: the waits below count them); such rows are
  // cleared, such channels' results are not stored.
  const int lrow = 8 * wave + (lane >> 4), piece = lane & 15;
  const int col = 16 * ((piece >> 1) ^ unit_swap(lrow)) + 8 * (piece & 1);  // channel the 16 bytes at this place hold (in rows lrow and lrow + 4)
  const int coln = n0 + col < N ? n0 + col : 0, colk = k0 + col < K ? k0 + col : 0;
  const bool far = max(ldy, ldx) > (1 << 25);  // (a stage's rows reach past 32-bit byte offsets)
  const uint32_t offn = 2u * ((uint32_t)lrow * (uint32_t)ldy + (uint32_t)coln), offk = 2u * ((uint32_t)lrow * (uint32_t)ldx + (uint32_t)colk);
  const uint32_t lds0 = lds_offset(smem);
  const auto fetch = [&](int stage) {
    const uint32_t dst = lds0 + (stage % kWgBuffers) * (2 * kWgHalf) + 8 * wave * kWgRow;
    const int t = t0 + stage * kWgStage;
    const uint16_t *pn = dy + (size_t)t * ldy, *pk = x + (size_t)t * ldx;
    if (t + kWgStage <= t1 && !far) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        load_to_lds16(pn + 4 * i * ldy, offn, dst + 4 * i * kWgRow);
        load_to_lds16(pk + 4 * i * ldx, offk, dst + 4 * i * kWgRow + kWgHalf);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const size_t row = min(lrow + 4 * i, t1 - 1 - t);
        load_to_lds16(pn + row * ldy + coln, dst + 4 * i * kWgRow);
        load_to_lds16(pk + row * ldx + colk, dst + 4 * i * kWgRow + kWgHalf);
      }
    }
  };
  // rows past the last token of the range contribute nothing: both operands' are zeroed (one of them might hold a NaN)
  const auto clear_tail = [&](int stage) {
    char* buf = smem + (stage % kWgBuffers) * (2 * kWgHalf);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = lrow + 4 * i;
      if (t0 + stage * kWgStage + row >= t1) {
        *reinterpret_cast<u32x4_t*>(buf + row * kWgRow + 16 * piece) = u32x4_t{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(buf + kWgHalf + row * kWgRow + 16 * piece) = u32x4_t{0u, 0u, 0u, 0u};
      }
    }
  };
  // byte offsets, inside an operand's stage, of this lane's part of the fragment of channel block b (32 channels), tokens
  // 8h .. +4 of a k-step: source lane = (token (l>>2)&3, channels 4*(l&3) of the group's sixteen).  (A row's swap hangs on the row's two
  // lowest bits: the same four tokens on, and in the next k-step.)
  int atn[2], atk[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int tok = 8 * h + ((lane >> 2) & 3), half = (lane >> 4) & 1;
    atn[b] = tok * kWgRow + 32 * (((wn >> 4) + 2 * (b ^ flip) + half) ^ unit_swap(tok)) + 8 * (lane & 3);
    atk[b] = kWgHalf + tok * kWgRow + 32 * (((wk >> 4) + 2 * b + half) ^ unit_swap(tok)) + 8 * (lane & 3);
  }
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{0.f};
  // The bias by sixteen 4x4x4 products against ones at a time: a row is four tokens of one channel, a lane's own, so that a channel that
  // overflowed keeps to itself (a 16x16x32 product has two channels in a row, told apart by zeros in the other operand: 0 x Inf is NaN).
  // Of the two waves that read the same channels either takes one block of 32.  A workgroup that does the bias takes longer than the others
  // and the launch waits for it; us, 32x32x16 products in one wave of the two / this: 25088 x 2048 x 384 63.4 / 58.5, 768 x 2048 106 / 100.5, 1168 x 384 43.5
  // / 40.6; lane sums by v_dot2 59.9, 101, 41.4.
  const bool with_bias = y.bpart && k0 == 0;
  f32x4acc_t accb[2] = {f32x4acc_t{0.f}, f32x4acc_t{0.f}};
  s16x4_t ones = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
  asm volatile("" : "+v"(ones));  // (in registers: made anew in every k-step otherwise)
  struct Frags {
    u32x4_t n[2], k[2];
  };
  const auto read = [&](const char* buf, int ks, Frags& f) {
    const auto frag = [&](int at) {
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(buf + at + ks * 16 * kWgRow));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(buf + at + (ks * 16 + 4) * kWgRow));
      return __builtin_bit_cast(u32x4_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
#pragma unroll
    for (int b = 0; b < 2; ++b) f.n[b] = frag(atn[b]), f.k[b] = frag(atk[b]);
  };
  const auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i][j] = mfma(f.n[i], f.k[j], acc[i][j]);
    if (with_bias) {
      const u32x4_t y = f.n[0];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        accb[q] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4_t, u32x2_t{y[2 * q], y[2 * q + 1]}), ones, accb[q], 0, 0, 0);
    }
  };
  for (int s = 0; s < kWgBuffers - 1; ++s)
    if (s < nstage) fetch(s);
  // A k-step's fragments are read while the one before is multiplied, across the stages too: behind a barrier the matrix pipe has the
  // last stage's second k-step to go on with (before the first stage: zeros).
  Frags f0, f1;
#pragma unroll
  for (int b = 0; b < 2; ++b) f1.n[b] = f1.k[b] = u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll 1
  for (int s = 0; s < nstage; ++s) {
    // this wave's share of stage s has landed: the (up to two) later stages' four loads each may still be out
    const int later = min(nstage - 1 - s, kWgBuffers - 2);
    if (later == 2) wait_vmem<2 * kWgLoads>();
    else if (later == 1) wait_vmem<kWgLoads>();
    else wait_vmem<0>();
    if (t0 + (s + 1) * kWgStage > t1) clear_tail(s);
    // (this wave's reads of stage s - 1 have returned: behind the barrier its buffer is fetched into)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const char* buf = smem + (s % kWgBuffers) * (2 * kWgHalf);
    read(buf, 0, f0);
    __builtin_amdgcn_sched_barrier(0);
    if (s + kWgBuffers - 1 < nstage) fetch(s + kWgBuffers - 1);
    multiply(f1);
    __builtin_amdgcn_sched_barrier(0);
    read(buf, 1, f1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f0);
    __builtin_amdgcn_sched_barrier(0);
  }
  multiply(f1);
  float* part = y.part + (size_t)split * N * K;
  const auto store = [&](bool whole) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int k = k0 + wk + 32 * j + r;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const int n = n0 + wn + 32 * (i ^ flip) + 8 * (c >> 2) + 4 * h + (c & 3);
          if (whole || (n < N && k < K)) part[(size_t)n * K + k] = acc[i][j][c];
        }
      }
  };
  if (n0 + kWgTile <= N && k0 + kWgTile <= K) store(true);
  else store(false);
  if (with_bias) {
    const f32x4acc_t both = accb[0] + accb[1];
    float sum = both[0];
#pragma unroll
    for (int c = 1; c < 4; ++c) sum = (lane & 3) == c ? both[c] : sum;
    sum += __shfl_xor(sum, 32);
    const int n = n0 + wn + 32 * flip + r;
    if (h == 0 && n < N) y.bpart[(size_t)split * N + n] = sum;
  }
}

// A launch for the sums that several kernels have left partial rows of.  Behind each of them a launch of its own took 4.7 us, most of it the launch: 72 of a
// training pass of twelve blocks are 24, or 48 with large partial tiles, which are added up at once (train_block.cpp).  Sums in the order they had there.
struct SumLaunch {
  vig_sum_jobs jobs;
  int first[VIG_SUM_JOBS];  // a job's first block
};

// fours: a block has as many columns of four values as an eighth of its threads and eight groups of rows, whose sums are added in LDS in order
template <int THREADS>
__device__ __forceinline__ void sum_fours(const vig_sum_job& y, int block, f32x4_t (*sums)[THREADS / 8]) {
  const int col = threadIdx.x % (THREADS / 8), grp = threadIdx.x / (THREADS / 8);
  const long long n4 = y.cols / 4, i = (long long)block * (THREADS / 8) + col;
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (i < n4) {
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(y.part) + i;
#pragma unroll 4
    for (int k = grp; k < y.rows; k += 8) s += p[(long long)k * n4];
  }
  sums[grp][col] = s;
  __syncthreads();
  if (grp != 0 || i >= n4) return;
#pragma unroll
  for (int k = 1; k < 8; ++k) s += sums[k][col];
  if ((reinterpret_cast<uintptr_t>(y.out) & 15) == 0) {
    reinterpret_cast<f32x4_t*>(y.out)[i] = s;
  } else {  // (a caller's bias gradient may start anywhere)
#pragma unroll
    for (int k = 0; k < 4; ++k) y.out[4 * i + k] = s[k];
  }
}

// 1024 threads where there are sums of few columns, which have all rows of a column under way (four slices of rows to each of 256 take 138 registers,
// and the other form from eight waves a SIMD to three: a node's sums of ViG-S at 25 088 rows 19 us, with these 13 to 14); 256 where there are none.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void sum_jobs_kernel(SumLaunch a) {
  __shared__ __align__(16) char room[THREADS * 16];
  int which = 0;
  for (int i = 1; i < a.jobs.count; ++i) which = (int)blockIdx.x >= a.first[i] ? i : which;
  const vig_sum_job& y = a.jobs.job[which];
  const int block = (int)blockIdx.x - a.first[which];
  if (THREADS == 256 || y.fours) sum_fours<THREADS>(y, block, reinterpret_cast<f32x4_t(*)[THREADS / 8]>(room));
  else if constexpr (THREADS == 1024) sum_columns(y.part, y.out, y.rows, y.cols, block, reinterpret_cast<float(*)[17]>(room));
}

long long wgrad_tiles(int N, int K) { return (long long)((N + kWgTile - 1) / kWgTile) * ((K + kWgTile - 1) / kWgTile); }

// Token ranges of some layers that go out together: the number with the least estimated time, from what was measured for 1 to 128 ranges of
// 23 layers and nodes of ViG-T, -S and -B at 100 to 50 176 rows, inputs in the L2s and not.  A workgroup alone on its CU takes 8.8 ns a row, two on
// one CU 11.6; three make a pair and one behind it, with 1.4 us to fill the pipes again, and every round behind
// the first adds 7 % to all of it: the ranges no longer walk in step through what the caches hold.  Partial tiles cost a launch, the result written, a
// pass of the adding kernel for eight ranges and, for what is written and read back between the two, 3.1 us times the 0.56th power of the millions of them
// (the more there are, the more of that hides under the loops).  Beyond eight ranges a multiple of eight keeps a range's tiles on one XCD: 3.6 %.
// 0.7 % off the best of all counts on average, where "as many as fill the chip in one round" was 6.4 % off; more than 2 % behind that rule at 12 of 736 points, by
// 0.4 us at most.  us, that rule / this one: both MLP layers of ViG-S, 784 rows (4 ranges) 21 / 14.5; 2320 x 768, 784 rows 24.6 / 15.6; 1024 x 192, 4 704 rows (19
// ranges) 19.1 / 17.4; 384 x 16, 784 rows (4) 9.3 / 7.7; 2048 x 384, 25 088 rows 58.7 / 58.4.
float wgrad_estimate(long long T, long long tiles, float melems, int s) {
  const long long per = ((T + s - 1) / s + kWgStage - 1) / kWgStage * kWgStage;
  const long long deep = (tiles * ((T + per - 1) / per) + 255) / 256;  // workgroups a CU has to do
  const long long rounds = (deep + 1) >> 1;
  float us = ((deep >> 1) * 0.0116f + (deep & 1) * 0.0088f) * per * (0.93f + 0.07f * rounds) + 1.4f * rounds;
  if (s > 1) us += 0.3f + 0.55f * melems + 0.1f * ((s + 7) / 8) + 3.1f * powf(s * melems, 0.56f);
  return s > 8 && s % 8 ? 1.036f * us : us;
}
int wgrad_splits(long long T, const LinearWgrad* layers, int count) {
  long long tiles = 0;
  float melems = 0.f;
  for (int i = 0; i < count; ++i) tiles += wgrad_tiles(layers[i].N, layers[i].K), melems += 1e-6f * layers[i].N * layers[i].K;
  const long long most = std::min<long long>(128, std::min((T + 63) / 64, 2048 / tiles));
  int best = 1;
  float least = wgrad_estimate(T, tiles, melems, 1);
  for (int s = 2; s <= most; s += s < 24 ? 1 : 4) {
    const float us = wgrad_estimate(T, tiles, melems, s);
    if (us < least) least = us, best = s;
  }
  return best;
}

}  // namespace

bool linear_wgrad_supported(long long T, int N, int K) {
  return T > 0 && T < 0x7fffffffLL - 4096 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 && N <= (1 << 20) && K <= (1 << 20);
}
// Past 256 tiles a layer's own number of ranges fits the chip better than one number for all, and from here on the loops are all that counts: both MLP
// layers of ViG-B, us, together / one behind the other: 6 272 rows 99 / 108, 12 544 174 / 181, 16 384 220 / 226, 18 000 245 / 239, 25 088 348 / 326, 50 176 722 / 656.
static bool wgrad_together(long long T, const LinearWgrad* layers, int count) {
  long long tiles = 0;
  for (int i = 0; i < count; ++i) tiles += wgrad_tiles(layers[i].N, layers[i].K);
  return count == 1 || tiles <= 256 || T <= 16384;
}
size_t linear_wgrad_workspace(long long T, const LinearWgrad* layers, int count) {
  if (!wgrad_together(T, layers, count)) {
    size_t most = 0;
    for (int i = 0; i < count; ++i) most = std::max(most, linear_wgrad_workspace(T, layers + i, 1));
    return most;
  }
  size_t floats = 0;
  for (int i = 0; i < count; ++i) floats += ((size_t)layers[i].N * layers[i].K + layers[i].N + 3) / 4 * 4;
  return wgrad_splits(T, layers, count) * floats * sizeof(float);
}

int launch_sum_jobs(const vig_sum_jobs& jobs, hipStream_t stream) {
  if (jobs.count < 1) return 0;
  if (jobs.count > VIG_SUM_JOBS) return -22;
  SumLaunch a{};
  a.jobs = jobs;
  long long blocks = 0;
  bool only_fours = true;
  for (int i = 0; i < jobs.count; ++i) only_fours = only_fours && jobs.job[i].fours;
  const int four_columns = only_fours ? 32 : 128;
  for (int i = 0; i < jobs.count; ++i) {
    const vig_sum_job& y = jobs.job[i];
    if (!y.part || !y.out || y.cols <= 0 || y.rows <= 0 || (y.fours && (y.cols % 4 || (reinterpret_cast<uintptr_t>(y.part) & 15)))) return -22;
    a.first[i] = (int)blocks;
    blocks += y.fours ? (y.cols / 4 + four_columns - 1) / four_columns : (y.cols + 15) / 16;
    if (blocks > 0x7fffffffLL / 256) return -22;
  }
  hipLaunchKernelGGL((only_fours ? sum_jobs_kernel<256> : sum_jobs_kernel<1024>), dim3((unsigned)blocks), dim3(only_fours ? 256 : 1024), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// later: the sums over token ranges are left to it, where the layers go out together
int launch_linear_wgrad(const LinearWgrad* layers, int count, long long T, void* workspace, vig_sum_jobs* later, hipStream_t stream) {
  static bool done[64] = {};
  constexpr int lds = kWgBuffers * 2 * kWgHalf;
  if (count < 1 || count > kWgradLayers) return -22;
  if (!wgrad_together(T, layers, count)) {
    int rc = 0;
    for (int i = 0; i < count && rc == 0; ++i) rc = launch_linear_wgrad(layers + i, 1, T, workspace, nullptr, stream);  // (one workspace for all)
    return rc;
  }
  if (!allow_lds(reinterpret_cast<const void*>(linear_wgrad_kernel), lds, done)) return -5;
  WgradArgs a{};
  vig_sum_jobs own{}, &sums = later ? *later : own;
  long long tiles = 0;
  for (int i = 0; i < count; ++i) tiles += wgrad_tiles(layers[i].N, layers[i].K);
  if (tiles > 0x7fffffffLL / 256) return -22;
  const int want = wgrad_splits(T, layers, count);
  a.T = (int)T, a.layers = count, a.tiles = (int)tiles;
  a.per = (int)(((T + want - 1) / want + kWgStage - 1) / kWgStage * kWgStage);
  a.splits = (int)((T + a.per - 1) / a.per);
  const bool sum = a.splits > 1;
  float* ws = (float*)workspace;
  tiles = 0;
  for (int i = 0; i < count; ++i) {
    const LinearWgrad& l = layers[i];
    WgradLayer& y = a.layer[i];
    const size_t weights = (size_t)a.splits * l.N * l.K;
    y.dy = (const uint16_t*)l.dy, y.x = (const uint16_t*)l.x, y.ldy = l.ldy, y.ldx = l.ldx, y.N = l.N, y.K = l.K;
    y.part = sum ? ws : l.dw;
    y.bpart = l.db ? (sum ? ws + weights : l.db) : nullptr;
    y.tn = (l.N + kWgTile - 1) / kWgTile, y.first = (int)tiles;
    if (sum && !(put_off(sums, y.part, l.dw, a.splits, (long long)l.N * l.K, true) && (!l.db || put_off(sums, y.bpart, l.db, a.splits, l.N, true)))) return -22;
    ws += (weights + (l.db ? (size_t)a.splits * l.N : 0) + 3) / 4 * 4;
    tiles += wgrad_tiles(l.N, l.K);
  }
  hipLaunchKernelGGL(linear_wgrad_kernel, dim3(8 * ((a.splits * a.tiles + 7) / 8)), dim3(256), lds, stream, a);
  if (hipGetLastError() != hipSuccess) return -5;
  return later ? 0 : launch_sum_jobs(own, stream);
}

}  // namespace vig
