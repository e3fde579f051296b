// gate_proj and the SwiGLU product of the block's MLP in one kernel, for contractions as short as the hidden size
// (K = 16 * KS <= 384):
//   out[t, c] = g * sigmoid(g) * u,   g = A[t, :] . W[c, :],   u = A[t, :] . W[I + c, :]      (W = [2*I, K])
// bf16 operands, fp32 accumulation, bf16 out; the product is taken on g and u rounded to bf16, the values the
// separate layer would have stored (flash-linear-attention/fla/modules/activations.py:109-113 on the two halves of
// gate_proj's output, classification/models/vig.py:492-495), so the [T, 2*I] intermediate never exists.
//
// The same kernel without the SwiGLU makes 64 channels a wave of a plain layer, and for training it keeps both.
//
// With K this short a wave's whole slice of W fits in registers: a wave keeps the 32 gate rows and the 32 matching
// up rows of one channel tile as matrix-instruction A operands for the life of the workgroup, eight waves cover 256
// channels, and the workgroup streams 32-token tiles of A through LDS, double-buffered: the next tile travels from
// memory straight into its buffer (direct-to-LDS loads, whole token rows per wave, no registers) during the matrix
// instructions of the current one, and every 16-byte LDS read, issued three k-steps ahead of its use, feeds two
// v_mfma_f32_32x32x16_bf16.  The two waves of a SIMD take turns on its matrix and vector pipes (see the loop).  Matrix
// rows are assigned channels so that a lane ends with 16 consecutive channels of one token (32 contiguous bytes).
// Workgroups of the same column group are spread over the token tiles; the column groups of one token tile run on the
// same XCD (workers are a multiple of the XCD count apart in block index), so a tile of A leaves HBM once.
#include "common.h"
#include "launch.h"

namespace vig {

namespace {

constexpr int kLinWaves = 8;

// This wave's LDS writes done, then the barrier, and nothing else: global requests and stores issued before it stay in
// flight.  (A fence would drain them: the compiler counts loads that land in LDS as LDS writes.  Whoever reads what
// such a load brings waits for it by itself.)
__device__ __forceinline__ void tile_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Matrix row i of a weight tile holds this channel of its 32: lane (r, h) of the product ends with channels 16h .. 16h+15.
__device__ __forceinline__ int channel_of_row(int i) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); }

// A wave's NT tiles of 32 rows of W (the tile's first row at `first[j]`, K = 16 * KS elements apart) into its registers as
// matrix operands: w[j][t] = elements 16t + 8h .. of lane (r, h)'s row.  Fetched straight into registers that is 32 bytes of
// 32 rows an instruction, four times each 128-byte line, and the lines of eight waves do not stay in the 32 KB L1: 14 us
// of a launch at K 384, 8 at K 192.  So the rows travel in 128-byte pieces through a ring of kRing 4 KB buffers of the wave in
// LDS (no barrier; unit u of row i lies at place u ^ (i & 7), so that the lanes served together hit different banks).
// `ring` is free for other use behind the next barrier.
constexpr int kRing = 2;
template <int KS, int NT>
__device__ __forceinline__ void load_weight_tiles(u32x4_t (&w)[NT][KS], const uint16_t* const* first, const char* ring, int lane) {
  static_assert(KS % 4 == 0, "whole pieces");
  constexpr int K = 16 * KS, KC = KS / 4, NQ = NT * KC;
  const int r = lane & 31, h = lane >> 5, row = lane >> 3, unit = (lane & 7) ^ row;
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_offset(ring));
  int off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) off[i] = channel_of_row(8 * i + row) * K + 8 * unit;
  const auto fetch = [&](int q) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds16(first[q / KC] + off[i] + 64 * (q % KC), ring0 + (q % kRing) * 4096 + 1024 * i);
  };
#pragma unroll
  for (int q = 0; q < kRing; ++q) fetch(q);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q + 1 < NQ) wait_vmem<4 * (kRing - 1)>();
    else wait_vmem<0>();
    const char* buf = ring + (q % kRing) * 4096 + r * 128;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      w[q / KC][4 * (q % KC) + t] = *reinterpret_cast<const u32x4_t*>(buf + 16 * ((2 * t + h) ^ (r & 7)));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the buffer is filled again
    if (q + kRing < NQ) fetch(q + kRing);
  }
}

// The same for tiles of 32 columns of a W [K, ldw] (the products of a backward, d_x = d_y . W): pieces of 64 rows of 64 bytes, and
// ds_read_b64_tr_b16 hands every lane of a group of sixteen four contraction elements of its channel out of a 4 x 16 block.
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_t;
template <int KS, int NT>
__device__ __forceinline__ void load_weight_columns(u32x4_t (&w)[NT][KS], const uint16_t* const* first, int ldw, char* ring, int lane) {
  static_assert(KS % 4 == 0, "whole pieces");
  constexpr int KC = KS / 4, NQ = NT * KC;
  const int h = lane >> 5, half = (lane >> 4) & 1, block = lane & 3;  // (source lane: row (lane >> 2) & 3 of the block, four columns)
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_offset(ring));
  const int at = ((8 * h + ((lane >> 2) & 3)) * 32 + channel_of_row(16 * half + 4 * block)) * 2;
  const auto fetch = [&](int q) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load_to_lds16(first[q / KC] + (size_t)(64 * (q % KC) + 16 * i + (lane >> 2)) * ldw + 8 * (lane & 3),
                    ring0 + (q % kRing) * 4096 + 1024 * i);
  };
#pragma unroll
  for (int q = 0; q < kRing; ++q) fetch(q);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q + 1 < NQ) wait_vmem<4 * (kRing - 1)>();
    else wait_vmem<0>();
    char* buf = ring + (q % kRing) * 4096 + at;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(buf + 1024 * t));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(buf + 1024 * t + 256));
      const u32x2_t l = __builtin_bit_cast(u32x2_t, lo), u = __builtin_bit_cast(u32x2_t, hi);
      w[q / KC][4 * (q % KC) + t] = u32x4_t{l[0], l[1], u[0], u[1]};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (q + kRing < NQ) fetch(q + kRing);
  }
}

// What a wave makes of its two 32-row tiles of W (rows from c0 and from c1):
//   kSwiglu      c0 = gate, c1 = up channels of one tile: the SwiGLU product
//   kSwigluKept  the same, and the gate and up values themselves ([T, 2*I], what a backward reads)
//   kLinear      64 channels of a plain layer, + bias
//   kColumns     the same for W [K, N]
//   kSwigluBwd   one tile of columns of the down projection's W [K, N]: the gradient of the SwiGLU product (rounded to bf16, as
//                the separate layer would store it) goes through the product's backward with the kept gate and up values:
//                out = their gradients [T, 2*N]
enum LinForm { kSwiglu, kSwigluKept, kLinear, kColumns, kSwigluBwd };

// Bytes of LDS a wave turns its results in, none where they are stored as they lie.  Turned, an instruction writes whole 64-byte
// rows: K 192 with the values kept, 50176 x 512, 42 -> 36 us; the SwiGLU backward, 50176 tokens, K 384 113 -> 100, K 192 41 -> 38.
// The plain layers and the SwiGLU gain nothing at K 192, and at K 384 the addresses spill (50176 x 1280 53 -> 67 us).
constexpr int turn_bytes(int KS, LinForm f) { return f == kSwigluBwd ? 4096 : f == kSwigluKept && KS == 12 ? 6144 : 0; }

template <int KS, int NW, LinForm FORM>
__global__ __launch_bounds__(64 * NW, 2) void linear_regs_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                                 const uint16_t* __restrict__ bias, uint16_t* __restrict__ out,
                                                                 uint16_t* __restrict__ kept, int T, int N, int nworkers) {
  constexpr int K = 16 * KS;
  constexpr int kCols = K / 8;                 // 16-byte chunks per token row
  constexpr int kRow = K + 8;                  // LDS row stride in elements (conflict-free 16-byte reads)
  constexpr int kPer = 32 / NW;                // token rows per wave
  constexpr bool kPlain = FORM == kLinear || FORM == kColumns;
  constexpr int kStep = kPlain ? 64 : 32;                                       // channels per wave
  constexpr int kStores = FORM == kSwiglu ? 2 : FORM == kSwigluKept ? 6 : 4;   // of a whole tile's epilogue
  constexpr int kTiles = FORM == kSwigluBwd ? 1 : 2;
  static_assert(kCols <= 64 && 32 % NW == 0, "a wave loads whole token rows");
  extern __shared__ __align__(16) char smem[];
  // [biases][2][32][kRow][waves' results]; the weights' ring lies where the second of the two tiles will
  constexpr size_t kBias = FORM == kLinear ? 64 * NW * sizeof(float) : 0, kTile = 32 * kRow * sizeof(uint16_t);
  constexpr int kTurn = turn_bytes(KS, FORM);
  float* const bias_lds = reinterpret_cast<float*>(smem);
  uint16_t* buf = reinterpret_cast<uint16_t*>(smem + kBias);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int cg = blockIdx.x / nworkers, worker = blockIdx.x - cg * nworkers;
  const int ct = cg * NW + wave;  // this wave's channel tile
  const bool have = kStep * ct < N;
  if constexpr (FORM == kLinear) {
    for (int i = tid; i < 64 * NW; i += 64 * NW) bias_lds[i] = bias && cg * 64 * NW + i < N ? bf16_to_f32(bias[cg * 64 * NW + i]) : 0.f;
  }
  const int ntiles_t = (T + 31) / 32;
  // A tile travels from memory straight into its LDS buffer (no registers): lane i of a wave lands 16 i bytes behind
  // the wave's base, so a wave loads whole token rows (the first K/8 lanes, one 16-byte chunk each) to the rows' padded
  // places.  Token rows past the end are not requested: their rows of the buffer keep old data, and their products
  // are never stored.
  const uint32_t lds0 = lds_offset(buf);
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  auto fetch = [&](int tile, int which) {
    if (tile >= ntiles_t) return;
    const uint32_t base = lds0 + which * (32 * kRow * 2);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int row = i * NW + uwave;
      if (lane < kCols && tile * 32 + row < T)
        load_to_lds16(A + (size_t)tile * (32 * K) + (size_t)row * K + lane * 8, base + row * (kRow * 2));
    }
  };
  u32x4_t wt[kTiles][KS];
  f32x16_t g, u;
#pragma unroll
  for (int j = 0; j < 16; ++j) g[j] = 0.f, u[j] = 0.f;
  // the kept gate and up values behind a tile's gradients, fetched ahead of its products
  u32x4_t z[4];
  auto fetch_kept = [&](int tile) {
    const uint16_t* p = kept + (size_t)min(tile * 32 + r, T - 1) * 2 * N + (have ? 32 * ct : 0) + 16 * h;
    z[0] = *reinterpret_cast<const u32x4_t*>(p), z[1] = *reinterpret_cast<const u32x4_t*>(p + 8);
    z[2] = *reinterpret_cast<const u32x4_t*>(p + N), z[3] = *reinterpret_cast<const u32x4_t*>(p + N + 8);
  };
  auto store32 = [](uint16_t* dst, const u32x4_t& lo, const u32x4_t& hi) {
    *reinterpret_cast<u32x4_t*>(dst) = lo;
    *reinterpret_cast<u32x4_t*>(dst + 8) = hi;
  };
  // A lane ends with 16 channels of one token: stored as they lie, an instruction writes 16-byte pieces all over 32 rows.  Where
  // registers allow, the results are turned in a wave's own piece of LDS first (units swapped by the row, against bank
  // conflicts), so that four lanes write 64 consecutive bytes.
  char* const turn = smem + kBias + 2 * kTile + uwave * kTurn;
  // gate and up values (or their gradients) of a tile to [T, 2*N]
  auto store_pair = [&](int etile, uint16_t* base, const u32x4_t& glo, const u32x4_t& ghi, const u32x4_t& ulo, const u32x4_t& uhi) {
    if constexpr (kTurn > 0) {
      char* const mine = turn + r * 128;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((2 * h) ^ ((r >> 1) & 7))) = glo;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((2 * h + 1) ^ ((r >> 1) & 7))) = ghi;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((4 + 2 * h) ^ ((r >> 1) & 7))) = ulo;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((5 + 2 * h) ^ ((r >> 1) & 7))) = uhi;
      const int unit = lane & 7;
      uint16_t* const dst = base + (size_t)(etile * 32) * 2 * N + 32 * ct + 8 * (unit & 3) + (unit & 4 ? N : 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + (lane >> 3);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(turn + row * 128 + 16 * (unit ^ ((row >> 1) & 7)));
        if (have && etile * 32 + row < T) *reinterpret_cast<u32x4_t*>(dst + (size_t)row * 2 * N) = v;
      }
    } else if (have && etile * 32 + r < T) {
      uint16_t* dst = base + (size_t)(etile * 32 + r) * 2 * N + 32 * ct + 16 * h;
      store32(dst, glo, ghi);
      store32(dst + N, ulo, uhi);
    }
  };
  // one finished tile, 16 consecutive channels of one token per lane (SwiGLU on the rounded gate and up values)
  auto epilogue = [&](int etile) {
    const int token = etile * 32 + r;
    u32x4_t lo, hi, glo, ghi, ulo, uhi;
    if constexpr (FORM == kSwigluBwd) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t zg = z[j >> 2][j & 3], zu = z[2 + (j >> 2)][j & 3];
        float dg[2], du[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float d = bf16_to_f32(f32_to_bf16(g[2 * j + e]));
          const float gv = e ? bf16hi_to_f32(zg) : bf16lo_to_f32(zg), uv = e ? bf16hi_to_f32(zu) : bf16lo_to_f32(zu);
          const float sg = sigmoidf_(gv);
          du[e] = d * gv * sg;
          dg[e] = d * uv * sg * (1.f + gv * (1.f - sg));
        }
        (j < 4 ? glo : ghi)[j & 3] = pack_bf16x2(dg[0], dg[1]);
        (j < 4 ? ulo : uhi)[j & 3] = pack_bf16x2(du[0], du[1]);
      }
    } else if constexpr (FORM != kSwiglu) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        glo[j] = pack_bf16x2(g[2 * j], g[2 * j + 1]), ghi[j] = pack_bf16x2(g[8 + 2 * j], g[8 + 2 * j + 1]);
        ulo[j] = pack_bf16x2(u[2 * j], u[2 * j + 1]), uhi[j] = pack_bf16x2(u[8 + 2 * j], u[8 + 2 * j + 1]);
      }
    }
    if constexpr (FORM == kSwiglu || FORM == kSwigluKept) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float gs, us;
          if constexpr (FORM == kSwigluKept) {
            const uint32_t gp = j < 4 ? glo[j] : ghi[j - 4], up = j < 4 ? ulo[j] : uhi[j - 4];
            gs = e ? bf16hi_to_f32(gp) : bf16lo_to_f32(gp), us = e ? bf16hi_to_f32(up) : bf16lo_to_f32(up);
          } else {
            gs = bf16_to_f32(f32_to_bf16(g[2 * j + e])), us = bf16_to_f32(f32_to_bf16(u[2 * j + e]));
          }
          y[e] = gs * us * sigmoidf_(gs);
        }
        const uint32_t pk = pack_bf16x2(y[0], y[1]);
        if (j < 4) lo[j] = pk;
        else hi[j - 4] = pk;
      }
    }
    if constexpr (FORM == kSwigluBwd) store_pair(etile, out, glo, ghi, ulo, uhi);
    if constexpr (FORM == kSwigluKept) store_pair(etile, kept, glo, ghi, ulo, uhi);
    if constexpr (FORM == kSwigluKept && kTurn > 0) {
      char* const mine = turn + 4096 + r * 64;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((2 * h) ^ ((r >> 2) & 3))) = lo;
      *reinterpret_cast<u32x4_t*>(mine + 16 * ((2 * h + 1) ^ ((r >> 2) & 3))) = hi;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * i + (lane >> 2);
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(turn + 4096 + row * 64 + 16 * ((lane & 3) ^ ((row >> 2) & 3)));
        if (have && etile * 32 + row < T) *reinterpret_cast<u32x4_t*>(out + (size_t)(etile * 32 + row) * N + 32 * ct + 8 * (lane & 3)) = v;
      }
    } else if (FORM != kSwigluBwd && have && token < T) {
      if constexpr (kPlain) {
        uint16_t* dst = out + (size_t)token * N + 64 * ct + 16 * h;
        store32(dst, glo, ghi);
        store32(dst + 32, ulo, uhi);
      } else {
        store32(out + (size_t)token * N + 32 * ct + 16 * h, lo, hi);
      }
    }
  };
  // this tile's products: operand reads run kAhead k-steps ahead of the matrix instructions that use them
  auto products = [&](const uint16_t* mine) {
    if constexpr (FORM == kLinear) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t bg = *reinterpret_cast<const f32x4_t*>(bias_lds + 64 * wave + 16 * h + 4 * j),
                      bu = *reinterpret_cast<const f32x4_t*>(bias_lds + 64 * wave + 32 + 16 * h + 4 * j);
#pragma unroll
        for (int e = 0; e < 4; ++e) g[4 * j + e] = bg[e], u[4 * j + e] = bu[e];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) g[j] = 0.f, u[j] = 0.f;
    }
    const uint16_t* xrow = mine + r * kRow + 8 * h;
    constexpr int kAhead = FORM == kSwiglu || FORM == kSwigluBwd || KS < 24 ? 3 : 2;  // (as the registers allow)
    u32x4_t x[kAhead];
#pragma unroll
    for (int t = 0; t < kAhead; ++t) x[t] = *reinterpret_cast<const u32x4_t*>(xrow + 16 * t);
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      const u32x4_t xt = x[t % kAhead];
      g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wt[0][t]), __builtin_bit_cast(bf16x8_t, xt),
                                                  g, 0, 0, 0);
      if constexpr (kTiles == 2)
        u = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wt[kTiles - 1][t]), __builtin_bit_cast(bf16x8_t, xt),
                                                    u, 0, 0, 0);
      if (t + kAhead < KS) x[t % kAhead] = *reinterpret_cast<const u32x4_t*>(xrow + 16 * (t + kAhead));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  fetch(worker, 0);
  {
    char* const ring = smem + kBias + kTile + uwave * (kRing * 4096);
    const int c0 = have ? kStep * (cg * NW + uwave) : 0;
    if constexpr (FORM == kColumns || FORM == kSwigluBwd) {
      const uint16_t* const first[2] = {W + c0, W + c0 + 32};
      load_weight_columns<KS, kTiles>(wt, first, N, ring, lane);
    } else {
      const uint16_t* const w0 = W + (size_t)c0 * K;
      const uint16_t* const first[2] = {w0, w0 + (size_t)(FORM == kLinear ? 32 : N) * K};
      load_weight_tiles<KS, 2>(wt, first, ring, lane);
    }
  }
  int cur = 0;
  bool stored = false;  // an epilogue's stores were issued after the current tile's loads (a full tile's: only the last
                        // tile of all, behind which nothing is waited for, may be short)
  for (int tile = worker; tile < ntiles_t; tile += nworkers, cur ^= 1) {
    const uint16_t* mine = buf + cur * (32 * kRow);
    // this thread's chunks of the tile have landed; the stores of an epilogue behind them may still be on their way
    // (waiting for those too, as a full barrier does, cost a tile the latency of a store)
    if (stored) wait_vmem<kStores>();
    else wait_vmem<0>();
    tile_barrier();  // the tile is complete; the other buffer was last read before the previous barrier
    if constexpr (FORM == kSwigluBwd) fetch_kept(tile);
    fetch(tile + nworkers, cur ^ 1);
    // The two waves of a SIMD (w and w + 4 of eight) take turns on its two pipes: the lower wave runs this tile's matrix
    // instructions first and its epilogue after; the upper wave first runs the epilogue of its PREVIOUS tile
    // (its accumulators waited in registers) and then this tile's matrix instructions.  So one wave's vector work
    // runs under the other's matrix work in both halves of a tile's time, with one barrier per tile as before.  (Four
    // waves: the second wave of a SIMD is another workgroup's.)
    if (NW == 4 || wave < NW / 2) {
      products(mine);
      epilogue(tile);  // (straight-line after the matrix instructions: no run-time branch in between)
      stored = have;
    } else {
      stored = have && tile > worker;
      if (tile > worker) epilogue(tile - nworkers);
      products(mine);
    }
  }
  if (NW > 4 && wave >= NW / 2 && worker < ntiles_t)  // the upper waves' last tile
    epilogue(worker + ((ntiles_t - 1 - worker) / nworkers) * nworkers);
}

template <int KS, int NW, LinForm FORM>
int launch_linear_regs_t(const void* A, const void* W, const void* bias, void* out, void* kept, long long T, int N, int num_cu,
                         hipStream_t stream) {
  constexpr int K = 16 * KS, kStep = FORM == kLinear || FORM == kColumns ? 64 : 32;
  constexpr size_t tile = 32 * (K + 8) * sizeof(uint16_t), ring = (size_t)NW * kRing * 4096;
  constexpr size_t two = tile + NW * turn_bytes(KS, FORM);
  constexpr size_t lds = (FORM == kLinear ? 64 * NW * sizeof(float) : 0) + tile + (two > ring ? two : ring);
  static bool done[64] = {};
  if (!allow_lds((const void*)linear_regs_kernel<KS, NW, FORM>, lds, done)) return -5;
  const int ncg = (N / kStep + NW - 1) / NW;
  const long long ntiles_t = (T + 31) / 32;
  // eight waves a CU; workers a multiple of 8 so that the column groups of a token tile share an XCD
  int nworkers = num_cu * 8 / NW / ncg / 8 * 8;
  if (nworkers < 8) nworkers = 8;
  if (nworkers > ntiles_t) nworkers = (int)ntiles_t;
  hipLaunchKernelGGL((linear_regs_kernel<KS, NW, FORM>), dim3(ncg * nworkers), dim3(64 * NW), lds, stream, (const uint16_t*)A,
                     (const uint16_t*)W, (const uint16_t*)bias, (uint16_t*)out, (uint16_t*)kept, (int)T, N, nworkers);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

// compute units of the current device, 0 on an error
int cu_count() {
  constexpr int kMaxDevices = 64;
  static int num_cu_dev[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  if (num_cu_dev[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    num_cu_dev[dev] = n > 0 ? n : 256;
  }
  return num_cu_dev[dev];
}

// ---------------------------------------------------------------------------
// The mixer's epilogue and o_proj in one kernel:
//   y[t, h, :] = rms(o[b, h, l, :]) w_g sigmoid(g) + rms(loc[t, h, :]) w_l (1 - sigmoid(g))   (optionally y <- y sigmoid(y)),
//   out[t, :]  = y[t, :] . W[c, :]                                   (W = o_proj.weight [C, H*Dv], K = H*Dv = 16 * KS)
// with t = b*L + l, the head norms over the Dv = 64 channels of a (token, head), g = g_lin rows of pitch ldg
// (classification/models/vig.py:444-463).  y is rounded to bf16 as the separate blend kernel would store it and never
// leaves the chip: the workgroup computes a 32-token tile of it straight into the LDS buffer the matrix instructions
// read (double-buffered).  The o / loc / g octets of the next tile travel from memory straight into thread-private
// LDS slots (no registers: lane i of a wave lands at the wave's slot base + 16 i) while the matrix instructions of the
// current tile run.  NW waves hold TPW 32-channel tiles of W each as matrix-instruction operands for the life of the
// workgroup, so one workgroup makes whole output rows (C = 32 * TPW * NW) and every tile of y is computed once.
// ---------------------------------------------------------------------------
// value of the lane a DPP control names (inside a row of 16 lanes)
template <int CTRL>
__device__ __forceinline__ float lane_permuted(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// kept (KEPT): y as well, which a backward reads.
template <int KS, int NW, int TPW, bool KEPT>
__global__ __launch_bounds__(64 * NW) void blend_linear_kernel(const uint16_t* __restrict__ o,
                                                              const uint16_t* __restrict__ loc,
                                                              const uint16_t* __restrict__ glin,
                                                              const float* __restrict__ w_g,
                                                              const float* __restrict__ w_l,
                                                              const uint16_t* __restrict__ W,
                                                              uint16_t* __restrict__ out, uint16_t* __restrict__ kept,
                                                              int T, int L, int H, long long ldg, float eps, int silu_out) {
  constexpr int K = 16 * KS;
  constexpr int C = 32 * TPW * NW;             // TPW 32-channel tiles of W per wave
  constexpr int kThreads = 64 * NW;
  constexpr int kCols = K / 8;                 // channel octets per token row
  constexpr int kRow = K + 8;                  // LDS row stride in elements (conflict-free 16-byte reads)
  constexpr int kChunks = 32 * kCols;          // channel octets of a 32-token tile
  constexpr int kPer = kChunks / kThreads;     // octets per thread
  static_assert(kChunks % kThreads == 0, "whole octets per thread");
  static_assert(kThreads % kCols == 0, "a thread's octets share their column");
  extern __shared__ __align__(16) char smem[];
  uint16_t* buf = reinterpret_cast<uint16_t*>(smem);  // [2][32][kRow]
  float* wnorm = reinterpret_cast<float*>(smem + (size_t)2 * 32 * kRow * sizeof(uint16_t));  // w_g | w_l, 64 floats each
  // thread-private slots for the fetched octets of the tile that comes next: [octet i][o, loc, g][thread]
  u32x4_t* park = reinterpret_cast<u32x4_t*>(smem + (size_t)2 * 32 * kRow * sizeof(uint16_t) + 128 * sizeof(float));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, h = lane >> 5;
  u32x4_t wt[TPW][KS];  // channel tiles TPW * wave ..
  {
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    const uint16_t* first[TPW];
#pragma unroll
    for (int j = 0; j < TPW; ++j) first[j] = W + (size_t)(32 * (TPW * uwave + j)) * K;
    load_weight_tiles<KS, TPW>(wt, first, smem + uwave * (kRing * 4096), lane);
    __syncthreads();  // the rings' place becomes the buffers'
  }
  if (tid < 128) wnorm[tid] = tid < 64 ? w_g[tid] : w_l[tid - 64];
  const int ntiles_t = (T + 31) / 32;
  const float* wg8 = wnorm + ((tid % kCols) & 7) * 8;  // (kThreads % kCols == 0: a thread's octets share their column)
  const float* wl8 = wg8 + 64;
  // requests this thread's octets of a tile into its slots; tokens past the end are not requested (their rows of y
  // hold whatever the slots held: their products are never stored)
  const int col = tid % kCols, row0 = tid / kCols;  // this thread's octets: column col of rows row0 + kRowStep * i
  constexpr int kRowStep = kThreads / kCols;
  const size_t o_col = ((size_t)(col >> 3) * L) * 64 + (col & 7) * 8;  // head col / 8, channels 8 (col % 8) ..
  const size_t o_batch = (size_t)H * L * 64;
  const uint32_t park0 = __builtin_amdgcn_readfirstlane(lds_offset(park) + wave * (64 * 16));
  auto fetch = [&](int tile) {
#pragma unroll 1
    for (int i = 0; i < kPer; ++i) {  // (one octet's addresses at a time: the weight tiles leave few registers)
      const int t = tile * 32 + row0 + kRowStep * i;
      if (tile < ntiles_t && t < T) {
        const unsigned b = (unsigned)t / (unsigned)L, l = (unsigned)t - b * (unsigned)L;
        const uint32_t slot = park0 + (i * 3) * (kThreads * 16);  // (wave-uniform; lanes 16 B apart)
        load_to_lds16(o + b * o_batch + (size_t)l * 64 + o_col, slot);
        load_to_lds16(loc + (size_t)t * K + col * 8, slot + kThreads * 16);
        load_to_lds16(glin + (size_t)t * ldg + col * 8, slot + 2 * kThreads * 16);
      }
    }
  };
  const int nworkers = gridDim.x;
  // the blend of this thread's octets of a tile (they wait in its slots), straight into the tile's operand buffer
  // (stored: the stores of a tile's result were issued behind the octets' loads and may still be on their way; waited for,
  // their latency was part of every tile)
  auto blend = [&](uint16_t* mine, bool stored, int tile) {
    if (stored) wait_vmem<2 * TPW>();
    else wait_vmem<0>();
#pragma unroll 1
    for (int i = 0; i < kPer; ++i) {
      const u32x4_t po = park[(i * 3 + 0) * kThreads + tid], pl = park[(i * 3 + 1) * kThreads + tid],
                    pg = park[(i * 3 + 2) * kThreads + tid];
      float fo[8], fl[8], fg[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        fo[2 * j] = bf16_to_f32((uint16_t)(po[j] & 0xffffu)), fo[2 * j + 1] = bf16_to_f32((uint16_t)(po[j] >> 16));
        fl[2 * j] = bf16_to_f32((uint16_t)(pl[j] & 0xffffu)), fl[2 * j + 1] = bf16_to_f32((uint16_t)(pl[j] >> 16));
        fg[2 * j] = bf16_to_f32((uint16_t)(pg[j] & 0xffffu)), fg[2 * j + 1] = bf16_to_f32((uint16_t)(pg[j] >> 16));
      }
      float so = 0.f, sl = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) so += fo[j] * fo[j], sl += fl[j] * fl[j];
      // the eight lanes of a (token, head): lane ^ 1, lane ^ 2 inside the quad, then the other quad of the eight
      so += lane_permuted<0xB1>(so), sl += lane_permuted<0xB1>(sl);    // quad_perm:[1,0,3,2]
      so += lane_permuted<0x4E>(so), sl += lane_permuted<0x4E>(sl);    // quad_perm:[2,3,0,1]
      so += lane_permuted<0x141>(so), sl += lane_permuted<0x141>(sl);  // row_half_mirror
      const float ro = rsqrtf(so * (1.0f / 64.0f) + eps);
      const float rl = rsqrtf(sl * (1.0f / 64.0f) + eps);
      float e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float sg = sigmoidf_(fg[j]);
        e[j] = fo[j] * ro * wg8[j] * sg + fl[j] * rl * wl8[j] * (1.f - sg);
      }
      if (silu_out) {
        asm volatile("");  // (a real branch: as a select, the second sigmoid is computed for every caller)
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = e[j] * sigmoidf_(e[j]);
      }
      u32x4_t y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = pack_bf16x2(e[2 * j], e[2 * j + 1]);
      *reinterpret_cast<u32x4_t*>(mine + (row0 + kRowStep * i) * kRow + col * 8) = y;
      if constexpr (KEPT) {  // (older than the loads of the tile after the next: the waits do not count these)
        const int t = tile * 32 + row0 + kRowStep * i;
        if (t < T) *reinterpret_cast<u32x4_t*>(kept + (size_t)t * K + col * 8) = y;
      }
    }
  };
  // this wave's products of a staged tile, and its rows of the result
  auto products = [&](const uint16_t* mine, int tile) {
    f32x16_t acc[TPW];
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
    const uint16_t* xrow = mine + r * kRow + 8 * h;
    constexpr int kAhead = TPW == 2 ? 3 : 1;  // operand reads this many k-steps ahead of the matrix instructions that
                                              // use them, where the registers allow
    u32x4_t x[kAhead];
#pragma unroll
    for (int t = 0; t < kAhead; ++t) x[t] = *reinterpret_cast<const u32x4_t*>(xrow + 16 * t);
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      const u32x4_t xt = x[t % kAhead];
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wt[j][t]),
                                                         __builtin_bit_cast(bf16x8_t, xt), acc[j], 0, 0, 0);
      if (t + kAhead < KS) x[t % kAhead] = *reinterpret_cast<const u32x4_t*>(xrow + 16 * (t + kAhead));
      if (TPW == 2) __builtin_amdgcn_sched_barrier(0);
    }
    // (no run-time branch between the matrix instructions and the first read of their results)
    const int token = tile * 32 + r;
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      u32x4_t lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = pack_bf16x2(acc[j][2 * e], acc[j][2 * e + 1]);
        hi[e] = pack_bf16x2(acc[j][8 + 2 * e], acc[j][8 + 2 * e + 1]);
      }
      if (token < T) {
        uint16_t* dst = out + (size_t)token * C + 32 * (TPW * wave + j) + 16 * h;
        *reinterpret_cast<u32x4_t*>(dst) = lo;
        *reinterpret_cast<u32x4_t*>(dst + 8) = hi;
      }
    }
  };
  // The waves take turns on the two pipes of their SIMD: waves 4 .. 7 (one per SIMD) first blend their octets of the
  // NEXT tile into the other buffer and then run this tile's matrix instructions; the other waves multiply first and
  // blend after (measured: 55.7 -> 52.7 us per layer at B256; the other split of the waves gained half of that).  One barrier per tile: behind it every wave has finished with tile i - 1's buffer
  // (being refilled now) and tile i's is complete.
  __syncthreads();  // the norm weights are in place
  fetch(blockIdx.x);
  blend(buf, false, blockIdx.x);
  fetch(blockIdx.x + nworkers);
  tile_barrier();
  int cur = 0;
  for (int tile = blockIdx.x; tile < ntiles_t; tile += nworkers, cur ^= 1) {
    const uint16_t* mine = buf + cur * (32 * kRow);
    uint16_t* next = buf + (cur ^ 1) * (32 * kRow);
    const bool more = tile + nworkers < ntiles_t;
    if ((wave >> 2) != 1) {
      products(mine, tile);
      if (more) {
        blend(next, true, tile + nworkers);
        fetch(tile + 2 * nworkers);
      }
    } else {
      if (more) {
        blend(next, tile != (int)blockIdx.x, tile + nworkers);
        fetch(tile + 2 * nworkers);
      }
      products(mine, tile);
    }
    tile_barrier();  // (the requests for the tile after the next and this tile's stores stay in flight)
  }
}

template <int KS, int NW, int TPW, bool KEPT>
int launch_blend_linear_t(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l,
                          const void* W, void* out, void* kept, long long T, int L, int H, long long ldg, float eps, int silu_out,
                          int num_cu, hipStream_t stream) {
  constexpr int K = 16 * KS;
  constexpr size_t lds = (size_t)2 * 32 * (K + 8) * sizeof(uint16_t) + 128 * sizeof(float) + (size_t)(32 * K / 8) * 3 * sizeof(u32x4_t);
  static_assert(lds >= (size_t)NW * kRing * 4096, "the weights' rings fit");
  const long long ntiles_t = (T + 31) / 32;
  // K 192 leaves room for two workgroups to a CU, which blend and multiply at each other's loads (us, one / two: 32768 tokens 17.8 / 16.4,
  // 12544 9.7 / 8.9, 25088 16.5 / 15.1, with y kept 17.1 / 15.8, 50176 24.9 / 21.2); at K 384 LDS holds one.
  const int most = KS == 12 ? 2 * num_cu : num_cu, grid = ntiles_t < most ? (int)ntiles_t : most;
  static bool done[64] = {};
  if (!allow_lds((const void*)blend_linear_kernel<KS, NW, TPW, KEPT>, lds, done)) return -5;
  hipLaunchKernelGGL((blend_linear_kernel<KS, NW, TPW, KEPT>), dim3(grid), dim3(64 * NW), lds, stream, (const uint16_t*)o,
                     (const uint16_t*)loc, (const uint16_t*)glin, w_g, w_l, (const uint16_t*)W, (uint16_t*)out, (uint16_t*)kept, (int)T, L,
                     H, ldg, eps, silu_out);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace

// o_proj of a square block (d_model = H * Dv) with 64-channel heads, at the widths the weights fit the registers
bool blend_linear_supported(int H, int Dv, int C) { return Dv == 64 && C == H * Dv && (C == 384 || C == 192); }

int launch_blend_linear(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l,
                        const void* W, void* out, void* kept, int B, int H, int L, int Dv, int C, long long ldg, float eps,
                        int silu_out, hipStream_t stream) {
  if (!blend_linear_supported(H, Dv, C) || B <= 0 || L <= 0 || (long long)B * L > 0x7fffffffLL - 64 || ldg % 8 != 0 ||
      ldg < C)
    return -95;
  const long long T = (long long)B * L;
  // (there a row's inputs are read by several workgroups: a result over an input, which whole rows a workgroup allow, stays with those)
  const auto over = [&](const void* p, const void* q, long long bytes) {
    const uintptr_t a = (uintptr_t)p, b = (uintptr_t)q;
    return p && a < b + (uintptr_t)bytes && b < a + (uintptr_t)(2 * T * C);
  };
  const auto apart = [&](const void* p) { return !over(p, o, 2 * T * C) && !over(p, loc, 2 * T * C) && !over(p, glin, 2 * ((T - 1) * ldg + C)); };
  if (few_blend_linear(T, C) && apart(out) && apart(kept)) return launch_few_blend_linear(o, loc, glin, w_g, w_l, W, out, kept, T, L, C, ldg, eps, silu_out, stream);
  const int num_cu = cu_count();
  if (!num_cu) return -5;
  // twelve waves with one weight tile each (three per SIMD at 168 registers) at the wider size, six at the narrower
  if (kept)
    return C == 384 ? launch_blend_linear_t<24, 12, 1, true>(o, loc, glin, w_g, w_l, W, out, kept, T, L, H, ldg, eps, silu_out, num_cu, stream)
                    : launch_blend_linear_t<12, 6, 1, true>(o, loc, glin, w_g, w_l, W, out, kept, T, L, H, ldg, eps, silu_out, num_cu, stream);
  return C == 384 ? launch_blend_linear_t<24, 12, 1, false>(o, loc, glin, w_g, w_l, W, out, kept, T, L, H, ldg, eps, silu_out, num_cu, stream)
                  : launch_blend_linear_t<12, 6, 1, false>(o, loc, glin, w_g, w_l, W, out, kept, T, L, H, ldg, eps, silu_out, num_cu, stream);
}

bool linear_swiglu_supported(int K, int I) { return (K == 384 || K == 192) && I % 32 == 0 && I >= 32; }

// Waves a workgroup, measured (four / eight, us): the turns of eight waves hide the long SwiGLU epilogue of K 384 with many tokens
// (25088 tokens 41.6 / 38.9, 50176 72 / 67); with few tokens, or with K 192, two independent workgroups of four
// fill the chip better (784 tokens 5.7 / 7.5, K 192: 50176 28.6 / 30.3).  Where the values are kept, eight waves spill
// (25088 tokens 50 / 65; a layer and a SwiGLU pass behind it: 84).
int launch_linear_swiglu(const void* A, const void* W, void* out, void* kept, long long T, int K, int I, hipStream_t stream) {
  if (!kept && few_swiglu(T, K, I)) return launch_few_swiglu(A, W, out, T, K, I, stream);
  if (!linear_swiglu_supported(K, I) || T <= 0 || T > 0x7fffffffLL - 64) return -95;
  const int num_cu = cu_count();
  if (!num_cu) return -5;
  if (kept)
    return K == 384 ? launch_linear_regs_t<24, 4, kSwigluKept>(A, W, nullptr, out, kept, T, I, num_cu, stream)
                    : launch_linear_regs_t<12, 4, kSwigluKept>(A, W, nullptr, out, kept, T, I, num_cu, stream);
  if (K == 192) return launch_linear_regs_t<12, 4, kSwiglu>(A, W, nullptr, out, nullptr, T, I, num_cu, stream);
  return T <= 1024 ? launch_linear_regs_t<24, 4, kSwiglu>(A, W, nullptr, out, nullptr, T, I, num_cu, stream)
                   : launch_linear_regs_t<24, 8, kSwiglu>(A, W, nullptr, out, nullptr, T, I, num_cu, stream);
}

bool linear_regs_supported(int K, int N) { return (K == 384 || K == 192) && N % 64 == 0 && N >= 64; }

// Against the library's products (us, library / this): K 384: 16384 rows and up; 25088 rows N 1280 33 / 31, N 2048 61 / 45, N 384
// 26 / 18, N 1024 42 / 26; 50176 rows 66 / 53, 130 / 77, 42 / 25, 58 / 42.  K 192: 32768 rows N 640 26 / 18, 50176 32 / 23,
// 100352 58 / 40.  Fewer rows: regs_rows (gemm.hip).  Bound by its stores.
int launch_linear_regs(const void* x, const void* w, const void* bias, void* y, long long T, int N, int K, hipStream_t stream) {
  if (!linear_regs_supported(K, N) || T <= 0 || T > 0x7fffffffLL - 64) return -95;
  const int num_cu = cu_count();
  if (!num_cu) return -5;
  return K == 384 ? launch_linear_regs_t<24, 4, kLinear>(x, w, bias, y, nullptr, T, N, num_cu, stream)
                  : launch_linear_regs_t<12, 4, kLinear>(x, w, bias, y, nullptr, T, N, num_cu, stream);
}

// d_x = d_y . W for W [K, N] as it lies (K the layer's width out, N its width in)
int launch_linear_columns(const void* x, const void* w, void* y, long long T, int N, int K, hipStream_t stream) {
  if (!linear_regs_supported(K, N) || T <= 0 || T > 0x7fffffffLL - 64) return -95;
  const int num_cu = cu_count();
  if (!num_cu) return -5;
  return K == 384 ? launch_linear_regs_t<24, 4, kColumns>(x, w, nullptr, y, nullptr, T, N, num_cu, stream)
                  : launch_linear_regs_t<12, 4, kColumns>(x, w, nullptr, y, nullptr, T, N, num_cu, stream);
}

int launch_linear_swiglu_bwd(const void* d_out, const void* w_down, const void* kept, void* d_kept, long long T, int K, int I,
                             hipStream_t stream) {
  if (!linear_swiglu_supported(K, I) || T <= 0 || T > 0x7fffffffLL - 64) return -95;
  const int num_cu = cu_count();
  if (!num_cu) return -5;
  void* const z = const_cast<void*>(kept);  // (read only in this form)
  return K == 384 ? launch_linear_regs_t<24, 4, kSwigluBwd>(d_out, w_down, nullptr, d_kept, z, T, I, num_cu, stream)
                  : launch_linear_regs_t<12, 4, kSwigluBwd>(d_out, w_down, nullptr, d_kept, z, T, I, num_cu, stream);
}

}  // namespace vig
