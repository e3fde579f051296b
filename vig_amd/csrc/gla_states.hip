// Segment states of long sequences (gfx950), bf16, Dk = 32, Dv = 64: per (sequence, segment, direction) what the
// segment's tokens contribute to the state that leaves it, U = sum_t w_t k_t v_t^T, and the segment's total decay; for the
// backward also the gradient states, the same sums over (q, d_o).
//   plain set:     forward  w_t = exp(gates of the tokens behind t),  reverse  w_t = exp(gates of the tokens before t)
//   gradient set:  forward  w_t = exp(gates up to and with t),        reverse  w_t = exp(gates from t on)
// (flash-linear-attention/fla/ops/gla/chunk_fuse.py:76-97 carries the state chunk by chunk; :413-518 its gradient.)
//
// One workgroup per (sequence, segment), each wave two 32-token tiles.  Everything is read with tokens in the contraction slots
// (mfma_tiles.h), so a lane owns channels: a tile's cumulative gates come out of a triangular-ones product in the layout that
// weights the keys and feeds the next product, and the tiles' totals, exchanged through LDS, anchor the weights at the segment's
// edge as one addition per channel.  The waves' sums meet in LDS.  The weighted key goes in as two bf16
// pieces (17 bits) against v as it is: no range to guard, and the kernel waits for memory, not for the matrix pipe.
// The lanes' upper half, which holds no channel, carries the other direction: one pass serves both.  (64 channels, which fill the lanes,
// have gla_mfma.hip's state pass.)
// Whole op, us, against the chunked kernel's state pass (one workgroup of eight waves per CU, four chunks walked each
// way): 24 sequences of 4096 tokens 47.5 -> 44.9, 45 of 1679 44.9 -> 41.7, 147 of 534 43.6 -> 40.5.
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

struct StateArgs {
  const uint16_t *k, *v, *gf, *gb;  // gb null: forward direction only
  const uint16_t *q, *d_o;          // gradient set (blockIdx.z = 1), or null
  float *slots, *grad_slots;        // [sequence][segment][2] slots of kGlaStateFloats
  int L, seg_len, nseg;
  // k, v inside wider rows: strides (batch, head, token) in elements; gates made from rank-16 rows (low_ld elements apart), see gla_tiles.hip
  long long sk[3], sv[3], low_ld;
  const uint16_t *low, *up_w, *up_b;
  float inv_norm, clamp;
  int H;
};

constexpr int kStateTiles = 16;  // most tiles of a segment
constexpr int kStateRedBytes = 64 * 64 * 4;
constexpr int state_lds(int waves) { return kStateTiles * 64 * 4 + waves * kStateRedBytes; }

// tokens j that row token i of the cumulative product adds up: before or behind i, with or without i itself
__device__ __forceinline__ uint32_t token_bits(bool before, bool with_own, int i) {
  const uint32_t lower = (1u << i) - 1u, own = 1u << i;
  return (before ? lower : ~(lower | own)) | (with_own ? own : 0u);
}

// the state's product of one tile: U[pk][pv] += (k w)^T v
__device__ __forceinline__ void add_tile(const u32x4_t (&kf)[2][2], const u32x4_t (&vf)[2][2], const f32x16_t (&G)[2],
                                         const float (&off)[2], f32x16_t (&U)[2][2]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      u32x4_t hi, lo;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float a = bf16lo_to_f32(kf[t][p][x]) * exp2_fast((G[p][8 * t + 2 * x] + off[p]) * kLog2e);
        const float b = bf16hi_to_f32(kf[t][p][x]) * exp2_fast((G[p][8 * t + 2 * x + 1] + off[p]) * kLog2e);
        hi[x] = pack_bf16x2(a, b);
        lo[x] = pack_bf16x2(a - bf16lo_to_f32(hi[x]), b - bf16hi_to_f32(hi[x]));
      }
#pragma unroll
      for (int pv = 0; pv < 2; ++pv) {
        U[p][pv] = mfma(hi, vf[t][pv], U[p][pv]);
        U[p][pv] = mfma(lo, vf[t][pv], U[p][pv]);
      }
    }
}

// LOW: one matrix instruction per channel parity makes a tile's gates of both directions from its rank-16 rows, where the lanes
// would have read them.
__device__ __forceinline__ void lowrank_gates(u32x4_t x, u32x4_t w, float bias, float inv_norm, float clamp, int rows, int h,
                                              u32x4_t (&gate)[2]) {
  f32x16_t acc = {0.f};
  acc = mfma(x, w, acc);
  lowrank_to_gates(acc, bias, inv_norm, clamp, rows, h, gate);
}

}  // namespace

template <bool LOW>
__global__ __launch_bounds__(512, 2) void gla_states_kernel(StateArgs a) {
  extern __shared__ __align__(16) char lds[];
  constexpr int NG = 2, DK = 16 * NG;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const bool grad = !LOW && blockIdx.z != 0, bidir = LOW || a.gb != nullptr;
  const int seq = blockIdx.x, seg = blockIdx.y;
  float* tot = reinterpret_cast<float*>(lds);  // [tile][p][lane row]
  char* red = lds + kStateTiles * 64 * 4;

  // ---- loads of both tiles ----
  const unsigned ch2 = cpair<NG>(r & 15);
  uint32_t gD[2][2][8], kD[2][2][8], vD[2][2][8];
  const int batch = LOW ? seq / a.H : 0, head = LOW ? seq - batch * a.H : 0;
  u32x4_t lowx[2], loww[2];
  uint32_t lowb[2];
  if (LOW) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int c = ((r >> 4) * a.H + head) * DK + 2 * (int)ch2 + p;
      loww[p] = *reinterpret_cast<const u32x4_t*>(a.up_w + 16 * (size_t)c + 8 * h);
      lowb[p] = a.up_b[c];
    }
  }
  const unsigned base = (4u * h) * (2u * DK) + 4u * ch2;
  size_t at[2];
  int rows[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // (all gates first: the totals are out, and the first tile's products at work, while the rest arrives)
    const int tok = seg * a.seg_len + 32 * (2 * w + i);
    rows[i] = __builtin_amdgcn_readfirstlane(max(0, min(32, min(a.L, (seg + 1) * a.seg_len) - tok)));
    at[i] = LOW ? (size_t)(rows[i] > 0 ? tok : 0) : (size_t)seq * a.L + (rows[i] > 0 ? tok : 0);
    if constexpr (LOW) {
      const unsigned pitch = 2u * (unsigned)a.low_ld;
      const rsrc_t rl = chunk_rsrc(a.low + ((long long)batch * a.L + (long long)at[i]) * a.low_ld, rows[i], pitch);
      lowx[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rl, (unsigned)r * pitch + 16u * h, 0, 0));
      continue;
    }
    const rsrc_t rf = chunk_rsrc(a.gf + at[i] * DK, rows[i], 2 * DK);
    const rsrc_t rb = chunk_rsrc((bidir ? a.gb : a.gf) + at[i] * DK, bidir ? rows[i] : 0, 2 * DK);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned off = base + (unsigned)jmap(t, 0, e) * (2u * DK);
        // (a lane of the other half reads beyond the descriptor: zero)
        const uint32_t f = __builtin_amdgcn_raw_buffer_load_b32(rf, r < 16 ? off : kOutOfRange, 0, 0);
        const uint32_t b = __builtin_amdgcn_raw_buffer_load_b32(rb, r < 16 ? kOutOfRange : off, 0, 0);
        gD[i][t][e] = f | b;
      }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (LOW) {
      const unsigned pk = 2u * (unsigned)a.sk[2], pv = 2u * (unsigned)a.sv[2];
      const rsrc_t rk = chunk_rsrc(a.k + batch * a.sk[0] + head * a.sk[1] + (long long)at[i] * a.sk[2], rows[i], pk);
      const rsrc_t rv = chunk_rsrc(a.v + batch * a.sv[0] + head * a.sv[1] + (long long)at[i] * a.sv[2], rows[i], pv);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          kD[i][t][e] = __builtin_amdgcn_raw_buffer_load_b32(rk, (4u * h) * pk + 4u * ch2, (unsigned)jmap(t, 0, e) * pk, 0);
      issue_tdwords_pitched<0, 2, 4>(rv, r, h, pv, vD[i]);
      continue;
    }
    const rsrc_t rk = chunk_rsrc((grad ? a.q : a.k) + at[i] * DK, rows[i], 2 * DK);
    const rsrc_t rv = chunk_rsrc((grad ? a.d_o : a.v) + at[i] * 64, rows[i], 128);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) kD[i][t][e] = __builtin_amdgcn_raw_buffer_load_b32(rk, base + (unsigned)jmap(t, 0, e) * (2u * DK), 0, 0);
    issue_tdwords<0, 2, 4>(rv, r, h, vD[i]);
  }

  // ---- the tiles' totals, to everybody ----
  u32x4_t gfrag[2][2][2];
  float own[2][2];
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (!LOW) finish_tfrags<2>(gD[i], gfrag[i]);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if constexpr (LOW) {
        u32x4_t gate[2];
        lowrank_gates(lowx[i], loww[p], __uint_as_float(lowb[p] << 16), a.inv_norm, a.clamp, rows[i], h, gate);
        gfrag[i][0][p] = gate[0], gfrag[i][1][p] = gate[1];
      }
      f32x16_t T = {0.f};
      T = mfma(ones, gfrag[i][0][p], T);
      T = mfma(ones, gfrag[i][1][p], T);
      own[i][p] = T[0];
      if (h == 0) tot[(2 * w + i) * 64 + 32 * p + r] = T[0];
    }
  }
  lds_barrier();
  float before[2] = {0.f, 0.f}, behind[2] = {0.f, 0.f};
#pragma unroll 1
  for (int t = 0; t < 2 * waves; ++t)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const float x = tot[t * 64 + 32 * p + r];
      before[p] += t < 2 * w ? x : 0.f;
      behind[p] += t > 2 * w + 1 ? x : 0.f;
    }

  // ---- decays ----
  float* out = (grad ? a.grad_slots : a.slots) + ((size_t)seq * a.nseg + seg) * 2 * kGlaStateFloats;
  if (w == 0 && h == 0 && !grad) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const float all = before[p] + own[0][p] + own[1][p] + behind[p];
      out[(r >> 4) * kGlaStateFloats + 64 * 64 + 2 * ch2 + p] = exp2_fast(all * kLog2e);
    }
  }

  // ---- weights, products, the waves' sums ----
  f32x16_t U[2][2] = {{{0.f}, {0.f}}, {{0.f}, {0.f}}};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    u32x4_t kf[2][2], vf[2][2];
    finish_tfrags<2>(kD[i], kf);
    finish_tfrags<2>(vD[i], vf);
    f32x16_t G[2];
    float off[2];
    const bool up = grad;  // the lower lane half's (forward) direction adds up the tokens before
    const uint32_t bits = token_bits(up, grad, r) >> (4 * h);
    const u32x4_t tri0 = keep_masks<0>(bits) & 0x3F803F80u, tri1 = keep_masks<1>(bits) & 0x3F803F80u;
    const uint32_t obits = token_bits(!up, grad, r) >> (4 * h);
    const u32x4_t otri0 = keep_masks<0>(obits) & 0x3F803F80u, otri1 = keep_masks<1>(obits) & 0x3F803F80u;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      f32x16_t g = {0.f}, o = {0.f};
      g = mfma(tri0, gfrag[i][0][p], g);
      G[p] = mfma(tri1, gfrag[i][1][p], g);
      o = mfma(otri0, gfrag[i][0][p], o);
      o = mfma(otri1, gfrag[i][1][p], o);
#pragma unroll
      for (int c = 0; c < 16; ++c) G[p][c] = r < 16 ? G[p][c] : o[c];
      const float b = before[p] + (i == 1 ? own[0][p] : 0.f), e = behind[p] + (i == 0 ? own[1][p] : 0.f);
      off[p] = (r >= 16) != up ? b : e;
    }
    add_tile(kf, vf, G, off, U);
  }
  char* mine = red + w * kStateRedBytes;
#pragma unroll
  for (int pk = 0; pk < 2; ++pk)
#pragma unroll
    for (int pv = 0; pv < 2; ++pv)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4_t x = {U[pk][pv][4 * g], U[pk][pv][4 * g + 1], U[pk][pv][4 * g + 2], U[pk][pv][4 * g + 3]};
        *reinterpret_cast<f32x4_t*>(unit_ptr(mine, (pk * 2 + pv) * 4 + g, lane)) = x;
      }
  lds_barrier();
  for (int i = threadIdx.x; i < 16 * 64; i += blockDim.x) {
    f32x4_t x = *reinterpret_cast<const f32x4_t*>(red + 16 * i);
    for (int o = 1; o < waves; ++o) x += *reinterpret_cast<const f32x4_t*>(red + o * kStateRedBytes + 16 * i);
    // (register quads 0, 1 are the forward direction's, 2, 3 the reverse one's)
    const int u = i >> 6, g = u & 3;
    if (g < 2 || bidir) *reinterpret_cast<f32x4_t*>(out + (g >> 1) * kGlaStateFloats + (((u & ~3) | (g & 1)) * 64 + (i & 63)) * 4) = x;
  }
}

// Contributions and decays of every (sequence, segment of seg_len tokens, direction) to `slots`; with q and d_o the gradient
// states to `grad_slots` in the same launch.
int launch_gla_states(const GlaArgs& a, int seg_len, int nseg, float* slots, const void* q, const void* d_o, float* grad_slots) {
  const int NT = (seg_len + 31) / 32;
  if (NT < 1 || NT > kStateTiles || nseg > 65535) return -22;
  StateArgs s{(const uint16_t*)a.k, (const uint16_t*)a.v, (const uint16_t*)a.g_fwd, (const uint16_t*)a.g_bwd,
              (const uint16_t*)q, (const uint16_t*)d_o, slots, grad_slots, a.L, seg_len, nseg};
  const int waves = (NT + 1) / 2;
  const dim3 grid(a.B * a.H, nseg, q ? 2 : 1), block(64 * waves);
  static bool done[64] = {}, done_low[64] = {};
  if (a.Dk != 32) return -95;
  if (a.low) {
    if (q || !a.k_strides || !a.v_strides) return -22;
    for (int j = 0; j < 3; ++j) s.sk[j] = a.k_strides[j], s.sv[j] = a.v_strides[j];
    s.low = (const uint16_t*)a.low, s.up_w = (const uint16_t*)a.up_w, s.up_b = (const uint16_t*)a.up_b;
    s.low_ld = a.low_ld, s.inv_norm = a.inv_norm, s.clamp = a.clamp, s.H = a.H;
    if (!allow_lds(reinterpret_cast<const void*>(gla_states_kernel<true>), state_lds(kStateTiles / 2), done_low)) return -5;
    hipLaunchKernelGGL(gla_states_kernel<true>, grid, block, state_lds(waves), a.stream, s);
  } else {
    if (!allow_lds(reinterpret_cast<const void*>(gla_states_kernel<false>), state_lds(kStateTiles / 2), done)) return -5;
    hipLaunchKernelGGL(gla_states_kernel<false>, grid, block, state_lds(waves), a.stream, s);
  }
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

}  // namespace vig
