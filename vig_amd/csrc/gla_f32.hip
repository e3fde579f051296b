// Bidirectional GLA forward of fp32 tensors on the matrix cores (gfx950), Dk in {32, 64}, Dv = 64: the tile-pair scheme of
// gla_tiles.hip (one workgroup per sequence of up to seven 32-token tiles, one wave per query tile, longer sequences as
// segments linked by states) with every operand in three bf16 pieces (f32_tiles.h), so that inputs, products and sums
// keep fp32's precision.
//
// What bounds it: the matrix pipe and the vector instructions that cut operands into pieces, about equally.  A wave
// meets NT + 1 key tiles: 48 matrix instructions of 32 clocks per tile pair at Dk = 64, beside 300 vector instructions
// (q^ over the tile just passed and into pieces, the score tile into pieces).  In pieces a key tile takes 12 KB of LDS
// and so does a value tile, so the two directions take turns: forward operands, barrier, forward walk, barrier, then
// the reverse ones in the same 73 KB; with the values' 84 KB one workgroup fills a CU.  Query tiles are dealt to the
// waves so that the two waves of a SIMD walk the same number of tiles together in either direction.
// The token-recurrent kernel this replaces for these shapes is bound by its serial chain of L tokens.
// B 32, H 6, L 197, D 64: 181 us before; measured figures at launch_gla_f32.
//
// Decays per tile as in gla_tiles.hip, in log2 units: G = inclusive cumulative gate in the direction's walk order, T the
// tile's total, q^ = q 2^G for the walk, k^ = k 2^(T-G) published, q' = q 2^(G-T) against k^ for the wave's own tile (one
// set of key pieces serves both).  Only q' grows, so the form holds while |G| <= 40 in every channel of every tile (a mean
// gate of -0.87 per token) and the inputs stay below 1e12.  A workgroup that meets stronger gates does its tokens again with
// operands for any gates (prepare32_any); inputs beyond the bound, gates that grow and gates that are no numbers take the
// serial form (serial_segment).  All sequences strongly gated: B 32, H 6, L 197, D 64 81 us (mildly gated 37; the
// token-recurrent kernel 182, the serial form, one wave of a workgroup, 1069); 768 sequences 233 us (112 / 221 / 3214).
#include <algorithm>

#include "f32_tiles.h"

namespace vig {

namespace {

constexpr float kRange32 = 40.0f;
constexpr float kMagnitude32 = 1e12f;

struct F32Geo {
  int L, NT, nseg;      // tokens per sequence, tiles per segment, segments per sequence
  const float* states;  // long sequences: scanned slots; null: whole sequences
  // from sequence `whole` on a (whole) sequence's directions go to two workgroups, the reverse one leaving its outputs in `half`: 32 NT
  // rows a sequence
  int whole;
  float* half;
};

template <int NG>
struct F32Lds {
  static constexpr int KB = NG * 3072;  // one k^ tile
  static constexpr int VB = 12288;      // one V tile
  int v, d, sc, flag, total;
  __host__ __device__ explicit F32Lds(int NT) {
    v = (NT - 1) * KB;
    d = v + NT * VB;
    sc = d + NT * 256;
    flag = sc + NT * 256;
    total = flag + 64;
  }
};

// Operands of one direction for this wave's tile: q^ (kept), k^ and the tile's decays (published), the masked diagonal
// scores P.  Returns (wave-uniform) whether the tile is outside the form's range.
template <int NG, bool FWD>
__device__ __forceinline__ bool prepare32(const f32x8_t (&q)[NG], const f32x8_t (&k)[NG], f32x8_t (&g)[NG], float* sc,
                                          float* dtab, char* kreg, int lane, f32x8_t (&qh)[NG], f32x16_t& P) {
  constexpr int HC = 8 * NG;
  const int r = lane & 31, h = lane >> 5;
  float top = 0.f;
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    f32x8_t own = g[c] * kLog2e, p;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = prefix32(own[e]);
      top = fmaxf(top, fabsf(p[e]));
      if (r == 31) sc[HC * h + 8 * c + e] = p[e];
    }
    g[c] = FWD ? p : p - own;  // reverse: what lies before the token, T minus it is G
  }
  wave_lds_sync();
  const float tl = sc[lane & (16 * NG - 1)];
  const bool wide = __builtin_amdgcn_ballot_w64(!(top <= kRange32) || !(fabsf(tl) <= kRange32)) != 0;
  if (lane < 16 * NG) dtab[lane] = exp2_fast(tl);
  wave_lds_sync();
  __builtin_amdgcn_sched_barrier(0);
  P = f32x16_t{0.f};
  f32x16_t Ps = {0.f};
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    const f32x8_t T = lds_f32x8(sc + HC * h + 8 * c), D = lds_f32x8(dtab + HC * h + 8 * c);
    const f32x8_t rest = FWD ? T - g[c] : g[c];  // T - G
    f32x8_t qt, kh;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      kh[e] = k[c][e] * exp2_fast(rest[e]);
      qt[e] = q[c][e] * exp2_fast(-rest[e]);
    }
    const P3 kp = split8(kh);
    if (kreg) store_p3(kreg, c, lane, kp);
    mfma6(kp, split8(qt), P, Ps);
    qh[c] = qt * D;
    __builtin_amdgcn_sched_barrier(0);  // (piece by piece: sixteen channels' factors at once would not fit)
  }
  // keep the pairs the direction sees: register 4g + m is key 8g + 4h + m, the lane's query is r
  const int rel = r - 4 * h;
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const int j = 8 * (c >> 2) + (c & 3);
    const bool keep = FWD ? j <= rel : j >= rel;
    P[c] = keep ? P[c] + Ps[c] : 0.f;
  }
  return wide;
}

// x where every bit of m is set, y where none is (one instruction; a choice by condition became branches here)
__device__ __forceinline__ float pick(uint32_t m, float x, float y) {
  return __uint_as_float((__float_as_uint(x) & m) | (__float_as_uint(y) & ~m));
}

// The same for any gates that do not grow (sums down to -inf): no factor is ever above one.  A pair of tokens (query i, key j)
// differs first in some bit m of its numbers; the start of the upper half of their common 2m tokens lies between them, and
// the decay splits there: the query's gates summed over its own m tokens up to it (inc), the key's over the rest of its m
// tokens (exc), both plain sums of gates.  A token is a query or a key of a level, never both, so one operand holds both,
// and a level is one product of it with itself of which the level's pairs are taken.  Five levels and the pair i = j (which
// decays nothing) take the place of the one product above; the vector instructions of a level bound it: 700 of them beside
// 24 matrix instructions at Dk = 64.
template <int NG, bool FWD>
__device__ __forceinline__ void prepare32_any(const f32x8_t (&q)[NG], const f32x8_t (&k)[NG], f32x8_t (&inc)[NG], float* dtab,
                                              char* kreg, int lane, f32x8_t (&qh)[NG], f32x16_t& P) {
  constexpr int HC = 8 * NG;
  const int r = lane & 31, h = lane >> 5;
  f32x8_t exc[NG];
  float dot = 0.f;
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    inc[c] *= kLog2e;
    exc[c] = f32x8_t{0.f};
#pragma unroll
    for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(q[c][e], k[c][e], dot);
  }
  dot += __shfl_xor(dot, 32, 64);
#pragma unroll
  for (int c = 0; c < 16; ++c) P[c] = 8 * (c >> 2) + (c & 3) + 4 * h == r ? dot : 0.f;
#pragma unroll 1
  for (int m = 1; m < 32; m *= 2) {
    const uint32_t query = ((r & m) != 0) == FWD ? ~0u : 0u;
    // the lane that holds the whole sum of the other m tokens
    const int other = 4 * (32 * h + (FWD ? (r ^ m) | (m - 1) : (r ^ m) & ~(m - 1)));
    f32x16_t Pm = {0.f}, Ps = {0.f};
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      f32x8_t x;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = pick(query, q[c][e], k[c][e]) * exp2_fast(pick(query, inc[c][e], exc[c][e]));
        const float t = __uint_as_float(__builtin_amdgcn_ds_bpermute(other, __float_as_uint(inc[c][e])));
        inc[c][e] += pick(query, t, 0.f);
        exc[c][e] += pick(query, 0.f, t);
      }
      const P3 p = split8(x);
      mfma6(p, p, Pm, Ps);
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const int key = 8 * (c >> 2) + (c & 3) + 4 * h;
      const bool mine = ((r ^ key) & -m) == m && (FWD ? r > key : key > r);
      P[c] = mine ? Pm[c] + Ps[c] : P[c];
    }
  }
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    f32x8_t kh;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = exp2_fast(inc[c][e]);
      kh[e] = k[c][e] * exp2_fast(exc[c][e]);
      qh[c][e] = q[c][e] * d;
      if (r == (FWD ? 31 : 0)) dtab[HC * h + 8 * c + e] = d;
    }
    if (kreg) store_p3(kreg, c, lane, split8(kh));
  }
}

// O^T += V^T P
__device__ __forceinline__ void apply_values32(const f32x16_t& P, char* vreg, int lane, f32x16_t (&O)[2]) {
  const P3 p[2] = {split8(half_of<0>(P)), split8(half_of<1>(P))};
#pragma unroll
  for (int pv = 0; pv < 2; ++pv) {
    f32x16_t Os = {0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t) mfma6(load_p3(vreg, 2 * t + pv, lane), p[t], O[pv], Os);
    O[pv] += Os;
  }
}

template <int NG>
__device__ __forceinline__ void decay_q(const float* d, int h, f32x8_t (&qh)[NG]) {
#pragma unroll
  for (int c = 0; c < NG; ++c) qh[c] *= lds_f32x8(d + 8 * NG * h + 8 * c);
}

// outward walk over the other tiles of one direction
template <int NG, bool FWD>
__device__ __forceinline__ void walk32(char* lds, const F32Lds<NG>& lay, int ti, int NT, int lane, f32x8_t (&qh)[NG],
                                       f32x16_t (&O)[2]) {
  const int n = FWD ? ti : NT - 1 - ti;
#pragma unroll 1
  for (int s = 1; s <= n; ++s) {
    const int j = FWD ? ti - s : ti + s;
    if (s > 1) decay_q<NG>(reinterpret_cast<const float*>(lds + lay.d) + 64 * (FWD ? j + 1 : j - 1), lane >> 5, qh);
    // matrix and vector instructions in turns: left to itself the compiler put the cutting of a tile's operands into one run in
    // front of its products (B 64, H 6, L 196, Dk 32 51.7 -> 48.9 us, one image 23.2 -> 21.7)
    __builtin_amdgcn_iglp_opt(0);
    char* kreg = lds + (FWD ? j : j - 1) * F32Lds<NG>::KB;
    f32x16_t P = {0.f}, Ps = {0.f};
#pragma unroll
    for (int c = 0; c < NG; ++c) mfma6(load_p3(kreg, c, lane), split8(qh[c]), P, Ps);
    P += Ps;
    apply_values32(P, lds + lay.v + j * F32Lds<NG>::VB, lane, O);
  }
}

// what the state entering the segment adds: O^T += S_in^T q^, q^ anchored at the segment's edge
template <int NG, bool FWD>
__device__ __forceinline__ void apply_state32(const float* slot, const float* edge, bool cross, int lane, f32x8_t (&qh)[NG],
                                              f32x16_t (&O)[2]) {
  if (cross) decay_q<NG>(edge, lane >> 5, qh);
#pragma unroll
  for (int pv = 0; pv < 2; ++pv) {
    f32x16_t Os = {0.f};
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(slot + ((pv * 4 + c) * 64 + lane) * 4);
      const f32x4_t b = *reinterpret_cast<const f32x4_t*>(slot + (((2 + pv) * 4 + c) * 64 + lane) * 4);
      mfma6(split8(__builtin_shufflevector(a, b, 0, 4, 1, 5, 2, 6, 3, 7)), split8(qh[c]), O[pv], Os);
    }
    O[pv] += Os;
  }
}

// One direction of a segment, token by token (any gates, any magnitudes): one wave, lane = value channel, the state's
// column in registers, rows of q, k, exp(g) staged through LDS four tokens at a time.  Outputs go to (or are added to)
// obuf [n][64].
template <int NG, bool FWD>
__device__ __forceinline__ void serial_direction(const float* q, const float* k, const float* v, const float* g, int n,
                                                 const float* slot, float* stage, float* obuf, bool add, int lane) {
  constexpr int DK = 16 * NG;
  float S[DK];
#pragma unroll
  for (int c = 0; c < DK; ++c) S[c] = slot ? slot[state_index<NG>(c, lane)] : 0.f;
  const int nb = (n + 3) / 4;
  for (int ib = 0; ib < nb; ++ib) {
    const int t0 = 4 * (FWD ? ib : nb - 1 - ib);
    wave_lds_sync();
    for (int i = lane; i < 4 * DK; i += 64) {
      const int t = t0 + i / DK;
      const bool ok = t < n;
      const size_t at = (size_t)t * DK + i % DK;
      stage[i] = ok ? q[at] : 0.f;
      stage[4 * DK + i] = ok ? k[at] : 0.f;
      stage[8 * DK + i] = ok ? __expf(g[at]) : 1.f;
    }
    wave_lds_sync();
    for (int it = 0; it < 4; ++it) {
      const int u = FWD ? it : 3 - it, t = t0 + u;
      if (t >= n) continue;
      const float vv = v[(size_t)t * 64 + lane];
      float po = 0.f;
#pragma unroll
      for (int c = 0; c < DK; ++c) {
        S[c] = S[c] * stage[8 * DK + u * DK + c] + stage[4 * DK + u * DK + c] * vv;
        po += stage[u * DK + c] * S[c];
      }
      obuf[t * 64 + lane] = add ? obuf[t * 64 + lane] + po : po;
    }
  }
}

template <int NG, int DIRS>  // 1 forward, 2 reverse
__device__ __noinline__ void serial_segment(const float* q, const float* k, const float* v, const float* gf, const float* gb,
                                            float* o, const float* slots, int n, int stage_at, float oscale) {
  extern __shared__ __align__(16) char lds[];
  float* obuf = reinterpret_cast<float*>(lds);
  float* stage = reinterpret_cast<float*>(lds + stage_at);
  const int lane = threadIdx.x & 63;
  lds_barrier();  // everyone is done with the tiles
  if (threadIdx.x >= 64) return;
  if (DIRS & 1) serial_direction<NG, true>(q, k, v, gf, n, slots, stage, obuf, false, lane);
  if (DIRS & 2)
    serial_direction<NG, false>(q, k, v, gb, n, slots ? slots + kGlaStateFloats : nullptr, stage, obuf, DIRS == 3, lane);
  for (int t = 0; t < n; ++t) o[(size_t)t * 64 + lane] = oscale * obuf[t * 64 + lane];
}

// Where a workgroup's tokens and this wave's tile lie.
template <int NG>
struct F32Place {
  const float *q, *k, *v, *gf, *gb, *slots;  // the segment's first token; states that enter it, or null
  float* o;
  int n, NT, ti;  // tokens left from the segment's start on, tiles, this wave's tile
  rsrc_t rq, rk, rv, rgf, rgb, ro;  // its tile's rows
};
template <int NG, int DIRS, bool HALVES>
__device__ __forceinline__ F32Place<NG> f32_place(const float* q, const float* k, const float* v, const float* gf, const float* gb,
                                                  float* o, const F32Geo& geo) {
  constexpr int DK = 16 * NG;
  F32Place<NG> p;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // waves w and w + 4 share a SIMD: tiles NT-1-w and w together see NT + 3 - w - (NT-1-w) ... the same number of tiles
  // in both directions
  p.NT = geo.NT, p.ti = w < 4 ? p.NT - 1 - w : w - 4;
  int seq = blockIdx.x, seg = blockIdx.y;
  const int which = (int)blockIdx.x - geo.whole;
  if (HALVES) seg = 0, seq = which < 0 ? blockIdx.x : geo.whole + (which >> 1);
  const int first = 32 * seg * p.NT;
  const size_t at = (size_t)seq * geo.L + first;
  p.n = geo.L - first;
  p.q = q + at * DK, p.k = k + at * DK, p.v = v + at * 64, p.gf = gf + at * DK, p.gb = (DIRS & 2 ? gb : gf) + at * DK;
  p.o = DIRS == 2 ? geo.half + (size_t)(which >> 1) * (32 * p.NT) * 64 : o + at * 64;
  p.slots = geo.states ? geo.states + ((size_t)seq * geo.nseg + seg) * 2 * kGlaStateFloats : nullptr;
  const int nvalid = __builtin_amdgcn_readfirstlane(max(0, min(32, p.n - 32 * p.ti)));
  const int tile = 32 * p.ti;
  p.rq = chunk_rsrc(p.q + tile * DK, nvalid, 4 * DK), p.rk = chunk_rsrc(p.k + tile * DK, nvalid, 4 * DK);
  p.rv = chunk_rsrc(p.v + tile * 64, nvalid, 256), p.ro = chunk_rsrc(p.o + tile * 64, nvalid, 256);
  p.rgf = chunk_rsrc(p.gf + tile * DK, nvalid, 4 * DK), p.rgb = chunk_rsrc(p.gb + tile * DK, nvalid, 4 * DK);
  return p;
}

enum F32Range { kInRange = 0, kGatesBeyond = 1, kValuesBeyond = 2 };

// The walk of both directions; ANY: with prepare32_any, over the values' pieces that the pass before left in LDS.  Returns
// (workgroup-uniform) what is beyond the form's range, before anything is stored.
template <int NG, int DIRS, bool ANY>
__device__ __forceinline__ int f32_pass(const F32Place<NG>& p, char* lds, float oscale) {
  constexpr bool F1 = DIRS != 2;  // the first direction, or the only one
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int NT = p.NT, ti = p.ti;
  const F32Lds<NG> lay(NT);
  char* vreg = lds + lay.v + ti * F32Lds<NG>::VB;
  float* sc = reinterpret_cast<float*>(lds + lay.sc) + 64 * ti;
  float* dall = reinterpret_cast<float*>(lds + lay.d);
  int* flags = reinterpret_cast<int*>(lds + lay.flag);
  const auto beyond = [&](int why) { return __builtin_amdgcn_ballot_w64(lane < NT && (flags[lane < NT ? lane : 0] & why)) != 0; };

  f32x8_t xq[NG], xk[NG], xg[NG], qh[NG];
  f32x16_t P, O[2] = {f32x16_t{0.f}, f32x16_t{0.f}};
  char* kreg = F1 ? (ti < NT - 1 ? lds + ti * F32Lds<NG>::KB : nullptr) : (ti > 0 ? lds + (ti - 1) * F32Lds<NG>::KB : nullptr);
  if (ANY) {
    lds_barrier();  // everyone has read the flags
    float grows = 0.f, sum = 0.f;
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      if (!(DIRS & (1 << dir))) continue;
      load_rows_f32<NG>(dir ? p.rgb : p.rgf, r, h, xg);
#pragma unroll
      for (int c = 0; c < NG; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) grows = fmaxf(grows, xg[c][e]), sum += xg[c][e];
    }
    // (a gate that grows: 32 tokens of the largest stay in the range; sums of -inf are fine, of no number are not)
    const bool refused = __builtin_amdgcn_ballot_w64(!(grows * (32 * kLog2e) <= kRange32) || sum != sum) != 0;
    if (lane == 0) flags[ti] = refused ? kGatesBeyond : kInRange;
    lds_barrier();
    if (beyond(kGatesBeyond)) return kGatesBeyond;
    load_rows_f32<NG>(F1 ? p.rgf : p.rgb, r, h, xg);
    load_rows_f32<NG>(p.rq, r, h, xq);
    load_rows_f32<NG>(p.rk, r, h, xk);
    prepare32_any<NG, F1>(xq, xk, xg, dall + 64 * ti, kreg, lane, qh, P);
    apply_values32(P, vreg, lane, O);
    lds_barrier();
  } else {
    float mag = 0.f;
    {
      f32x8_t xv[2][2];
      load_pairs_f32(p.rv, r, h, xv);
      load_rows_f32<NG>(F1 ? p.rgf : p.rgb, r, h, xg);
      load_rows_f32<NG>(p.rq, r, h, xq);
      load_rows_f32<NG>(p.rk, r, h, xk);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int pv = 0; pv < 2; ++pv) {
          store_p3(vreg, 2 * t + pv, lane, split8(xv[pv][t]));
          mag += sum_abs(xv[pv][t]);  // (a sum: NaN and inf stay visible)
        }
    }
#pragma unroll
    for (int c = 0; c < NG; ++c) mag += sum_abs(xq[c]) + sum_abs(xk[c]);
    const bool large = __builtin_amdgcn_ballot_w64(!(mag < kMagnitude32)) != 0;
    __builtin_amdgcn_sched_barrier(0);  // (the values' registers are free before the operands' are needed: 35.5 -> 34.8 us)
    const bool wide = prepare32<NG, F1>(xq, xk, xg, sc, dall + 64 * ti, kreg, lane, qh, P);
    wave_lds_sync();
    apply_values32(P, vreg, lane, O);
    if (lane == 0) flags[ti] = large ? kValuesBeyond : wide ? kGatesBeyond : kInRange;
    lds_barrier();
    if (beyond(kGatesBeyond | kValuesBeyond)) return beyond(kValuesBeyond) ? kValuesBeyond : kGatesBeyond;
  }
  walk32<NG, F1>(lds, lay, ti, NT, lane, qh, O);
  if (p.slots)
    apply_state32<NG, F1>(p.slots + (F1 ? 0 : kGlaStateFloats), dall + (F1 ? 0 : 64 * (NT - 1)), F1 ? ti > 0 : ti < NT - 1, lane, qh, O);
  if (DIRS == 3) {
    int r2 = r;
    asm volatile("" : "+v"(r2));  // (fetched again: carried across the walk, q and k would take 64 registers)
    load_rows_f32<NG>(p.rgb, r2, h, xg);
    load_rows_f32<NG>(p.rq, r2, h, xq);
    load_rows_f32<NG>(p.rk, r2, h, xk);
    lds_barrier();  // the forward keys and decays have been read
    kreg = ti > 0 ? lds + (ti - 1) * F32Lds<NG>::KB : nullptr;
    if (ANY) {
      prepare32_any<NG, false>(xq, xk, xg, dall + 64 * ti, kreg, lane, qh, P);
      apply_values32(P, vreg, lane, O);
      lds_barrier();
    } else {
      const bool wide = prepare32<NG, false>(xq, xk, xg, sc, dall + 64 * ti, kreg, lane, qh, P);
      apply_values32(P, vreg, lane, O);
      if (lane == 0) flags[ti] = wide ? kGatesBeyond : kInRange;
      lds_barrier();
      if (beyond(kGatesBeyond)) return kGatesBeyond;
    }
    walk32<NG, false>(lds, lay, ti, NT, lane, qh, O);
    if (p.slots) apply_state32<NG, false>(p.slots + kGlaStateFloats, dall + 64 * (NT - 1), ti < NT - 1, lane, qh, O);
  }
  // lane (r, h) holds channels [32h, 32h + 32) of token r: register 4g + m of O[pv] is channel 32h + 8g + 2m + pv
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u32x4_t x;
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = __float_as_uint(O[m & 1][2 * i + (m >> 1)] * oscale);
    __builtin_amdgcn_raw_buffer_store_b128(x, p.ro, (unsigned)r * 256u + 128u * h + 16u * i, 0, 0);
  }
  return kInRange;
}

// The kernel's argument block as the hardware lays it out (every argument at its natural alignment).
struct F32KernArgs {
  const float *q, *k, *v, *gf, *gb;
  float* o;
  F32Geo geo;
  float oscale;
};
static_assert(offsetof(F32KernArgs, geo) == 6 * sizeof(void*) && offsetof(F32KernArgs, oscale) == 48 + sizeof(F32Geo) && alignof(F32Geo) == 8,
              "F32KernArgs has to mirror the parameter list of gla_f32_kernel");

// What is beyond the range, as a function of its own: its registers stay out of the common path's allocation.  (Arguments of a
// called function come in vector registers, and a descriptor built from one puts a loop around every load: the function
// reads the kernel's own through the argument block.)
template <int NG, int DIRS, bool HALVES>
__device__ __noinline__ void f32_beyond(const F32KernArgs* ka_in, int why) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass has no constant address space to copy the geometry from)
  extern __shared__ __align__(16) char lds[];
  const uint64_t kp = reinterpret_cast<uint64_t>(ka_in);
  typedef const F32KernArgs __attribute__((address_space(4))) * KernArgPtr;
  const KernArgPtr ka = (KernArgPtr)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(kp >> 32)) << 32) |
                                     (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)kp));
  const F32Geo geo = ka->geo;
  const auto p = f32_place<NG, DIRS, HALVES>(ka->q, ka->k, ka->v, ka->gf, ka->gb, ka->o, geo);
  if (__builtin_amdgcn_readfirstlane(why) == kGatesBeyond && f32_pass<NG, DIRS, true>(p, lds, ka->oscale) == kInRange) return;
  serial_segment<NG, DIRS>(p.q, p.k, p.v, p.gf, p.gb, p.o, p.slots, min(32 * p.NT, p.n), p.NT * 8192, ka->oscale);
#endif
}

}  // namespace

template <int NG, int DIRS, bool HALVES>
__global__ __launch_bounds__(512, 2) void gla_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                         const float* __restrict__ v, const float* __restrict__ gf,
                                                         const float* __restrict__ gb, float* __restrict__ o, F32Geo geo,
                                                         float oscale) {
  extern __shared__ __align__(16) char lds[];
  const F32KernArgs* ka = (const F32KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  if constexpr (!HALVES) {
    const int why = f32_pass<NG, DIRS, false>(f32_place<NG, DIRS, false>(q, k, v, gf, gb, o, geo), lds, oscale);
    if (why != kInRange) f32_beyond<NG, DIRS, false>(ka, why);
  } else {
    const int which = (int)blockIdx.x - geo.whole;
    if (which < 0) {
      const int why = f32_pass<NG, 3, false>(f32_place<NG, 3, true>(q, k, v, gf, gb, o, geo), lds, oscale);
      if (why != kInRange) f32_beyond<NG, 3, true>(ka, why);
    } else if ((which & 1) == 0) {
      const int why = f32_pass<NG, 1, false>(f32_place<NG, 1, true>(q, k, v, gf, gb, o, geo), lds, oscale);
      if (why != kInRange) f32_beyond<NG, 1, true>(ka, why);
    } else {
      const int why = f32_pass<NG, 2, false>(f32_place<NG, 2, true>(q, k, v, gf, gb, o, geo), lds, oscale);
      if (why != kInRange) f32_beyond<NG, 2, true>(ka, why);
    }
  }
}

// What the reverse workgroups of sequences in two halves left is added to the forward ones' (a workgroup: a quarter of a sequence).
__global__ __launch_bounds__(256) void gla_f32_add_kernel(float* __restrict__ o, F32Geo geo) {
  const float* half = geo.half + (size_t)blockIdx.x * (32 * geo.NT) * 64;
  float* to = o + (size_t)(geo.whole + blockIdx.x) * geo.L * 64;
  for (int i = (blockIdx.y * 256 + threadIdx.x) * 4; i < geo.L * 64; i += 4096)
    *reinterpret_cast<f32x4_t*>(to + i) += *reinterpret_cast<const f32x4_t*>(half + i);
}

// State pass of a long sequence: what every segment adds to the state of each direction, U = sum_t 2^(gates walked after
// t) k_t^T v_t, and the segment's decay, into the slots of gla_segment_scan_kernel.  Grid (sequence, segment, set); wave =
// (direction, half pv of the value channels), no LDS and no barrier: lane-row rho of a fragment owns NG/2 key channels, so the
// gates of a tile are summed token by token in its own registers (groups of four tokens alternate between the lane
// halves) and the tiles are taken against the walk order, so every exponent is a plain sum of gates, exact for any gates.
// Set 1 is the gradient states' pass of the backward: q for k, d_o for v, the directions' gates exchanged, each token's own
// gate included.
template <int NG>
__global__ __launch_bounds__(256, 2) void gla_f32_state_kernel(const float* __restrict__ k0, const float* __restrict__ v0,
                                                               const float* __restrict__ q1, const float* __restrict__ do1,
                                                               const float* __restrict__ gf, const float* __restrict__ gb,
                                                               float* __restrict__ ws, float* __restrict__ grad_ws,
                                                               int* __restrict__ flags, int L, int NT,
                                                               int nseg) {
  constexpr int DK = 16 * NG, NP = NG / 2;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int dir = w >> 1, pv = w & 1;
  const bool grad = blockIdx.z != 0;
  if (flags && blockIdx.y == 0 && !grad && threadIdx.x == 0) flags[blockIdx.x] = 0;
  const float* kk = grad ? q1 : k0;
  const float* vv = grad ? do1 : v0;
  const float* gg = (dir == 0) != grad ? gf : gb;
  const size_t seq0 = (size_t)blockIdx.x * L;
  const int first = 32 * NT * (int)blockIdx.y;
  // first key channel of this lane-row
  const int ch = NG == 4 ? 2 * cpair<4>(r) : 16 * ((r >> 2) & 1) + 8 * ((r >> 3) & 1) + 2 * (r & 3) + (r >> 4);
  const int vch = 2 * cpair<4>(r) + pv;
  float run[NP];
  f32x16_t acc[NP], accs[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) run[p] = 0.f, acc[p] = accs[p] = f32x16_t{0.f};
#pragma unroll 1
  for (int it = 0; it < NT; ++it) {
    const int tok = first + 32 * (dir == 0 ? NT - 1 - it : it);
    const int nvalid = __builtin_amdgcn_readfirstlane(max(0, min(32, L - tok)));
    if (nvalid == 0) continue;
    const rsrc_t rk = chunk_rsrc(kk + (seq0 + tok) * DK, nvalid, 4 * DK), rg = chunk_rsrc(gg + (seq0 + tok) * DK, nvalid, 4 * DK);
    const rsrc_t rv = chunk_rsrc(vv + (seq0 + tok) * 64, nvalid, 256);
    float xk[NP][16], xg[NP][16], xv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const unsigned at = (unsigned)(jmap(i >> 3, 0, i & 7) + 4 * h);
      if (NP == 2) {
        const u32x2_t a = __builtin_amdgcn_raw_buffer_load_b64(rg, at * (4u * DK) + 4u * ch, 0, 0);
        const u32x2_t b = __builtin_amdgcn_raw_buffer_load_b64(rk, at * (4u * DK) + 4u * ch, 0, 0);
        xg[0][i] = __uint_as_float(a[0]), xg[NP - 1][i] = __uint_as_float(a[1]);
        xk[0][i] = __uint_as_float(b[0]), xk[NP - 1][i] = __uint_as_float(b[1]);
      } else {
        xg[0][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rg, at * (4u * DK) + 4u * ch, 0, 0));
        xk[0][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, at * (4u * DK) + 4u * ch, 0, 0));
      }
      xv[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, at * 256u + 4u * vch, 0, 0));
    }
    P3 pvv[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) pvv[t] = split8(octet(xv, t));
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float tot[4], other[4];
#pragma unroll
      for (int i = 0; i < 16; ++i) xg[p][i] *= kLog2e;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        tot[u] = (xg[p][4 * u] + xg[p][4 * u + 1]) + (xg[p][4 * u + 2] + xg[p][4 * u + 3]);
        other[u] = __shfl_xor(tot[u], 32, 64);
      }
      // registers 4u .. 4u + 3 are tokens 8u + 4h + (0 .. 3)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float mine = dir == 0 ? tot[3 - x] : tot[x], theirs = dir == 0 ? other[3 - x] : other[x];
        // the half whose four tokens come first against the walk order: the upper one forward, the lower one reverse
        const bool late = (h == 1) != (dir == 0);
        float s = late ? run[p] + theirs : run[p];
        run[p] += mine + theirs;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          if (dir == 0) {
            const int i = 4 * (3 - x) + (3 - y);
            const float ex = grad ? s + xg[p][i] : s;
            s += xg[p][i];
            xk[p][i] *= exp2_fast(ex);
          } else {
            const int i = 4 * x + y;
            const float ex = grad ? s + xg[p][i] : s;
            s += xg[p][i];
            xk[p][i] *= exp2_fast(ex);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) mfma6(split8(octet(xk[p], t)), pvv[t], acc[p], accs[p]);
    }
  }
  float* slot = (grad ? grad_ws : ws) + (((size_t)blockIdx.x * nseg + blockIdx.y) * 2 + dir) * kGlaStateFloats;
#pragma unroll
  for (int p = 0; p < NP; ++p) acc[p] += accs[p];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int u = NG == 4 ? (p * 2 + pv) * 4 + g : ((g >> 1) * 2 + pv) * 4 + (g & 1);
      const f32x4_t x = {acc[p][4 * g], acc[p][4 * g + 1], acc[p][4 * g + 2], acc[p][4 * g + 3]};
      *reinterpret_cast<f32x4_t*>(slot + (u * 64 + lane) * 4) = x;
    }
  if (pv == 0 && h == 0) {
#pragma unroll
    for (int p = 0; p < NP; ++p) slot[64 * 64 + ch + p] = exp2_fast(run[p]);
  }
}

// Measured at B 32, H 6, L 197, D 64 (58 MB): 37 us per call (34.7 in a captured run), token-recurrent kernel 181 us.
constexpr int kF32MaxLds = 160 * 1024;

bool gla_f32_supported(const GlaArgs& a) {
  return a.io_dtype == 0 && a.gate_dtype == 0 && (a.Dk == 64 || a.Dk == 32) && a.Dv == 64 && !a.init_state && !a.final_state &&
         !a.state_pass && !a.gate_w && !a.q_strides && !a.k_strides && !a.v_strides && gla_f32_segments(a.L) <= 65535 &&
         (gla_f32_segments(a.L) == 1 || (long long)a.B * a.H * 2 <= 65535);
}
static size_t f32_states(long long nseq, int L, int NT) {
  return (size_t)nseq * (((L + 31) / 32 + NT - 1) / NT) * 2 * kGlaStateFloats * sizeof(float);
}
// Whole sequences whose directions go to two workgroups: what is left over of full rounds of the chip, where that fills no more than
// half of one, from five tiles on.  us, whole / halves: Dk 32: 18 sequences of 185 tokens 21.0 / 16.2, 120 of 196 23.9 / 22.1, 384 50.3 /
// 48.0; Dk 64: 18 of 185 30.0 / 21.9, 60 of 196 33.4 / 26.6, 384 71.7 / 65.5.  Below, the second launch and its memory cost what the
// halves gain (Dk 32, 18 of 64 10.4 / 9.7; 108 of 85 called one by one 11.9 / 12.4), and so they do for segments (12 of 1031 28.0 / 30.4).
template <int NG>
static int f32_fwd_halves(int n, int NT) {
  const int slots = 256 * std::max(1, std::min(kF32MaxLds / F32Lds<NG>(NT).total, 8 / NT)), rest = n % slots;
  return NT >= 5 && 2 * rest <= slots ? rest : 0;
}
static size_t f32_half_bytes(int Dk, long long n, int NT) {
  if (n > 0x3fffffff) return 0;
  return (size_t)(Dk == 64 ? f32_fwd_halves<4>((int)n, NT) : f32_fwd_halves<2>((int)n, NT)) * 32 * NT * 64 * sizeof(float);
}
// (a call with room for segments of seven tiles only gets those; the halves' room is the last to go)
size_t gla_f32_least_workspace(int B, int H, int L, int Dk, int Dv) {
  return (Dk != 64 && Dk != 32) || Dv != 64 || gla_f32_segments(L) == 1 ? 0 : f32_states((long long)B * H, L, gla_f32_segment_tiles(L));
}
size_t gla_f32_workspace(int B, int H, int L, int Dk, int Dv, bool bidir) {
  if ((Dk != 64 && Dk != 32) || Dv != 64 || (long long)B * H > 65535) return gla_f32_least_workspace(B, H, L, Dk, Dv);
  const int NT = gla_f32_fine_tiles((long long)B * H, L), nseg = ((L + 31) / 32 + NT - 1) / NT;
  return nseg > 1 ? f32_states((long long)B * H, L, NT) : bidir ? f32_half_bytes(Dk, (long long)B * H, NT) : 0;
}

template <int NG, bool BIDIR>
static int launch_f32_t(const GlaArgs& a, F32Geo geo) {
  constexpr int DIRS = BIDIR ? 3 : 1;
  static bool done[64] = {}, done_halves[64] = {};
  if (!allow_lds(reinterpret_cast<const void*>(gla_f32_kernel<NG, DIRS, false>), kF32MaxLds, done)) return -5;
  if constexpr (BIDIR)
    if (!allow_lds(reinterpret_cast<const void*>(gla_f32_kernel<NG, 3, true>), kF32MaxLds, done_halves)) return -5;
  const F32Lds<NG> lay(geo.NT);
  if (lay.total > kF32MaxLds || geo.NT * 8192 + 12 * 16 * NG * 4 > lay.total) return -95;
  if (geo.states) {
    hipLaunchKernelGGL((gla_f32_state_kernel<NG>), dim3(a.B * a.H, geo.nseg), dim3(BIDIR ? 256 : 128), 0, a.stream,
                       (const float*)a.k, (const float*)a.v, nullptr, nullptr, (const float*)a.g_fwd, (const float*)a.g_bwd,
                       (float*)a.workspace, (float*)nullptr, (int*)nullptr, a.L, geo.NT, geo.nseg);
    const int rc = launch_gla_segment_scan((float*)a.workspace, nullptr, a.B * a.H, geo.nseg, BIDIR ? 2 : 1, NG, a.stream);
    if (rc) return rc;
  }
  auto kernel = gla_f32_kernel<NG, DIRS, false>;
  dim3 grid(a.B * a.H, geo.nseg);
  int halves = 0;
  if constexpr (BIDIR) {
    const long long n = (long long)a.B * a.H;
    const size_t need = geo.nseg == 1 ? f32_half_bytes(16 * NG, n, geo.NT) : 0;
    if (need > 0 && a.workspace && need <= a.workspace_bytes) {
      kernel = gla_f32_kernel<NG, 3, true>;
      halves = f32_fwd_halves<NG>((int)n, geo.NT);
      geo.whole = (int)n - halves, geo.half = (float*)a.workspace;
      grid = dim3((unsigned)(n + halves));
    }
  }
  hipLaunchKernelGGL(kernel, grid, dim3(64 * geo.NT), lay.total, a.stream, (const float*)a.q, (const float*)a.k, (const float*)a.v,
                     (const float*)a.g_fwd, (const float*)a.g_bwd, (float*)a.o, geo, a.scale * a.out_scale);
  if (halves) hipLaunchKernelGGL(gla_f32_add_kernel, dim3(halves, 4), dim3(256), 0, a.stream, (float*)a.o, geo);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_gla_f32_states(int NG, const float* k, const float* v, const float* q, const float* d_o, const float* gf,
                          const float* gb, float* slots, float* grad_slots, int* flags, int nseq, int L, int NT, int nseg, hipStream_t stream) {
  // (a causal call has no reverse gates: its second direction's slots are computed with the forward ones and not read)
  const float* g2 = gb ? gb : gf;
  if (NG == 4)
    hipLaunchKernelGGL((gla_f32_state_kernel<4>), dim3(nseq, nseg, 2), dim3(256), 0, stream, k, v, q, d_o, gf, g2, slots, grad_slots, flags, L, NT,
                       nseg);
  else
    hipLaunchKernelGGL((gla_f32_state_kernel<2>), dim3(nseq, nseg, 2), dim3(256), 0, stream, k, v, q, d_o, gf, g2, slots, grad_slots, flags, L, NT,
                       nseg);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_gla_f32(const GlaArgs& a) {
  F32Geo geo{};
  geo.L = a.L;
  const long long nseq = (long long)a.B * a.H;
  geo.NT = gla_f32_fine_tiles(nseq, a.L);
  if (geo.NT * 32 < a.L && f32_states(nseq, a.L, geo.NT) > a.workspace_bytes) geo.NT = gla_f32_segment_tiles(a.L);
  geo.nseg = ((a.L + 31) / 32 + geo.NT - 1) / geo.NT;
  geo.states = geo.nseg > 1 ? (const float*)a.workspace : nullptr;
  if (a.Dk == 64) return a.g_bwd ? launch_f32_t<4, true>(a, geo) : launch_f32_t<4, false>(a, geo);
  return a.g_bwd ? launch_f32_t<2, true>(a, geo) : launch_f32_t<2, false>(a, geo);
}

}  // namespace vig
