// Backward of the bidirectional GLA op for fp32 tensors on the matrix cores (gfx950), Dk in {32, 64}, Dv = 64: one workgroup
// per sequence of up to eight 32-token tiles (longer ones as segments linked by states), wave w owns the queries and the
// keys of tile w.
//
// Per direction (forward written out; the reverse one mirrors it), with the decays of gla_f32.hip, d' = scale * d_o and
// A = d' v^T, P = q^ k^T masked to the pairs the direction keeps:
//   queries i:  acc <- D_j * acc + k^_j^T A_ij over the key tiles j <= i;                    dq_i = 2^(G-T) * acc
//   keys j:     acc <- acc + W * (q^_i^T A_ij), dv_j += d'_i^T P_ij over the query tiles i >= j, W the decays of the tiles
//               in between (k^ carries them for P);                                          dk_j = 2^(T-G) * acc
//   gates:      dg_t = sum over i >= t of q_i dq_i - k_i dk_i.
// Three loops per direction, one product pair each (A with k^ for dq, P with d' for dv, A with q^ for dk), so that what a
// loop reads of other tiles fits LDS already cut into pieces: 12 KB of v or d' and 6 KB of k^ or q^ a tile at 32 key
// channels (at 64 the latter stay fp32 rows of 8.5 KB and are cut as they are read).  The order forward dq, dv, dk, reverse
// dk, dv, dq leaves d' where it is over the turn.  At 32 key channels both directions' loops of a kind run between the same
// barriers (backward_both) where LDS has room for that.
//
// What bounds it: the matrix pipe (108 instructions of 32 clocks per tile pair and direction at Dk = 32) and, beside it, the
// cutting of the score tiles; measured figures at launch_gla_backward_f32.  The token-recurrent kernel (gla_backward.hip)
// serves the sequences that leave the tile form's range: they are flagged.
#include "f32_tiles.h"
#include <algorithm>
#include <type_traits>

namespace vig {

namespace {

constexpr float kRange32 = 40.0f;
constexpr float kMagnitude32 = 1e12f;

struct BwdF32Geo {
  int L, NT, nseg;
  float s;              // scale * out_scale
  const float *states, *grad_states;  // scanned slots of the forward states and of the gradient states; null: whole sequences
  // An item is a sequence's segment, numbered (segment, sequence); from `whole` on an item's directions go to two workgroups, the
  // reverse one leaving its dq, dk, dv in `half`: per item 32 NT rows of dq, then of dk, then of dv.
  int nseq, whole;
  float* half;
};

// byte offsets: per tile the operand over key channels (k^ or q^) and the one over value channels (v or d'), decays,
// scratch, totals of the gate gradient; carries, flags.  BOTH: key operands and tables of either direction.
template <int NG, bool BOTH = false>
struct BwdF32Lds {
  // key operand cut into pieces (6 KB a tile), as fp32 rows (8.5 KB), or as fp32 octets where the lanes want them (4 KB)
  static constexpr bool PIECES = NG == 2 && !BOTH, OCTETS = BOTH;
  static_assert(!BOTH || NG == 2, "");
  static constexpr int SK = 16 * NG + 4;   // floats between fp32 rows (16-byte aligned, rows four banks apart)
  static constexpr int KB = OCTETS ? 4096 : PIECES ? NG * 3072 : 32 * SK * 4, VB = 12288;
  int k, v, d, sc, tot, carry, flag, total;
  __host__ __device__ explicit BwdF32Lds(int NT, int dir = 0) {
    constexpr int sets = BOTH ? 2 : 1;
    k = dir * NT * KB;
    v = sets * NT * KB;
    d = v + NT * VB + dir * NT * 768;
    sc = d + NT * 256;
    tot = sc + NT * 256;
    carry = v + NT * VB + sets * NT * 768;
    flag = carry + 512;
    total = flag + 64;
  }
};

// channel of lane-row r in a fragment whose rows are key channels (part p of NG/2), so that an accumulator's register
// 4g + m of lane half h is channel 8*NG*h + n, n = row_register(p, 4g + m)
template <int NG>
__device__ __forceinline__ int key_row(int r, int p) {
  return NG == 4 ? 2 * cpair<4>(r) + p : 16 * ((r >> 2) & 1) + 8 * ((r >> 3) & 1) + 2 * (r & 3) + (r >> 4);
}
template <int NG>
constexpr int acc_part(int n) {  // which accumulator holds channel offset n of the lane half
  return NG == 4 ? (n & 1) : 0;
}
template <int NG>
constexpr int acc_reg(int n) {  // ... and in which register
  return NG == 4 ? 4 * (n >> 3) + ((n >> 1) & 3) : 4 * (2 * (n & 1) + (n >> 3)) + ((n >> 1) & 3);
}
// accumulators -> rows' octets
template <int NG>
__device__ __forceinline__ void unpack_acc(const f32x16_t (&acc)[NG / 2], f32x8_t (&x)[NG]) {
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) x[c][e] = acc[acc_part<NG>(8 * c + e)][acc_reg<NG>(8 * c + e)];
}
template <int NG>
__device__ __forceinline__ void scale_acc(f32x16_t (&acc)[NG / 2], const float* d, int h) {
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    const f32x8_t x = lds_f32x8(d + 8 * NG * h + 8 * c);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[acc_part<NG>(8 * c + e)][acc_reg<NG>(8 * c + e)] *= x[e];
  }
}

// column octet t of a tile in LDS: tokens jmap(t, h, 0..7) of one channel
__device__ __forceinline__ f32x8_t column(const float* tile, int stride, int t, int h, int ch) {
  f32x8_t x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = tile[jmap(t, h, e) * stride + ch];
  return x;
}

template <int NG>
__device__ __forceinline__ void store_rows(rsrc_t rows, int r, int h, const f32x8_t (&x)[NG]) {
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4_t y = {x[c][4 * i], x[c][4 * i + 1], x[c][4 * i + 2], x[c][4 * i + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, y), rows, (unsigned)r * (64u * NG) + 32u * NG * h + 32u * c + 16u * i, 0, 0);
    }
}

// suffix sums over the 32 lanes of each half (SUFFIX) or prefix sums, the lane's own value included
template <bool SUFFIX>
__device__ __forceinline__ float scan32(float x, int lane) {
  if (!SUFFIX) return prefix32(x);
  x += dpp_or_zero<0x101, 0xf>(x);
  x += dpp_or_zero<0x102, 0xf>(x);
  x += dpp_or_zero<0x104, 0xf>(x);
  x += dpp_or_zero<0x108, 0xf>(x);
  const float upper = __shfl(x, (lane & 32) | 16, 64);  // what the half's second row of sixteen sums to
  return (lane & 16) ? x : x + upper;
}

// T - G of the direction's gates; the tile's totals to sc, its decays to dtab.  Returns whether it is out of range.
// (rest: the gates' rows on entry)
template <int NG, bool FWD>
__device__ __forceinline__ bool gate_factors(float* sc, float* dtab, int lane, f32x8_t (&rest)[NG]) {
  constexpr int HC = 8 * NG;
  const int r = lane & 31, h = lane >> 5;
  float top = 0.f;
  wave_lds_sync();
#pragma unroll
  for (int c = 0; c < NG; ++c) {
    const f32x8_t own = rest[c] * kLog2e;
    f32x8_t p;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = prefix32(own[e]);
      top = fmaxf(top, fabsf(p[e]));
      if (r == 31) sc[HC * h + 8 * c + e] = p[e];
    }
    rest[c] = FWD ? p : p - own;
  }
  wave_lds_sync();
  const float tl = sc[lane & (16 * NG - 1)];
  const bool wide = __builtin_amdgcn_ballot_w64(!(top <= kRange32) || !(fabsf(tl) <= kRange32)) != 0;
  if (lane < 16 * NG) dtab[lane] = exp2_fast(tl);
  if (FWD) {
#pragma unroll
    for (int c = 0; c < NG; ++c) rest[c] = lds_f32x8(sc + HC * h + 8 * c) - rest[c];
  }
  return wide;
}

template <int NG>
__device__ __forceinline__ void write_rows(float* tile, int r, int h, const f32x8_t (&x)[NG]) {
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<f32x4_t*>(tile + r * BwdF32Lds<NG>::SK + 8 * NG * h + 8 * c + 4 * i) =
          f32x4_t{x[c][4 * i], x[c][4 * i + 1], x[c][4 * i + 2], x[c][4 * i + 3]};
}
// a lane's octet u of a tile
__device__ __forceinline__ void store_octet(char* tile, int u, int lane, const f32x8_t& x) {
  *reinterpret_cast<f32x4_t*>(unit_ptr(tile, 2 * u, lane)) = f32x4_t{x[0], x[1], x[2], x[3]};
  *reinterpret_cast<f32x4_t*>(unit_ptr(tile, 2 * u + 1, lane)) = f32x4_t{x[4], x[5], x[6], x[7]};
}
__device__ __forceinline__ f32x8_t load_octet(char* tile, int u, int lane) {
  const f32x4_t a = *reinterpret_cast<const f32x4_t*>(unit_ptr(tile, 2 * u, lane)), b = *reinterpret_cast<const f32x4_t*>(unit_ptr(tile, 2 * u + 1, lane));
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
// the key operand of this wave's tile for a contraction over channels (rows stay rows) ...
template <int NG, class Lay>
__device__ __forceinline__ void stage_key_rows(char* tile, int lane, const f32x8_t (&x)[NG]) {
  if (Lay::PIECES) {
#pragma unroll
    for (int c = 0; c < NG; ++c) store_p3(tile, c, lane, split8(x[c]));
  } else if (Lay::OCTETS) {
#pragma unroll
    for (int c = 0; c < NG; ++c) store_octet(tile, c, lane, x[c]);
  } else {
    write_rows<NG>(reinterpret_cast<float*>(tile), lane & 31, lane >> 5, x);
  }
}
// ... or over tokens (channels in the rows).  `rows`: where the rows are turned over: the region itself, or with OCTETS, which has no
// room for padded rows, one of the wave's that is filled afterwards.
template <int NG, class Lay>
__device__ __forceinline__ void stage_key_columns(char* tile, char* turn, int lane, const f32x8_t (&x)[NG]) {
  const int r = lane & 31, h = lane >> 5;
  float* rows = reinterpret_cast<float*>(turn);
  write_rows<NG>(rows, r, h, x);
  if (Lay::PIECES || Lay::OCTETS) {  // (the regions are this wave's until the next barrier)
    wave_lds_sync();
    f32x8_t y[NG / 2][2];
#pragma unroll
    for (int p = 0; p < NG / 2; ++p)
#pragma unroll
      for (int t = 0; t < 2; ++t) y[p][t] = column(rows, Lay::SK, t, h, key_row<NG>(r, p));
    wave_lds_sync();
#pragma unroll
    for (int p = 0; p < NG / 2; ++p)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (Lay::PIECES) store_p3(tile, 2 * p + t, lane, split8(y[p][t]));
        else store_octet(tile, 2 * p + t, lane, y[p][t]);
      }
    wave_lds_sync();
  }
}
template <int NG, class Lay>
__device__ __forceinline__ P3 key_columns(char* tile, int lane, int p, int t) {
  if (Lay::PIECES) return load_p3(tile, 2 * p + t, lane);
  if (Lay::OCTETS) return split8(load_octet(tile, 2 * p + t, lane));
  return split8(column(reinterpret_cast<const float*>(tile), Lay::SK, t, lane >> 5, key_row<NG>(lane & 31, p)));
}
template <int NG, class Lay>
__device__ __forceinline__ P3 key_rows(char* tile, int lane, int c) {
  if (Lay::PIECES) return load_p3(tile, c, lane);
  if (Lay::OCTETS) return split8(load_octet(tile, c, lane));
  return split8(lds_f32x8(reinterpret_cast<const float*>(tile) + (lane & 31) * Lay::SK + 8 * NG * (lane >> 5) + 8 * c));
}
// the value operand: v or d' rows in pieces, or turned over (fetched that way): four octets as they come from memory
__device__ __forceinline__ void stage_values(char* tile, int lane, const f32x8_t (&y)[4], float s) {
#pragma unroll
  for (int c = 0; c < 4; ++c) store_p3(tile, c, lane, split8(y[c] * s));
}
__device__ __forceinline__ void load_columns(rsrc_t rows, int r, int h, f32x8_t (&y)[4]) {  // unit 2t + pv
  f32x8_t z[2][2];
  load_pairs_f32(rows, r, h, z);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int pv = 0; pv < 2; ++pv) y[2 * t + pv] = z[pv][t];
}

__device__ __forceinline__ f32x8_t exp2_octet(f32x8_t x) {
  f32x8_t y;
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = exp2_fast(x[e]);
  return y;
}

// A^T or A tile: rows from LDS (value operand, rows), columns the wave's own rows
__device__ __forceinline__ f32x16_t value_scores(char* tile, int lane, const P3 (&own)[4]) {
  f32x16_t big = {0.f}, small = {0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) mfma6(load_p3(tile, c, lane), own[c], big, small);
  return big + small;
}
template <bool LOWER>  // keep rows <= column (LOWER) or rows >= column: register 4g + m is row 8g + 4h + m
__device__ __forceinline__ void mask_tile(f32x16_t& P, int r, int h) {
  const int rel = r - 4 * h;
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const int j = 8 * (c >> 2) + (c & 3);
    P[c] = (LOWER ? j <= rel : j >= rel) ? P[c] : 0.f;
  }
}

// queries of this wave's tile over the key tiles of one direction: dq (without the final 2^(G-T)); LDS: k^ columns, v rows
template <int NG, bool FWD, class Lay>
__device__ __forceinline__ void query_loop(const Lay& lay, char* lds, int ti, int NT, int lane, const P3 (&own)[4],
                                           const float* state, f32x16_t (&acc)[NG / 2]) {
  constexpr int NP = NG / 2;
  const int r = lane & 31, h = lane >> 5;
#pragma unroll
  for (int p = 0; p < NP; ++p) acc[p] = f32x16_t{0.f};
  if (state) {  // S_in d'^T, rows key channels
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x16_t small = {0.f};
      const int ch = key_row<NG>(r, p);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f32x8_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = state[state_index<NG>(ch, 32 * h + 8 * c + e)];
        mfma6(split8(x), own[c], acc[p], small);
      }
      acc[p] += small;
    }
  }
  const int n = FWD ? ti : NT - 1 - ti;
#pragma unroll 1
  for (int s = 0; s <= n; ++s) {
    const int j = FWD ? s : NT - 1 - s;
    scale_acc<NG>(acc, reinterpret_cast<const float*>(lds + lay.d) + 64 * j, h);
    f32x16_t A = value_scores(lds + lay.v + j * Lay::VB, lane, own);
    if (s == n) mask_tile<FWD>(A, r, h);
    const P3 a[2] = {split8(half_of<0>(A)), split8(half_of<1>(A))};
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x16_t small = {0.f};
#pragma unroll
      for (int t = 0; t < 2; ++t) mfma6(key_columns<NG, Lay>(lds + lay.k + j * Lay::KB, lane, p, t), a[t], acc[p], small);
      acc[p] += small;
    }
  }
}

// keys of this wave's tile over the query tiles of one direction, the values' gradient: dv += d'^T P; kh enters as k^;
// LDS: q^ rows, d' columns
template <int NG, bool FWD, class Lay>
__device__ __forceinline__ void value_loop(const Lay& lay, char* lds, int ti, int NT, int lane, f32x8_t (&kh)[NG],
                                           const float* dstate, float s, f32x16_t (&dv)[2]) {
  const int r = lane & 31, h = lane >> 5;
  const float* tl = reinterpret_cast<const float*>(lds + lay.sc) + 64 * ti;
  // against the own tile's queries: k 2^-G
#pragma unroll
  for (int c = 0; c < NG; ++c) kh[c] *= exp2_octet(-lds_f32x8(tl + 8 * NG * h + 8 * c));
  const int n = FWD ? NT - 1 - ti : ti;
#pragma unroll 1
  for (int x = 0; x <= n; ++x) {
    const int i = FWD ? ti + x : ti - x;
    char* qt = lds + lay.k + i * Lay::KB;
    char* dt = lds + lay.v + i * Lay::VB;
    f32x16_t P = {0.f}, small_p = {0.f};
#pragma unroll
    for (int c = 0; c < NG; ++c) mfma6(key_rows<NG, Lay>(qt, lane, c), split8(kh[c]), P, small_p);
    P += small_p;
    if (x == 0) mask_tile<!FWD>(P, r, h);
    const P3 p3[2] = {split8(half_of<0>(P)), split8(half_of<1>(P))};
#pragma unroll
    for (int pv = 0; pv < 2; ++pv) {
      f32x16_t small = {0.f};
#pragma unroll
      for (int t = 0; t < 2; ++t) mfma6(load_p3(dt, 2 * t + pv, lane), p3[t], dv[pv], small);
      dv[pv] += small;
    }
    // on to the next tile: over the one just met (the own tile: from its start to its end)
#pragma unroll
    for (int c = 0; c < NG; ++c)
      kh[c] *= lds_f32x8(reinterpret_cast<const float*>(lds + lay.d) + 64 * i + 8 * NG * h + 8 * c);
  }
  if (dstate) {  // the gradient state entering from the far side: dv += dS^T k^
#pragma unroll
    for (int pv = 0; pv < 2; ++pv) {
      f32x16_t small = {0.f};
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(dstate + ((pv * 4 + c) * 64 + lane) * 4);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(dstate + (((2 + pv) * 4 + c) * 64 + lane) * 4);
        mfma6(split8(s * __builtin_shufflevector(a, b, 0, 4, 1, 5, 2, 6, 3, 7)), split8(kh[c]), dv[pv], small);
      }
      dv[pv] += small;
    }
  }
}

// ... and the keys': dk (without the final 2^(T-G)); LDS: q^ columns, d' rows
template <int NG, bool FWD, class Lay>
__device__ __forceinline__ void key_loop(const Lay& lay, char* lds, int ti, int NT, int lane, const P3 (&own)[4],
                                         const float* dstate, float s, f32x16_t (&acc)[NG / 2]) {
  constexpr int NP = NG / 2;
  const int r = lane & 31, h = lane >> 5;
  const float* tl = reinterpret_cast<const float*>(lds + lay.sc) + 64 * ti;
  f32x8_t W[NG];  // decays since the end of the own tile; first 2^-T, the own queries' distance to it
#pragma unroll
  for (int c = 0; c < NG; ++c) W[c] = exp2_octet(-lds_f32x8(tl + 8 * NG * h + 8 * c));
#pragma unroll
  for (int p = 0; p < NP; ++p) acc[p] = f32x16_t{0.f};
  const auto add = [&](int p, const f32x16_t& tmp) {
#pragma unroll
    for (int n = 0; n < 8 * NG; ++n)
      if (acc_part<NG>(n) == p)
        acc[p][acc_reg<NG>(n)] = __builtin_fmaf(W[n >> 3][n & 7], tmp[acc_reg<NG>(n)], acc[p][acc_reg<NG>(n)]);
  };
  const int n = FWD ? NT - 1 - ti : ti;
#pragma unroll 1
  for (int x = 0; x <= n; ++x) {
    const int i = FWD ? ti + x : ti - x;
    f32x16_t A = value_scores(lds + lay.v + i * Lay::VB, lane, own);
    if (x == 0) mask_tile<!FWD>(A, r, h);
    const P3 a[2] = {split8(half_of<0>(A)), split8(half_of<1>(A))};
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x16_t tmp = {0.f}, small = {0.f};
#pragma unroll
      for (int t = 0; t < 2; ++t) mfma6(key_columns<NG, Lay>(lds + lay.k + i * Lay::KB, lane, p, t), a[t], tmp, small);
      add(p, tmp + small);
    }
#pragma unroll
    for (int c = 0; c < NG; ++c)
      W[c] *= lds_f32x8(reinterpret_cast<const float*>(lds + lay.d) + 64 * i + 8 * NG * h + 8 * c);
  }
  if (dstate) {  // dk += W (dS v^T)
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x16_t tmp = {0.f}, small = {0.f};
      const int ch = key_row<NG>(r, p);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f32x8_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = s * dstate[state_index<NG>(ch, 32 * h + 8 * c + e)];
        mfma6(split8(x), own[c], tmp, small);
      }
      add(p, tmp + small);
    }
  }
}

// per key channel sum over the value channels of S * dS (a direction's gate gradient enters a segment with it)
template <int NG>
__device__ __forceinline__ void carry_sums(const float* S, const float* dS, float s, float* out, int lane) {
#pragma unroll
  for (int pk = 0; pk < 2; ++pk)
#pragma unroll
    for (int cq = 0; cq < NG; ++cq) {
      f32x4_t x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int pv = 0; pv < 2; ++pv) {
        const int at = (((pk * 2 + pv) * 4 + cq) * 64 + lane) * 4;
        x += *reinterpret_cast<const f32x4_t*>(S + at) * *reinterpret_cast<const f32x4_t*>(dS + at);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float y = prefix32(x[m]);
        if ((lane & 31) == 31) out[8 * NG * (lane >> 5) + 8 * cq + 2 * m + pk] = s * y;
      }
    }
}

// DIRS: the directions this workgroup does, 1 forward, 2 reverse (of a bidirectional call it checks the ranges of both)
template <int NG, bool BIDIR, int DIRS>
__device__ __forceinline__ void backward_item(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                              const float* __restrict__ gf, const float* __restrict__ gb, const float* __restrict__ d_o,
                                              float* dq, float* dk, float* dv_out, float* dgf, float* dgb, int* flags_out,
                                              const BwdF32Geo geo, int seq, int seg, float* half, char* lds) {
  constexpr int DK = 16 * NG, NP = NG / 2;
  const int NT = geo.NT, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ti = w < 4 ? NT - 1 - w : w - 4;  // (the two waves of a SIMD meet NT + 1 tiles together, see gla_f32.hip)
  using Lay = BwdF32Lds<NG>;
  const Lay lay(NT);
  constexpr bool fwd_on = (DIRS & 1) != 0, rev_on = (DIRS & 2) != 0;
  const int tok = 32 * (seg * NT + ti);
  const int nvalid = __builtin_amdgcn_readfirstlane(max(0, min(32, geo.L - tok)));
  const size_t off = (size_t)seq * geo.L + tok;
  const rsrc_t rq = chunk_rsrc(q + off * DK, nvalid, 4 * DK), rk = chunk_rsrc(k + off * DK, nvalid, 4 * DK);
  const rsrc_t rv = chunk_rsrc(v + off * 64, nvalid, 256), rdo = chunk_rsrc(d_o + off * 64, nvalid, 256);
  const rsrc_t rdq = chunk_rsrc(fwd_on ? dq + off * DK : half + 32 * ti * DK, nvalid, 4 * DK);
  const rsrc_t rdk = chunk_rsrc(fwd_on ? dk + off * DK : half + 32 * (NT + ti) * DK, nvalid, 4 * DK);
  char* ktile = lds + ti * BwdF32Lds<NG>::KB;
  char* vtile = lds + lay.v + ti * BwdF32Lds<NG>::VB;
  float* sc = reinterpret_cast<float*>(lds + lay.sc) + 64 * ti;
  float* dtab = reinterpret_cast<float*>(lds + lay.d) + 64 * ti;
  float* tot = reinterpret_cast<float*>(lds + lay.tot);
  float* carry = reinterpret_cast<float*>(lds + lay.carry);
  int* flags = reinterpret_cast<int*>(lds + lay.flag);
  const size_t item = (size_t)seq * geo.nseg + seg;
  const float* st = geo.states ? geo.states + item * 2 * kGlaStateFloats : nullptr;
  const float* dst = geo.states ? geo.grad_states + item * 2 * kGlaStateFloats : nullptr;

  // Rows come from memory again for every loop that needs them (they would not fit in registers), asked for in front of
  // the barrier before their staging (168 -> 163 us against loads where they are used; asked for a whole loop ahead they
  // spilled: 181 us).
  constexpr bool KEEP = NG == 2;   // q and k stay in registers
  f32x8_t rest[NG], x[NG], xq[NG], xk[NG];  // T - G of the current direction; an operand on its way to LDS; rows of q and k
  f32x8_t nv[4], no[4];                     // value operands on their way: to LDS, and the wave's own
  P3 own[4];
  const auto set_own = [&](float s) {
#pragma unroll
    for (int c = 0; c < 4; ++c) own[c] = split8(no[c] * s);
  };
  const auto refetch = [&](bool q_too, bool k_too) {
    if (KEEP) return;
    if (q_too) load_rows_f32<NG>(rq, r, h, xq);
    if (k_too) load_rows_f32<NG>(rk, r, h, xk);
  };
  const auto decayed_keys = [&] {  // k^
#pragma unroll
    for (int c = 0; c < NG; ++c) x[c] = xk[c] * exp2_octet(rest[c]);
  };
  const auto decayed_queries = [&] {  // q^
#pragma unroll
    for (int c = 0; c < NG; ++c) x[c] = xq[c] * exp2_octet(lds_f32x8(sc + 8 * NG * h + 8 * c) - rest[c]);
  };
  const rsrc_t rgf = chunk_rsrc(gf + off * DK, nvalid, 4 * DK), rgb = chunk_rsrc(BIDIR ? gb + off * DK : gf, BIDIR ? nvalid : 0, 4 * DK);

  // ---- ranges; carries of the gate gradients into the segment ----
  // (the direction that comes first last: its factors stay)
  if (BIDIR) load_rows_f32<NG>(fwd_on ? rgb : rgf, r, h, rest);
  load_rows_f32<NG>(fwd_on ? rgf : rgb, r, h, x);
  load_rows_f32<NG>(rq, r, h, xq);
  load_rows_f32<NG>(rk, r, h, xk);
  load_rows_f32<4>(rv, r, h, nv);
  load_rows_f32<4>(rdo, r, h, no);
  float mag = 0.f;
  bool wide = false;
  if (BIDIR) wide = fwd_on ? gate_factors<NG, false>(sc, dtab, lane, rest) : gate_factors<NG, true>(sc, dtab, lane, rest);
#pragma unroll
  for (int c = 0; c < NG; ++c) rest[c] = x[c];
  wide |= fwd_on ? gate_factors<NG, true>(sc, dtab, lane, rest) : gate_factors<NG, false>(sc, dtab, lane, rest);
#pragma unroll
  for (int c = 0; c < NG; ++c) mag += sum_abs(xq[c]) + sum_abs(xk[c]);
#pragma unroll
  for (int c = 0; c < 4; ++c) mag += sum_abs(nv[c]) + sum_abs(no[c]);
  wide |= __builtin_amdgcn_ballot_w64(!(mag < kMagnitude32)) != 0;
  if (lane == 0) flags[ti] = wide;
  for (int d = w; d < 2; d += NT) {
    // forward: what lies to the right (the next segment's incoming state against the gradient state from there)
    const bool inner = st && (d == 0 ? seg + 1 < geo.nseg : seg > 0) && (d == 0 || BIDIR);
    if (inner)
      carry_sums<NG>(d == 0 ? st + 2 * kGlaStateFloats : st - kGlaStateFloats, d == 0 ? dst + kGlaStateFloats : dst, geo.s,
                     carry + 64 * d, lane);
    else
      carry[64 * d + lane] = 0.f;
  }
  if (fwd_on) {  // ---- forward direction, queries ----
    decayed_keys();
    stage_key_columns<NG, Lay>(ktile, ktile, lane, x);
    stage_values(vtile, lane, nv, 1.0f);
    set_own(geo.s);
  } else {  // ---- reverse direction, keys (as below, behind the forward one) ----
    decayed_queries();
    stage_key_columns<NG, Lay>(ktile, ktile, lane, x);
    stage_values(vtile, lane, no, geo.s);
#pragma unroll
    for (int c = 0; c < 4; ++c) own[c] = split8(nv[c]);
  }
  lds_barrier();
  const bool refused = __builtin_amdgcn_ballot_w64(lane < NT && flags[lane < NT ? lane : 0] != 0) != 0;
  if (threadIdx.x == 0 && (refused || geo.nseg == 1)) flags_out[seq] = refused;  // (both halves of an item: the same)
  if (refused) return;

  f32x16_t acc[NP], dv[2] = {f32x16_t{0.f}, f32x16_t{0.f}};
  f32x8_t z[NG];
  // a direction's gate gradient: q dq - k dk summed over the tokens behind (forward) or before (reverse)
  const auto gate_gradient = [&](auto fwd, const f32x8_t (&g)[NG], rsrc_t rdg, const float* dc) {
    constexpr bool FWD = decltype(fwd)::value;
    f32x8_t z[NG];
#pragma unroll
    for (int c = 0; c < NG; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        z[c][e] = scan32<FWD>(g[c][e], lane);
        if (r == (FWD ? 0 : 31)) tot[64 * ti + 8 * NG * h + 8 * c + e] = z[c][e];
      }
    lds_barrier();
    if (lane < 16 * NG) {  // (per channel: the tiles behind, from the far end)
      float sum = dc[lane];
      if (FWD) {
        for (int t = NT - 1; t > ti; --t) sum += tot[64 * t + lane];
      } else {
        for (int t = 0; t < ti; ++t) sum += tot[64 * t + lane];
      }
      sc[lane] = sum;
    }
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < NG; ++c) z[c] += lds_f32x8(sc + 8 * NG * h + 8 * c);
    store_rows<NG>(rdg, r, h, z);
  };
  if (fwd_on) {
    query_loop<NG, true>(lay, lds, ti, NT, lane, own, st, acc);
    load_columns(rdo, r, h, nv);
    refetch(true, true);
    {
      f32x8_t g[NG];
      unpack_acc<NG>(acc, g);
#pragma unroll
      for (int c = 0; c < NG; ++c) g[c] *= exp2_octet(-rest[c]);
      store_rows<NG>(rdq, r, h, g);  // parked (the same lanes add the reverse direction's)
#pragma unroll
      for (int c = 0; c < NG; ++c) g[c] *= xq[c];
      store_rows<NG>(chunk_rsrc(dgf + off * DK, nvalid, 4 * DK), r, h, g);
    }
    // ---- forward direction, keys ----
    lds_barrier();
    decayed_queries();
    stage_key_rows<NG, Lay>(ktile, lane, x);
    stage_values(vtile, lane, nv, geo.s);
    decayed_keys();
    lds_barrier();
    value_loop<NG, true>(lay, lds, ti, NT, lane, x, dst ? dst + kGlaStateFloats : nullptr, geo.s, dv);
    load_rows_f32<4>(rdo, r, h, nv);
    load_rows_f32<4>(rv, r, h, no);
    refetch(true, false);
    lds_barrier();
    decayed_queries();
    stage_key_columns<NG, Lay>(ktile, ktile, lane, x);
    stage_values(vtile, lane, nv, geo.s);
    set_own(1.0f);
    lds_barrier();
    const rsrc_t rdgf = chunk_rsrc(dgf + off * DK, nvalid, 4 * DK);
    key_loop<NG, true>(lay, lds, ti, NT, lane, own, dst ? dst + kGlaStateFloats : nullptr, geo.s, acc);
    load_rows_f32<NG>(rdgf, r, h, z);
    if (rev_on) load_rows_f32<NG>(rgb, r, h, x);
    refetch(BIDIR, true);
    {
      f32x8_t g[NG];
      unpack_acc<NG>(acc, g);
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        g[c] *= exp2_octet(rest[c]);
        z[c] -= xk[c] * g[c];
      }
      store_rows<NG>(rdk, r, h, g);
      gate_gradient(std::true_type{}, z, rdgf, carry);
    }
  }
  if (rev_on) {
    const rsrc_t rdgb = chunk_rsrc(dgb + off * DK, nvalid, 4 * DK);
    if (fwd_on) {
      lds_barrier();  // (the totals have been read)
      // ---- reverse direction, keys (d' rows stay) ----
#pragma unroll
      for (int c = 0; c < NG; ++c) rest[c] = x[c];
      gate_factors<NG, false>(sc, dtab, lane, rest);
      decayed_queries();
      stage_key_columns<NG, Lay>(ktile, ktile, lane, x);
      lds_barrier();
    }
    key_loop<NG, false>(lay, lds, ti, NT, lane, own, dst, geo.s, acc);
    load_columns(rdo, r, h, nv);
#pragma unroll
    for (int c = 0; c < NG; ++c) z[c] = f32x8_t{0.f};
    if (fwd_on) load_rows_f32<NG>(rdk, r, h, z);
    refetch(true, true);
    {
      f32x8_t kdk[NG];
      unpack_acc<NG>(acc, kdk);
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        kdk[c] *= exp2_octet(rest[c]);
        z[c] += kdk[c];
        kdk[c] *= xk[c];
      }
      store_rows<NG>(rdk, r, h, z);
      store_rows<NG>(rdgb, r, h, kdk);
    }
    lds_barrier();
    decayed_queries();
    stage_key_rows<NG, Lay>(ktile, lane, x);
    stage_values(vtile, lane, nv, geo.s);
    decayed_keys();
    lds_barrier();
    value_loop<NG, false>(lay, lds, ti, NT, lane, x, dst, geo.s, dv);
    load_rows_f32<4>(rv, r, h, nv);
    load_rows_f32<4>(rdo, r, h, no);
    refetch(false, true);
  }
  {
    const rsrc_t rdv = chunk_rsrc(fwd_on ? dv_out + off * 64 : half + (size_t)64 * NT * DK + 32 * ti * 64, nvalid, 256);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      u32x4_t o;
#pragma unroll
      for (int m = 0; m < 4; ++m) o[m] = __float_as_uint(dv[m & 1][2 * i + (m >> 1)]);
      __builtin_amdgcn_raw_buffer_store_b128(o, rdv, (unsigned)r * 256u + 128u * h + 16u * i, 0, 0);
    }
  }
  if (rev_on) {
    const rsrc_t rdgb = chunk_rsrc(dgb + off * DK, nvalid, 4 * DK);
    lds_barrier();
    // ---- reverse direction, queries ----
    decayed_keys();
    stage_key_columns<NG, Lay>(ktile, ktile, lane, x);
    stage_values(vtile, lane, nv, 1.0f);
    set_own(geo.s);
    lds_barrier();
    f32x8_t zq[NG];
    query_loop<NG, false>(lay, lds, ti, NT, lane, own, st ? st + kGlaStateFloats : nullptr, acc);
#pragma unroll
    for (int c = 0; c < NG; ++c) zq[c] = f32x8_t{0.f};
    if (fwd_on) load_rows_f32<NG>(rdq, r, h, zq);
    load_rows_f32<NG>(rdgb, r, h, z);
    refetch(true, false);
    f32x8_t g[NG];
    unpack_acc<NG>(acc, g);
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      g[c] *= exp2_octet(-rest[c]);
      zq[c] += g[c];
      g[c] = g[c] * xq[c] - z[c];
    }
    store_rows<NG>(rdq, r, h, zq);
    gate_gradient(std::false_type{}, g, rdgb, carry + 64);
  }
}

// Both directions of an item side by side, 32 key channels: the key operands of either fit as fp32 octets beside the value operand, so
// a wave runs a loop of one direction and the other's behind it, between the same two barriers.  Alone, a loop is over ti + 1 or
// NT - ti tiles, and most waves wait at the barrier for the one that meets all of them; together they are NT + 1 for every wave, and an
// item has 6 barriers instead of 15, stages the value operands three times instead of five and parks no dq, dk in the output.
// (The octets are cut as they are read, which costs 88 vector instructions a step.)  us, whole calls: 768 sequences of 196 tokens 240 -> 217,
// of 170 209 -> 186, of 150 184 -> 164, 240 of 196 78 -> 71.5, 48 of 1000 123 -> 116.
__device__ __forceinline__ void backward_both(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                              const float* __restrict__ gf, const float* __restrict__ gb, const float* __restrict__ d_o,
                                              float* dq, float* dk, float* dv_out, float* dgf, float* dgb, int* flags_out,
                                              const BwdF32Geo geo, int seq, int seg, char* lds) {
  constexpr int NG = 2, DK = 32;
  using Lay = BwdF32Lds<NG, true>;
  const int NT = geo.NT, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), ti = w;
  const Lay lay[2] = {Lay(NT, 0), Lay(NT, 1)};
  const int tok = 32 * (seg * NT + ti);
  const int nvalid = __builtin_amdgcn_readfirstlane(max(0, min(32, geo.L - tok)));
  const size_t off = (size_t)seq * geo.L + tok;
  const rsrc_t rv = chunk_rsrc(v + off * 64, nvalid, 256), rdo = chunk_rsrc(d_o + off * 64, nvalid, 256);
  const auto key_rsrc = [&](const float* p) { return chunk_rsrc(p + off * DK, nvalid, 4 * DK); };
  char* vtile = lds + lay[0].v + ti * Lay::VB;
  const auto ktile = [&](int d) { return lds + lay[d].k + ti * Lay::KB; };
  const auto sc = [&](int d) { return reinterpret_cast<float*>(lds + lay[d].sc) + 64 * ti; };
  const auto dtab = [&](int d) { return reinterpret_cast<float*>(lds + lay[d].d) + 64 * ti; };
  float* carry = reinterpret_cast<float*>(lds + lay[0].carry);
  int* flags = reinterpret_cast<int*>(lds + lay[0].flag);
  const size_t item = (size_t)seq * geo.nseg + seg;
  const float* st = geo.states ? geo.states + item * 2 * kGlaStateFloats : nullptr;
  const float* dst = geo.states ? geo.grad_states + item * 2 * kGlaStateFloats : nullptr;

  f32x8_t rest[2][NG], x[NG], xq[NG], xk[NG];  // T - G of either direction; an operand on its way to LDS; rows of q and k
  f32x8_t nv[4], no[4];                        // value operands on their way: to LDS, and the wave's own
  P3 own[4];
  const auto decayed_keys = [&](int d) {  // k^
#pragma unroll
    for (int c = 0; c < NG; ++c) x[c] = xk[c] * exp2_octet(rest[d][c]);
  };
  const auto decayed_queries = [&](int d) {  // q^
#pragma unroll
    for (int c = 0; c < NG; ++c) x[c] = xq[c] * exp2_octet(lds_f32x8(sc(d) + 8 * NG * h + 8 * c) - rest[d][c]);
  };

  // ---- ranges; carries of the gate gradients into the segment (as in backward_item) ----
  load_rows_f32<NG>(key_rsrc(gf), r, h, rest[0]);
  load_rows_f32<NG>(key_rsrc(gb), r, h, rest[1]);
  load_rows_f32<NG>(key_rsrc(q), r, h, xq);
  load_rows_f32<NG>(key_rsrc(k), r, h, xk);
  load_rows_f32<4>(rv, r, h, nv);
  load_rows_f32<4>(rdo, r, h, no);
  bool wide = gate_factors<NG, true>(sc(0), dtab(0), lane, rest[0]);
  wide |= gate_factors<NG, false>(sc(1), dtab(1), lane, rest[1]);
  float mag = 0.f;
#pragma unroll
  for (int c = 0; c < NG; ++c) mag += sum_abs(xq[c]) + sum_abs(xk[c]);
#pragma unroll
  for (int c = 0; c < 4; ++c) mag += sum_abs(nv[c]) + sum_abs(no[c]);
  wide |= __builtin_amdgcn_ballot_w64(!(mag < kMagnitude32)) != 0;
  if (lane == 0) flags[ti] = wide;
  for (int d = w; d < 2; d += NT) {
    if (st && (d == 0 ? seg + 1 < geo.nseg : seg > 0))
      carry_sums<NG>(d == 0 ? st + 2 * kGlaStateFloats : st - kGlaStateFloats, d == 0 ? dst + kGlaStateFloats : dst, geo.s,
                     carry + 64 * d, lane);
    else
      carry[64 * d + lane] = 0.f;
  }
  // ---- queries: k^ columns, v rows ----
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    decayed_keys(d);
    stage_key_columns<NG, Lay>(ktile(d), vtile, lane, x);
  }
  stage_values(vtile, lane, nv, 1.0f);
#pragma unroll
  for (int c = 0; c < 4; ++c) own[c] = split8(no[c] * geo.s);
  lds_barrier();
  const bool refused = __builtin_amdgcn_ballot_w64(lane < NT && flags[lane < NT ? lane : 0] != 0) != 0;
  if (threadIdx.x == 0 && (refused || geo.nseg == 1)) flags_out[seq] = refused;
  if (refused) return;

  f32x16_t acc[1], dv[2] = {f32x16_t{0.f}, f32x16_t{0.f}};
  f32x8_t g[NG], z[NG], sum[NG];
  const auto query_end = [&](int d, float* dg) {  // q dq of the direction waits in its gates' gradient
    unpack_acc<NG>(acc, g);
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      g[c] *= exp2_octet(-rest[d][c]);
      sum[c] = d ? sum[c] + g[c] : g[c];
      z[c] = g[c] * xq[c];
    }
    store_rows<NG>(key_rsrc(dg), r, h, z);
  };
  query_loop<NG, true>(lay[0], lds, ti, NT, lane, own, st, acc);
  query_end(0, dgf);
  query_loop<NG, false>(lay[1], lds, ti, NT, lane, own, st ? st + kGlaStateFloats : nullptr, acc);
  load_columns(rdo, r, h, nv);
  query_end(1, dgb);
  store_rows<NG>(key_rsrc(dq), r, h, sum);
  lds_barrier();
  // ---- values: q^ rows, d' columns ----
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    decayed_queries(d);
    stage_key_rows<NG, Lay>(ktile(d), lane, x);
  }
  stage_values(vtile, lane, nv, geo.s);
  lds_barrier();
  decayed_keys(0);
  value_loop<NG, true>(lay[0], lds, ti, NT, lane, x, dst ? dst + kGlaStateFloats : nullptr, geo.s, dv);
  decayed_keys(1);
  value_loop<NG, false>(lay[1], lds, ti, NT, lane, x, dst, geo.s, dv);
  load_rows_f32<4>(rdo, r, h, nv);
  load_rows_f32<4>(rv, r, h, no);
  const rsrc_t rdv = chunk_rsrc(dv_out + off * 64, nvalid, 256);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u32x4_t o;
#pragma unroll
    for (int m = 0; m < 4; ++m) o[m] = __float_as_uint(dv[m & 1][2 * i + (m >> 1)]);
    __builtin_amdgcn_raw_buffer_store_b128(o, rdv, (unsigned)r * 256u + 128u * h + 16u * i, 0, 0);
  }
  lds_barrier();
  // ---- keys: q^ columns, d' rows ----
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    decayed_queries(d);
    stage_key_columns<NG, Lay>(ktile(d), vtile, lane, x);
  }
  stage_values(vtile, lane, nv, geo.s);
#pragma unroll
  for (int c = 0; c < 4; ++c) own[c] = split8(no[c]);
  lds_barrier();
  // a direction's gate gradient: q dq - k dk summed over the tokens behind (forward) or before (reverse); here those of the tile
  f32x8_t zf[NG];
  const auto key_end = [&](auto fwd) {
    constexpr bool FWD = decltype(fwd)::value;
    constexpr int d = FWD ? 0 : 1;
    unpack_acc<NG>(acc, g);
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      g[c] *= exp2_octet(rest[d][c]);
      sum[c] = FWD ? g[c] : sum[c] + g[c];
      z[c] -= xk[c] * g[c];
    }
    float* tot = reinterpret_cast<float*>(lds + lay[d].tot) + 64 * ti;
#pragma unroll
    for (int c = 0; c < NG; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        z[c][e] = scan32<FWD>(z[c][e], lane);
        if (r == (FWD ? 0 : 31)) tot[8 * NG * h + 8 * c + e] = z[c][e];
      }
  };
  key_loop<NG, true>(lay[0], lds, ti, NT, lane, own, dst ? dst + kGlaStateFloats : nullptr, geo.s, acc);
  load_rows_f32<NG>(key_rsrc(dgf), r, h, z);
  key_end(std::true_type{});
#pragma unroll
  for (int c = 0; c < NG; ++c) zf[c] = z[c];
  key_loop<NG, false>(lay[1], lds, ti, NT, lane, own, dst, geo.s, acc);
  load_rows_f32<NG>(key_rsrc(dgb), r, h, z);
  key_end(std::false_type{});
  store_rows<NG>(key_rsrc(dk), r, h, sum);
  lds_barrier();
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const float* tot = reinterpret_cast<const float*>(lds + lay[d].tot);
    if (lane < DK) {  // (per channel: the tiles behind, from the far end, or before)
      float y = carry[64 * d + lane];
      if (d == 0) {
        for (int t = NT - 1; t > ti; --t) y += tot[64 * t + lane];
      } else {
        for (int t = 0; t < ti; ++t) y += tot[64 * t + lane];
      }
      sc(d)[lane] = y;
    }
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < NG; ++c) g[c] = (d == 0 ? zf[c] : z[c]) + lds_f32x8(sc(d) + 8 * NG * h + 8 * c);
    store_rows<NG>(key_rsrc(d == 0 ? dgf : dgb), r, h, g);
  }
}

}  // namespace

template <int NG, bool BIDIR, bool HALVES, bool BOTH>
__global__ __launch_bounds__(512, 2) void gla_backward_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ gf,
    const float* __restrict__ gb, const float* __restrict__ d_o, float* dq, float* dk, float* dv, float* dgf, float* dgb,
    int* flags, BwdF32Geo geo) {
  extern __shared__ __align__(16) char lds[];
  if constexpr (!HALVES && BOTH) {
    backward_both(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, blockIdx.x, blockIdx.y, lds);
  } else if constexpr (!HALVES) {  // (a kernel of its own: the three bodies in one cost the whole items 2 % at 64 channels)
    backward_item<NG, BIDIR, BIDIR ? 3 : 1>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, blockIdx.x, blockIdx.y, nullptr, lds);
  } else {
    const int which = (int)blockIdx.x - geo.whole, work = which < 0 ? blockIdx.x : geo.whole + (which >> 1);
    const int seg = work / geo.nseq, seq = work - seg * geo.nseq;
    float* half = geo.half + (size_t)max(which >> 1, 0) * (32 * geo.NT) * (32 * NG + 64);
    if (which < 0) {
      if constexpr (BOTH) backward_both(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, seq, seg, lds);
      else backward_item<NG, true, 3>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, seq, seg, half, lds);
    } else if ((which & 1) == 0) backward_item<NG, true, 1>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, seq, seg, half, lds);
    else backward_item<NG, true, 2>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, geo, seq, seg, half, lds);
  }
}

// What the reverse workgroups of items in two halves left is added to the forward ones' (a workgroup: a quarter of an item).
template <int DK>
__global__ __launch_bounds__(256) void gla_backward_f32_add_kernel(float* __restrict__ dq, float* __restrict__ dk, float* __restrict__ dv,
                                                                   BwdF32Geo geo) {
  const int work = geo.whole + blockIdx.x, seg = work / geo.nseq, seq = work - seg * geo.nseq, rows = 32 * geo.NT;
  const int first = seg * rows, valid = min(rows, geo.L - first);
  const float* half = geo.half + (size_t)blockIdx.x * rows * (2 * DK + 64);
  const size_t at = (size_t)seq * geo.L + first;
  const auto add = [&](float* to, const float* from, int width) {
    for (int i = (blockIdx.y * 256 + threadIdx.x) * 4; i < valid * width; i += 4096)
      *reinterpret_cast<f32x4_t*>(to + i) += *reinterpret_cast<const f32x4_t*>(from + i);
  };
  add(dq + at * DK, half, DK);
  add(dk + at * DK, half + rows * DK, DK);
  add(dv + at * 64, half + 2 * rows * DK, 64);
}

// Measured at B 64, H 6, L 196, Dk 32 (384 sequences, one to a CU; the last 128 in two halves): 126 us, a direction after the other 134, token-recurrent kernel 485 us.
// Of a wave's time a third is waiting: at the barriers, and for rows read with a lane per row (67 clocks of the CU's load path per
// 16-byte load instruction); matrix and vector pipe take a quarter and a third of the kernel's.
constexpr int kBwdF32MaxLds = 160 * 1024;

// Segments of up to seven tiles, as in the forward (eight would not fit beside 64 key channels).  A causal call of 225 to
// 256 tokens has no room for two segments' states in the workspace its size promises: the recurrent kernel keeps it.  It also
// keeps sequences of one of its token blocks at 64 key channels while they fill the chip no more than three times over (tile
// form / recurrent kernel, us: 6 sequences of 8 tokens 37.9 / 27.0, of 16 38.9 / 32.0, of 17 38.9 / 54.3; 768 of 16
// 57.4 / 50.4, of 17 58.4 / 83.7; 1536 of 8 67 / 77, of 16 77 / 99; one direction alike; 32 channels 23 / 26 at least).
bool gla_backward_f32_supported(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir) {
  if (Dk == 64 && L <= 16 && (long long)B * H <= 768) return false;
  return io_dtype == 0 && gate_dtype == 0 && (Dk == 64 || Dk == 32) && Dv == 64 && gla_f32_segments(L) <= 65535 &&
         (gla_f32_segments(L) == 1 || (long long)B * H * 4 <= 65535) && (bidir || L <= 224 || L > 256);
}
// Items whose directions go to two workgroups: what is left over of full rounds of the chip, where that fills no more than half of
// one.  A half takes 55 to 60 % of the whole (it loads and checks the same), and adding up takes 3 us.  us, whole / halves: Dk 32: 18
// sequences of 64 32 / 22.5, of 185 63.5 / 43.0, 120 of 196 74 / 55, 384 (256 and 128) 150 / 133 (before both directions of the whole ones ran side by side: 126); Dk 64: 18 of 64 56 / 34.5, 60 of 196 136
// / 88, 384 292 / 251.
template <int NG>
static int f32_halves(int n, int NT) {
  const int slots = 256 * std::max(1, std::min(kBwdF32MaxLds / BwdF32Lds<NG>(NT).total, 8 / NT)), rest = n % slots;
  return 2 * rest <= slots ? rest : 0;
}
// Both directions side by side (32 key channels) where that leaves a CU as many workgroups: three tiles and five to seven.  us, one after the
// other / side by side: 768 sequences of 120 tokens 115 / 152, 480 of 100 64 / 79, 1536 of 49 92 / 96; 768 of 90 93 / 90, of 150 184 / 164.
static bool f32_both(int NT) {
  const auto slots = [NT](int lds) { return std::min(kBwdF32MaxLds / lds, 8 / NT); };
  return slots(BwdF32Lds<2, true>(NT).total) == slots(BwdF32Lds<2>(NT).total);
}
template <int NG>
static size_t half_floats(int NT) { return (size_t)32 * NT * (32 * NG + 64); }

// what the halves of a long sequence's items want beside the states (those of whole sequences lie in the recurrent kernel's scratch)
size_t gla_backward_f32_extra(int B, int H, int L, int Dk, int Dv) {
  if ((Dk != 64 && Dk != 32) || Dv != 64 || L <= 256 || (long long)B * H * 4 > 65535) return 0;
  const int NT = gla_f32_fine_tiles((long long)B * H, L), n = B * H * (((L + 31) / 32 + NT - 1) / NT);
  return Dk == 64 ? f32_halves<4>(n, NT) * half_floats<4>(NT) * sizeof(float) : f32_halves<2>(n, NT) * half_floats<2>(NT) * sizeof(float);
}

template <int NG, bool BIDIR>
static int launch_bwd_f32_t(const float* q, const float* k, const float* v, const float* gf, const float* gb, const float* d_o,
                            float* dq, float* dk, float* dv, float* dgf, float* dgb, int* flags, void* room0, size_t bytes0,
                            void* room1, size_t bytes1, void* room2, size_t bytes2, int B, int H, int L, float s, hipStream_t stream) {
  static bool done[4][64] = {};
  BwdF32Geo geo{};
  geo.L = L;
  const int tiles = (L + 31) / 32;
  float *states = nullptr, *grads = nullptr;
  // the segments that fill the chip, or the next longer ones whose states have room
  const int most = gla_f32_segment_tiles(L);
  for (int NT = gla_f32_fine_tiles((long long)B * H, L); NT <= most; ++NT) {
    geo.NT = NT, geo.nseg = (tiles + NT - 1) / NT;
    const size_t set = geo.nseg == 1 ? 0 : (size_t)B * H * geo.nseg * 2 * kGlaStateFloats;
    const size_t n = set * sizeof(float);
    if (2 * n <= bytes0) states = (float*)room0, grads = states + set;
    else if (2 * n <= bytes1) states = (float*)room1, grads = states + set;
    else if (n <= bytes0 && n <= bytes1) states = (float*)room0, grads = (float*)room1;
    else continue;
    break;
  }
  if (!states) return -28;
  geo.s = s;
  int lds = BwdF32Lds<NG>(geo.NT).total;
  if (lds > kBwdF32MaxLds || geo.NT > 7) return -95;
  if (geo.nseg > 1) {
    geo.states = states, geo.grad_states = grads;
    int rc = launch_gla_f32_states(NG, k, v, q, d_o, gf, gb, states, grads, flags, B * H, L, geo.NT, geo.nseg, stream);
    if (rc) return rc;
    rc = launch_gla_segment_scan(states, grads, B * H, geo.nseg, 2, NG, stream);
    if (rc) return rc;
  }
  const int n = B * H * geo.nseg;
  geo.nseq = B * H, geo.whole = n;
  if (BIDIR) {
    const int rest = f32_halves<NG>(n, geo.NT);
    const size_t need = (size_t)rest * half_floats<NG>(geo.NT) * sizeof(float);
    const size_t used = geo.nseg == 1 ? 0 : (size_t)n * 2 * kGlaStateFloats * sizeof(float);  // of a room, by a set of states
    const size_t used0 = states == room0 && geo.nseg > 1 ? (grads == room1 ? used : 2 * used) : 0;
    const size_t used1 = geo.nseg > 1 ? (states == room1 ? 2 * used : grads == room1 ? used : 0) : 0;
    if (rest > 0) {
      if (used0 + need <= bytes0) geo.half = (float*)((char*)room0 + used0), geo.whole = n - rest;
      else if (used1 + need <= bytes1) geo.half = (float*)((char*)room1 + used1), geo.whole = n - rest;
      else if (need <= bytes2) geo.half = (float*)room2, geo.whole = n - rest;
    }
  }
  const bool halves = geo.whole < n;
  bool both = false;
  auto kernel = gla_backward_f32_kernel<NG, BIDIR, false, false>;
  dim3 grid(B * H, geo.nseg);
  if (halves) grid = dim3(2 * n - geo.whole);
  if constexpr (BIDIR) {
    if (halves) kernel = gla_backward_f32_kernel<NG, true, true, false>;
    if constexpr (NG == 2) {
      both = f32_both(geo.NT);
      if (both) kernel = halves ? gla_backward_f32_kernel<NG, true, true, true> : gla_backward_f32_kernel<NG, true, false, true>;
      if (both) lds = std::max(lds, BwdF32Lds<2, true>(geo.NT).total);
    }
  }
  if (!allow_lds(reinterpret_cast<const void*>(kernel), kBwdF32MaxLds, done[2 * both + halves])) return -5;
  hipLaunchKernelGGL(kernel, grid, dim3(64 * geo.NT), lds, stream, q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags,
                     geo);
  if (geo.whole < n) hipLaunchKernelGGL((gla_backward_f32_add_kernel<16 * NG>), dim3(n - geo.whole, 4), dim3(256), 0, stream, dq, dk, dv, geo);
  return hipGetLastError() == hipSuccess ? 0 : -5;
}

int launch_gla_backward_f32(const void* q, const void* k, const void* v, const void* gf, const void* gb, const void* d_o,
                            void* dq, void* dk, void* dv, void* dgf, void* dgb, int* flags, void* room0, size_t bytes0,
                            void* room1, size_t bytes1, void* room2, size_t bytes2, int B, int H, int L, int Dk, float s,
                            hipStream_t stream) {
#define VIG_BWD_F32(NG, BI)                                                                                                   \
  launch_bwd_f32_t<NG, BI>((const float*)q, (const float*)k, (const float*)v, (const float*)gf, (const float*)gb,             \
                           (const float*)d_o, (float*)dq, (float*)dk, (float*)dv, (float*)dgf, (float*)dgb, flags, room0, bytes0, room1, bytes1, \
                           room2, bytes2, B, H, L, s, stream)
  if (Dk == 64) return gb ? VIG_BWD_F32(4, true) : VIG_BWD_F32(4, false);
  return gb ? VIG_BWD_F32(2, true) : VIG_BWD_F32(2, false);
#undef VIG_BWD_F32
}

}  // namespace vig
