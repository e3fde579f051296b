// Backward of the bidirectional GLA op on MFMA tiles (gfx950): bf16 tensors and gates, Dk in {32, 64}, Dv = 64.
// L <= 256 is one slab per (batch, head); a longer sequence is cut into segments (<= 256 tokens), each
// handled like a slab plus three products with the states that link it to the other segments (see SEG below).
//
// Per direction the whole (batch, head) slab is one quadratic form (no chunk states): with G the inclusive
// cumulative log-gate along the direction and the anchor a = G_total / 2,
//   q~_i = q_i e^{G_i - a},  k~_j = k_j e^{a - G_j}   (both within e^{|G_total|/2} of the inputs),
//   P_ij = q~_i . k~_j,  A_ij = do_i . v_j            for the pairs the direction keeps (j <= i forward, j >= i reverse),
//   dv_j = s sum_i P_ij do_i,   dq_i = s e^{G_i - a} (.) sum_j A_ij k~_j,   dk_j = s e^{a - G_j} (.) sum_i A_ij q~_i,
//   dg_t = sum over the tokens i the gate of t acts on (i >= t forward, i <= t reverse) of q_i (.) dq_i - k_i (.) dk_i,
// s = scale * out_scale.  This is the natural-order form of flash-linear-attention/fla/ops/gla/chunk_fuse.py:413-518
// with one chunk per sequence; the flip-concat glue of classification/models/vig.py:407-426 never materialises.
//
// One persistent workgroup of 8 or 7 waves per CU (for short slabs two of 4 or, at Dk 64, 3, four of 2) walks slabs; wave w owns the 32-token
// tile w.
// Per direction the workgroup stages q~, k~ (and once v, do) as bf16 rows in LDS; then wave w accumulates dk, dv of its tile over
// the query tiles the direction keeps, and dq over the key tiles: score tiles P, A come out of the matrix cores in the
// register layout that feeds the next product directly (mfma_tiles.h), operands with tokens in the contraction slots are
// transposed by the LDS reads themselves.  The two directions take turns in LDS; a tile that is heavy in one direction is
// light in the other, so over both every wave does the same amount of work.  dg needs a running sum over tokens: inside the
// tile the lanes (= tokens) add up q dq - k dk by lane shifts, the tile totals are exchanged through LDS.  What the next
// direction (or slab) reads is fetched before this one's results are stored, and its cumulative gates and their tile
// totals are prepared before the second barrier.
// Two barriers per direction: staged q~ / k~, and the totals of q dq - k dk together with the next direction's gate
// totals; the second also tells that nobody reads this direction's staged rows any more.
//
// What bounds it (768 slabs of 196 tokens, Dk = 64): a slab's loads and stores come in bursts that all CUs make at the same time (a token
// asks for 1664 bytes, q and k in either direction, 49 us at the rate of a large copy; 1864 pass the memory, what fifteen spilled registers write
// among them), and its products wait for LDS reads with two waves a SIMD.  us, whole calls one behind the other, the flag pass with them, against operands read as dwords and
// put together by v_perm, dq ahead of dk, dv in loops of their own and the first direction's dq, dk parked in the output tensors:
// 768 x 196 Dk 64 103 to 105 -> 86 to 90, Dk 32 74 to 76 -> 57 to 60; 768 x 256 Dk 64 124 to 129 -> 106 to 112; 1200 x 128 84 -> 71; 24 x 2305 with the state passes, Dk 32 57 -> 47.5,
// Dk 64 82 -> 73; 384 x 57 Dk 64 23.4 -> 22.9, 600 x 64 27.0 -> 27.2, 1200 x 64 42.4 -> 39.7, 768 x 49
// 26.7 -> 26.4, forward alone 18.0 -> 18.4.
//
// Slabs whose gate totals exceed the anchor's range (|G_total| / 2 * log2(e) > 60 in some channel) are not computed
// here: the workgroup raises the slab's flag and the token-recurrent kernel, launched afterwards with that flag
// array, computes exactly those.
#include "common.h"
#include "launch.h"
#include "mfma_tiles.h"

namespace vig {

namespace {

constexpr int kBwdTiles = 8;  // most 32-token tiles per slab
// Staged rows are 128 bytes and lie without gaps; the 16-byte piece c of row i is found at place c ^ (i & 7), so that eight rows'
// pieces c cover every bank (rows padded to 144 bytes do too, but leave no room for `turn`).
constexpr int kRow = 64;
__device__ __forceinline__ int row_piece(int row, int c) { return row * kRow + ((c ^ (row & 7)) << 3); }
// LDS of a workgroup of TW tiles, one wave each
template <int TW>
struct BwdLds {
  static constexpr int mat = TW * 32 * kRow * 2;  // one staged (32 TW) x 64 bf16 matrix
  static constexpr int q = 0, d_o = mat, k = 2 * mat, v = 3 * mat;  // (those read together within a 16-bit offset)
  static constexpr int tot = 4 * mat;               // [TW][64] f32: gate totals of the tiles
  static constexpr int off = tot + TW * 64 * 4;     // [TW][64] f32: per wave, (prefix - anchor) of its tile
  static constexpr int dgtot = off + TW * 64 * 4;   // [TW][64] f32: totals of q dq - k dk of the tiles
  // [TW][parked units of 64 lanes x 16 B]: the first direction's dq (Dk = 64) while the second runs, where there is room for it.  Two tiles:
  // three of its four units, which leave four workgroups to a CU; the last one goes by way of the output tensor.  us, all four that
  // way / one / none, with three workgroups: 600 slabs of 64 tokens 27.6 / 26.9 / 26.8, 768 29.4 / 28.9 / 28.6, 1024 34.5 / 33.7 / 40.4; one 15.0 / 15.1 / 15.0.
  static constexpr int parked = TW == 7 || TW == 3 ? 4 : TW == 2 ? 3 : 0;
  static constexpr int park = dgtot + TW * 64 * 4;
  static constexpr int turn = park + TW * parked * 1024;  // [TW][16 rows] of results on their way out (store_rows)
  static constexpr bool turns(int ng) { return ng == 4 && TW >= 3; }
  static constexpr int total = turn + (turns(4) ? TW * 16 * kRow * 2 : 0);
};
constexpr float kBwdHalfRange = 60.0f;


// A lane's row of a staged matrix, as operand fragments of 8 consecutive channels (k-step ks, lane half h): piece 2 ks + h.
// The addresses stay in registers: what is read around them goes by instruction offsets.
struct RowPtr {
  lds_u16_t p[4];
  __device__ __forceinline__ RowPtr(lds_u16_t mat, int row, int h) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      p[ks] = mat + row_piece(row, 2 * ks + h);
      asm volatile("" : "+v"(p[ks]));
    }
  }
  __device__ __forceinline__ u32x4_t frag(int ks, int off = 0) const {
    typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4_t;
    return *(lds_u32x4_t*)(p[ks] + off);
  }
  __device__ __forceinline__ void advance(int by) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) p[ks] += by;
  }
};
// A lane's address for transposed fragments (tr_frag) of the tile at `mat`: its piece holds one of 16 NG / 4 groups of four channels
template <int NG>
__device__ __forceinline__ lds_u16_t tr_ptr(lds_u16_t mat, int lane) {
  const int row = 4 * (lane >> 5) + ((lane & 15) >> 2), ch = tr_row_channel<NG>(16 * ((lane >> 4) & 1) + 4 * (lane & 3));
  lds_u16_t at = mat + row_piece(row, ch >> 3) + (ch & 7);
  asm volatile("" : "+v"(at));
  return at;
}
// the NG pieces of a lane's half row
template <int NG>
__device__ __forceinline__ void store_row(uint16_t* mat, int row, int h, const u32x4_t (&x)[NG]) {
#pragma unroll
  for (int g = 0; g < NG; ++g) *reinterpret_cast<u32x4_t*>(mat + row_piece(row, NG * h + g)) = x[g];
}
__device__ __forceinline__ u32x4_t load_piece(const uint16_t* mat, int row, int c) {
  return *reinterpret_cast<const u32x4_t*>(mat + row_piece(row, c));
}

// accumulator tile (rows 8g+4h+m in registers, column = lane) -> operand fragments with its rows in the contraction
// slots, k-steps t = 0, 1
__device__ __forceinline__ void tile_frags(const f32x16_t& T, u32x4_t (&f)[2]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int x = 0; x < 4; ++x) f[t][x] = pack_bf16x2(T[8 * t + 2 * x], T[8 * t + 2 * x + 1]);
}

// keeps the entries of a diagonal tile the direction uses, in its operand fragments; ROWS_ARE_QUERIES: rows i, column j (else rows j,
// column i).  (On the packed values: a branch between the matrix instructions and the first vector read of their result
// left that read without its wait states in one build of this kernel.)
template <bool FWD, bool ROWS_ARE_QUERIES>
__device__ __forceinline__ void mask_diag(u32x4_t (&f)[2], int r, int h) {
  const uint32_t kept = (FWD == ROWS_ARE_QUERIES ? ~0u << r : ~0u >> (31 - r)) >> (4 * h);  // rows r .. 31, or 0 .. r
  f[0] &= keep_masks<0>(kept), f[1] &= keep_masks<1>(kept);
}

// accumulators of a tile's k channels and where channel c8 of octet gq lies in them (tr_row_channel)
template <int NG>
struct KeyAcc {
  f32x16_t a[NG / 2];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int p = 0; p < NG / 2; ++p) a[p] = f32x16_t{0.f};
  }
  __device__ __forceinline__ float get(int gq, int c8) const { return NG == 4 ? a[c8 >> 2][4 * gq + (c8 & 3)] : a[0][8 * gq + c8]; }
};

// dq^ of tile w += the key tile at `v` (rows) and `k` (transposed): A^T = v do^T, rows j, columns i
template <bool FWD, int NG>
__device__ __forceinline__ void add_dq(bool diag, const RowPtr& v, lds_u16_t k, const u32x4_t (&doB)[4], int r, int h, KeyAcc<NG>& dq) {
  f32x16_t T = {0.f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) T = mfma(v.frag(ks), doB[ks], T);
  u32x4_t f[2];
  tile_frags(T, f);
  if (diag) mask_diag<FWD, false>(f, r, h);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int p = 0; p < NG / 2; ++p) dq.a[p] = mfma(tr_frag<kRow>(k + 4 * p, t), f[t], dq.a[p]);
}

// dv, dk^ of tile w += the query tile at `q` (rows; do's lie `to_do` further), `qt` and `dt` (transposed): P = q~ k~^T,
// A = do v^T, rows i, columns j
template <bool FWD, int NG>
__device__ __forceinline__ void add_dv_dk(bool diag, const RowPtr& q, int to_do, lds_u16_t qt, lds_u16_t dt, const u32x4_t (&kB)[NG],
                                          const u32x4_t (&vB)[4], int r, int h, f32x16_t (&dv)[2], KeyAcc<NG>& dk) {
  f32x16_t P = {0.f}, A = {0.f};
#pragma unroll
  for (int ks = 0; ks < NG; ++ks) P = mfma(q.frag(ks), kB[ks], P);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) A = mfma(q.frag(ks, to_do), vB[ks], A);
  u32x4_t f[2];
  tile_frags(P, f);
  if (diag) mask_diag<FWD, true>(f, r, h);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int p = 0; p < 2; ++p) dv[p] = mfma(tr_frag<kRow>(dt + 4 * p, t), f[t], dv[p]);
  tile_frags(A, f);
  if (diag) mask_diag<FWD, true>(f, r, h);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int p = 0; p < NG / 2; ++p) dk.a[p] = mfma(tr_frag<kRow>(qt + 4 * p, t), f[t], dk.a[p]);
}

// The lane id, counted where it is asked for, in a copy that the compiler does not connect with the others: what is derived from it (rows,
// offsets) does not stay in registers across the phases between, and neither does the id.  Kept, it was spilled, and reloaded behind the stores
// that end a direction: the counter a load is waited for with goes down in the order of issue, so the wave waited for all it had just
// stored.  (With tile_rows, us: 768 slabs of 49 tokens, Dk 64 27.4 -> 25.8, of 65 37.3 -> 36.1, of 128 51.5 -> 47.2; one of 128 20.0 -> 19.2.)
__device__ __forceinline__ int fresh_lane() {
  uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
  asm volatile("" : "+v"(lane));
  return (int)lane;
}

// Valid tokens of tile w of a slab of L, by scalar instructions: a two-sided clamp becomes one vector instruction, whose result was kept from
// slab to slab, spilled and reloaded like the lane id.
__device__ __forceinline__ int tile_rows(int L, int w) {
  int n = max(L - 32 * w, 0);
  asm volatile("" : "+s"(n));
  return min(n, 32);
}

// Inclusive running sums over the 32 tokens of a lane half (lanes 32h .. 32h + 31, in lane order) for N values at
// once: four shifted adds inside the rows of 16 lanes (lanes shifted in from outside a row read zero), then lane 15 of
// the lower row added to every lane of the upper one.  Step by step over all values, so that consecutive lane-shift
// instructions never wait for each other's results.
template <int CTRL>
__device__ __forceinline__ float row_shifted(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL, int N>
__device__ __forceinline__ void add_row_shifted(float (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] += row_shifted<CTRL>(x[i]);
  __builtin_amdgcn_sched_barrier(0);
}
template <int N>
__device__ __forceinline__ void half_prefix_sums(float (&x)[N]) {
  __builtin_amdgcn_sched_barrier(0);
  add_row_shifted<0x111>(x);  // row_shr:1
  add_row_shifted<0x112>(x);  // row_shr:2
  add_row_shifted<0x114>(x);  // row_shr:4
  add_row_shifted<0x118>(x);  // row_shr:8
#pragma unroll
  for (int i = 0; i < N; ++i)  // row_bcast:15 into rows 1 and 3 (row mask 0b1010); rows 0 and 2 keep the zero
    x[i] += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x[i]), 0x142, 0xa, 0xf, false));
}

// the running sum of the token before (lane - 1), nothing for the first of the half
__device__ __forceinline__ float before_lane(float x, int r) {
  const float y = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true));  // wave_shr:1
  return r == 0 ? 0.f : y;
}

// A wave's 32 result rows of 16 NG bf16 channels (lane: the NG 16-byte pieces of its half row).  At Dk = 64 16 rows at a time go
// by way of `turn`, so that a store instruction writes one contiguous KB instead of 64 pieces of 16 bytes in as many 64-byte
// blocks: 768 slabs of 196 tokens 96.1 -> 90.6 us, 1200 of 128 83.5 -> 77.  Dk = 32 gains nothing by it (58.5, 59.1) and slabs of one
// or two tiles lose the latency (25.3 against 24.0).
template <int NG, int TW, bool PITCHED = false>
__device__ __forceinline__ void store_rows(uint16_t* turn, const u32x4_t (&x)[NG], rsrc_t out, int lane, unsigned pitch = 32u * NG) {
  const int r = lane & 31, h = lane >> 5;
  if constexpr (!BwdLds<TW>::turns(NG)) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
      __builtin_amdgcn_raw_buffer_store_b128(x[g], out, r * (PITCHED ? pitch : 32u * NG) + h * (16u * NG) + 16u * g, 0, 0);
  } else {
    lane = fresh_lane();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      wave_lds_sync();
      if ((r >> 4) == half) store_row<NG>(turn, r & 15, h, x);
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < NG / 2; ++j) {
        const int piece = 64 * j + lane;
        const int row = piece / (2 * NG), at = piece % (2 * NG);
        const unsigned to = PITCHED ? (16u * half + row) * pitch + 16u * at : 512u * NG * half + 16u * piece;
        __builtin_amdgcn_raw_buffer_store_b128(load_piece(turn, row, at), out, to, 0, 0);
      }
    }
  }
}

struct BwdSlab {
  const uint16_t *q, *k, *v, *gf, *gb, *d_o;
  uint16_t *dq, *dk, *dv, *dgf, *dgb;
  // segments of a long sequence only (direction 1 follows direction 0 in each array):
  const uint16_t *sp, *rp, *rpt;  // sqrt(D) S_in as [k channel][v], sqrt(D) R_out as [k channel][v] and as [v][k channel]
  const float* carry;             // [2 directions][2 partial sums][64]: q dq - k dk summed over the segments walked later
  int L;                          // tokens of this slab / segment
  // PITCHED: a token's q, k and v lie in one row of a matrix, their gradients in one of another; bytes from row to row
  unsigned in, out;
};

// What a wave loads for one direction of one slab (its own 32-token tile), issued one phase ahead.
template <int NG>
struct BwdLoads {
  uint32_t gD[2][8];             // gate dwords (tokens in the contraction slots)
  u32x4_t rawq[NG], rawk[NG];    // q and k rows
  u32x4_t rawv[4], rawd[4];      // v and do rows (first direction of a slab only)
};
struct BwdNext {  // the direction whose loads are issued while this one finishes
  BwdSlab sl;
  const uint16_t* g;
  int L;  // 0: nothing follows (empty descriptors, no memory traffic)
};
template <int NG>
__device__ __forceinline__ void issue_bwd_gate_loads(const BwdNext& n, int w, int r, int h, BwdLoads<NG>& ld) {
  constexpr int DK = 16 * NG;
  const int rows = tile_rows(n.L, w);
  issue_tdwords<0, 2, NG>(chunk_rsrc(n.g + (size_t)32 * w * DK, rows, 2 * DK), r, h, ld.gD);
}
template <int NG, bool PITCHED>
__device__ __forceinline__ void issue_bwd_qk_loads(const BwdNext& n, int w, int r, int h, BwdLoads<NG>& ld) {
  constexpr int DK = 16 * NG;
  const int rows = tile_rows(n.L, w);
  if constexpr (PITCHED) {
    const size_t t = (size_t)(16 * w) * n.sl.in;
    issue_raw_tile_pitched<NG>(chunk_rsrc(n.sl.q + t, rows, n.sl.in), 0, r, h, n.sl.in, ld.rawq);
    issue_raw_tile_pitched<NG>(chunk_rsrc(n.sl.k + t, rows, n.sl.in), 0, r, h, n.sl.in, ld.rawk);
    return;
  }
  const size_t tk = (size_t)32 * w * DK;
  issue_raw_tile<NG>(chunk_rsrc(n.sl.q + tk, rows, 2 * DK), 0, r, h, ld.rawq);
  issue_raw_tile<NG>(chunk_rsrc(n.sl.k + tk, rows, 2 * DK), 0, r, h, ld.rawk);
}
template <int NG, bool PITCHED>
__device__ __forceinline__ void issue_bwd_vdo_loads(const BwdNext& n, int w, int r, int h, BwdLoads<NG>& ld) {
  const int rows = tile_rows(n.L, w);
  const size_t tv = (size_t)32 * w * 64;
  if constexpr (PITCHED) issue_raw_tile_pitched<4>(chunk_rsrc(n.sl.v + (size_t)(16 * w) * n.sl.in, rows, n.sl.in), 0, r, h, n.sl.in, ld.rawv);
  else issue_raw_tile<4>(chunk_rsrc(n.sl.v + tv, rows, 128), 0, r, h, ld.rawv);
  issue_raw_tile<4>(chunk_rsrc(n.sl.d_o + tv, rows, 128), 0, r, h, ld.rawd);
}

// Tile-local cumulative gates of the direction whose gate dwords have arrived: G^T = g^T T, lane = token, registers =
// channels HC*h + 8g + 2m + p; the tile total (at the tile's last token in walking order) goes to `tot`.
template <bool FWD, int NG, int TW>
__device__ __forceinline__ void bwd_cumulate_gates(const BwdLoads<NG>& ld, int w, int lane, char* lds, f32x16_t (&G)[2]) {
  constexpr int HC = 8 * NG;
  const int r = lane & 31, h = lane >> 5;
  float* tot = reinterpret_cast<float*>(lds + BwdLds<TW>::tot);
  u32x4_t gfrag[2][2];
  finish_tfrags<2>(ld.gD, gfrag);  // (rows that carry no channel, NG = 2, hold zeros)
  const u32x4_t tri0 = tri_frag<FWD>(0, 0, r, h), tri1 = tri_frag<FWD>(1, 0, r, h);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    f32x16_t z = {0.f};
    z = mfma(gfrag[0][p], tri0, z);
    G[p] = mfma(gfrag[1][p], tri1, z);
  }
  if (r == (FWD ? 31 : 0)) {
#pragma unroll
    for (int c = 0; c < 4 * NG; ++c) {
      const int ch = HC * h + 8 * (c >> 2) + 2 * (c & 3);
      tot[w * 64 + ch] = G[0][c];
      tot[w * 64 + ch + 1] = G[1][c];
    }
  }
}

// Gates before tile w in walking order, minus the anchor (half the slab total), per channel, from the tile totals that the
// previous direction's tail (or the kernel's head) left one barrier ago.  False, for every wave alike, where the gates
// are out of range: same totals in every wave, and nothing has been stored yet.
template <bool FWD, int NG, int TW>
__device__ __forceinline__ bool bwd_anchor(int w, char* lds) {
  const int lane = fresh_lane();
  const float* tot = reinterpret_cast<const float*>(lds + BwdLds<TW>::tot) + (lane & (16 * NG - 1));
  float pre = 0.f, all = 0.f;
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    const float x = tot[t * 64];
    all += x;
    pre += (FWD ? (t < w) : (t > w)) ? x : 0.f;
  }
  reinterpret_cast<float*>(lds + BwdLds<TW>::off)[w * 64 + lane] = pre - 0.5f * all;
  const bool in_range = __builtin_amdgcn_ballot_w64(fabsf(all) * (0.5f * kLog2e) > kBwdHalfRange) == 0;
  wave_lds_sync();
  return in_range;
}

// One direction of one slab, for wave w (tile w).  dv accumulates over both directions (raw, unscaled).  The first
// direction (FIRST, not LAST) stages v and do and hands its dq and dk, rounded to bf16, to the second: in registers, or at
// Dk = 64, where the loops in between leave no room for dq, in LDS as far as there is room, else parked in the output tensor.  The second
// (LAST, not FIRST) adds its own to them and stores dq, dk, dv.  A one-direction (causal) launch runs a single direction that
// is both.  Registers set the order of the phases: dk and dv end before dq begins, and only e of the two factors is kept.
// SEG: the slab is a segment of a longer sequence.  With S_in the state entering it along the direction, R_out the
// gradient of the state leaving it, a = half the segment's gate total and ' = times e^a per k channel:
//   dq^_i += S_in' do_i,   dk^_j += R_out' v_j,   dv_j += R_out'^T k~_j
// (the e^{G_i - a}, e^{a - G_j} factors applied to dq^, dk^ at the end turn e^a into e^{G_i}, e^{T - G_j}), and the
// running sum of the gate gradient starts from the total of q dq - k dk over the segments walked later.
template <bool FWD, bool FIRST, bool LAST, int NG, bool SEG, int TW, bool PITCHED>
__device__ __forceinline__ void bwd_direction(const BwdSlab& sl, int L, int ntiles, int w, char* lds,
                                              float s, f32x16_t (&dv)[2], u32x4_t (&keepq)[NG], u32x4_t (&keepk)[NG],
                                              BwdLoads<NG>& ld, const BwdNext& nxt, f32x16_t (&G)[2]) {
  constexpr bool stage_vdo = FIRST;
  constexpr int kParkLds = NG == 4 && !(FIRST && LAST) ? BwdLds<TW>::parked : 0;
  constexpr bool kParkDq = NG == 4 && kParkLds < NG && !(FIRST && LAST);
  // Fetched ahead of the dq loop, or, where its registers do not hold that too (a fetched value that is spilled is waited
  // for at once), behind it: 1200 slabs of 128 tokens, Dk = 64 75 against 82 us with the gates early; 768 of 256 109 against 113
  // with the rows.
  constexpr bool kEarlyGates = !(LAST && kParkDq && TW <= 4);
  constexpr bool kEarlyRows = LAST && (NG == 2 || TW == 7 || TW == 3);
  constexpr int DK = 16 * NG;   // channels of q, k and the gates
  constexpr int HC = 8 * NG;    // channels per lane half
  int lane = fresh_lane();
  int r = lane & 31, h = lane >> 5;
  auto next_phase = [&] { lane = fresh_lane(), r = lane & 31, h = lane >> 5; };
  uint16_t* Q = reinterpret_cast<uint16_t*>(lds + BwdLds<TW>::q);
  uint16_t* K = reinterpret_cast<uint16_t*>(lds + BwdLds<TW>::k);
  uint16_t* V = reinterpret_cast<uint16_t*>(lds + BwdLds<TW>::v);
  uint16_t* DO = reinterpret_cast<uint16_t*>(lds + BwdLds<TW>::d_o);
  float* offs = reinterpret_cast<float*>(lds + BwdLds<TW>::off) + w * 64;
  float* dgtot = reinterpret_cast<float*>(lds + BwdLds<TW>::dgtot);
  const int rows = tile_rows(L, w);  // valid tokens of this wave's tile
  const size_t tk = (size_t)32 * w * DK, tv = (size_t)32 * w * 64;
  // where the tile's rows of dq and dk start (dv), and how far apart they are
  const size_t to_k = PITCHED ? (size_t)(16 * w) * sl.out : tk, to_v = PITCHED ? to_k : tv;
  const unsigned out_k = PITCHED ? sl.out : 2 * DK, out_v = PITCHED ? sl.out : 128;

  // ---- this tile's loads were issued a phase ago; v and do rows go to LDS once per slab (nobody reads the previous
  // slab's any more; the next barrier makes them visible) ----
  if (stage_vdo) {
    store_row<4>(V, 32 * w + r, h, ld.rawv);
    store_row<4>(DO, 32 * w + r, h, ld.rawd);
  }
  u32x4_t rawq[NG], rawk[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) rawq[i] = ld.rawq[i], rawk[i] = ld.rawk[i];

  // e = e^{G - a} per (token, channel): q~ = q e, k~ = k / e
  float e[2][4 * NG];
#pragma unroll
  for (int gq = 0; gq < NG; ++gq) {
    const f32x4_t o0 = *reinterpret_cast<const f32x4_t*>(offs + HC * h + 8 * gq);
    const f32x4_t o1 = *reinterpret_cast<const f32x4_t*>(offs + HC * h + 8 * gq + 4);
    const float o8[8] = {o0[0], o0[1], o0[2], o0[3], o1[0], o1[1], o1[2], o1[3]};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int p = 0; p < 2; ++p) e[p][4 * gq + m] = exp2_fast((G[p][4 * gq + m] + o8[2 * m + p]) * kLog2e);
  }
  {
    u32x4_t qt[NG], kt[NG];
#pragma unroll
    for (int gq = 0; gq < NG; ++gq)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = 4 * gq + m;
        const uint32_t wq = rawq[gq][m], wk = rawk[gq][m];
        qt[gq][m] = pack_bf16x2(bf16lo_to_f32(wq) * e[0][c], bf16hi_to_f32(wq) * e[1][c]);
        kt[gq][m] = pack_bf16x2(bf16lo_to_f32(wk) * __builtin_amdgcn_rcpf(e[0][c]), bf16hi_to_f32(wk) * __builtin_amdgcn_rcpf(e[1][c]));
      }
    store_row<NG>(Q, 32 * w + r, h, qt);
    store_row<NG>(K, 32 * w + r, h, kt);
  }
  // (only e is kept, not also 1 / e, which is needed again at the end)
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int c = 0; c < 4 * NG; ++c) asm volatile("" : "+v"(e[p][c]));
  lds_barrier();  // (2) q~, k~ of every tile visible

  next_phase();
  constexpr int kTile = 32 * kRow, kToDo = (BwdLds<TW>::d_o - BwdLds<TW>::q) / 2;
  const lds_u16_t Qs = (lds_u16_t)Q, Ks = (lds_u16_t)K, Vs = (lds_u16_t)V, Ds = (lds_u16_t)DO;
  // ---- dv and dk of tile w: over the query tiles I the direction keeps, both in one pass: the two score tiles of a step
  // are independent, so one's packs run under the other's matrix instructions ----
  KeyAcc<NG> dkh;
  dkh.zero();
  if (w < ntiles) {
    u32x4_t kB[NG], vB[4];
    {
      const RowPtr k(Ks + w * kTile, r, h);
#pragma unroll
      for (int ks = 0; ks < NG; ++ks) kB[ks] = k.frag(ks);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) vB[ks] = k.frag(ks, (BwdLds<TW>::v - BwdLds<TW>::k) / 2);
    }
    const int i0 = FWD ? w : 0, i1 = FWD ? ntiles : w + 1;
    RowPtr q(Qs + i0 * kTile, r, h);
    lds_u16_t qt = tr_ptr<NG>(Qs + i0 * kTile, lane), dt = NG == 4 ? qt : tr_ptr<4>(Ds + i0 * kTile, lane);
#pragma unroll 1
    for (int I = i0; I < i1; ++I, q.advance(kTile), qt += kTile, dt += kTile)
      add_dv_dk<FWD, NG>(I == w, q, kToDo, qt, NG == 4 ? qt + kToDo : dt, kB, vB, r, h, dv, dkh);
    if (SEG) {  // the gradient of the state leaving the segment, against this tile's k~ rows (dv) and v rows (dk)
      const uint16_t* rpt = sl.rpt + (FWD ? 0 : DK * 64) + tr_row_channel<4>(r) * DK + 8 * h;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int ks = 0; ks < NG; ++ks)
          dv[p] = mfma(*reinterpret_cast<const u32x4_t*>(rpt + 4 * p * DK + 16 * ks), kB[ks], dv[p]);
      const uint16_t* rp = sl.rp + (FWD ? 0 : DK * 64) + tr_row_channel<NG>(r) * 64 + 8 * h;
#pragma unroll
      for (int p = 0; p < NG / 2; ++p)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          dkh.a[p] = mfma(*reinterpret_cast<const u32x4_t*>(rp + 4 * p * 64 + 16 * ks), vB[ks], dkh.a[p]);
    }
  }
  next_phase();
  // ---- dv and dk (which the first direction hands to the second); X = q dq - k dk = s (q~ dq^ - k~ dk^): the exponentials
  // cancel, and the staged rows serve ----
  float X[2][4 * NG];
  uint16_t* turn = reinterpret_cast<uint16_t*>(lds + BwdLds<TW>::turn) + w * 16 * kRow;
  u32x4_t outv[4];
  if (LAST) {
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
#pragma unroll
      for (int m = 0; m < 4; ++m) outv[gq][m] = pack_bf16x2(dv[m >> 1][4 * gq + 2 * (m & 1)] * s, dv[m >> 1][4 * gq + 2 * (m & 1) + 1] * s);
  }
  {
#pragma unroll
    for (int gq = 0; gq < NG; ++gq) {
      const u32x4_t krow = load_piece(K, 32 * w + r, NG * h + gq);
      u32x4_t xk;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = 4 * gq + m;
        float b[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float dkc = dkh.get(gq, 2 * m + p);
          X[p][c] = (p ? bf16hi_to_f32(krow[m]) : bf16lo_to_f32(krow[m])) * dkc;
          b[p] = s * __builtin_amdgcn_rcpf(e[p][c]) * dkc;
          if (!FIRST) b[p] += p ? bf16hi_to_f32(keepk[gq][m]) : bf16lo_to_f32(keepk[gq][m]);
        }
        xk[m] = pack_bf16x2(b[0], b[1]);
      }
      keepk[gq] = xk;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // The counter that a load is waited for with goes down in the order of issue, stores included: a load behind a store waits for
  // that store.  So what is stored waits, packed, until what is fetched here is on its way.
  if (kParkDq && !FIRST) {
#pragma unroll
    for (int g = kParkLds; g < NG; ++g)
      keepq[g] = __builtin_amdgcn_raw_buffer_load_b128(chunk_rsrc(sl.dq + to_k, rows, out_k), r * out_k + h * (16u * NG) + 16u * g, 0, 0);
  }
  if (kEarlyGates) issue_bwd_gate_loads<NG>(nxt, w, r, h, ld);
  if (kEarlyRows) issue_bwd_qk_loads<NG, PITCHED>(nxt, w, r, h, ld);
  __builtin_amdgcn_sched_barrier(0);
  if (LAST) {
    store_rows<4, TW, PITCHED>(turn, outv, chunk_rsrc(sl.dv + to_v, rows, out_v), lane, out_v);
    store_rows<NG, TW, PITCHED>(turn, keepk, chunk_rsrc(sl.dk + to_k, rows, out_k), lane, out_k);
  }
  next_phase();
  // ---- dq of tile w: over the key tiles J the direction keeps ----
  KeyAcc<NG> dqh;
  dqh.zero();
  if (w < ntiles) {
    u32x4_t doB[4];
    {
      const RowPtr d(Ds + w * kTile, r, h);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) doB[ks] = d.frag(ks);
    }
    const int j0 = FWD ? 0 : w, j1 = FWD ? w + 1 : ntiles;
    RowPtr v(Vs + j0 * kTile, r, h);
    lds_u16_t k = tr_ptr<NG>(Ks + j0 * kTile, lane);
#pragma unroll 1
    for (int J = j0; J < j1; ++J, v.advance(kTile), k += kTile) add_dq<FWD, NG>(J == w, v, k, doB, r, h, dqh);
    if (SEG) {  // the state entering the segment: rows = the k channels of this lane's accumulator rows, over v
      const uint16_t* sp = sl.sp + (FWD ? 0 : DK * 64) + tr_row_channel<NG>(r) * 64 + 8 * h;
#pragma unroll
      for (int p = 0; p < NG / 2; ++p)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          dqh.a[p] = mfma(*reinterpret_cast<const u32x4_t*>(sp + 4 * p * 64 + 16 * ks), doB[ks], dqh.a[p]);
    }
  }
  next_phase();
  if (!FIRST) {
#pragma unroll
    for (int g = 0; g < kParkLds; ++g) keepq[g] = *reinterpret_cast<const u32x4_t*>(unit_ptr(lds + BwdLds<TW>::park, w * kParkLds + g, lane));
  }
  {
#pragma unroll
    for (int gq = 0; gq < NG; ++gq) {
      const u32x4_t qrow = load_piece(Q, 32 * w + r, NG * h + gq);
      u32x4_t xq;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = 4 * gq + m;
        float a[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float dqc = dqh.get(gq, 2 * m + p);
          X[p][c] = s * ((p ? bf16hi_to_f32(qrow[m]) : bf16lo_to_f32(qrow[m])) * dqc - X[p][c]);
          a[p] = s * e[p][c] * dqc;
          if (!FIRST) a[p] += p ? bf16hi_to_f32(keepq[gq][m]) : bf16lo_to_f32(keepq[gq][m]);
        }
        xq[m] = pack_bf16x2(a[0], a[1]);
      }
      keepq[gq] = xq;
    }
  }
  // the next direction's rows travel while this one finishes
  next_phase();
  if (!kEarlyGates) issue_bwd_gate_loads<NG>(nxt, w, r, h, ld);
  if (!kEarlyRows) issue_bwd_qk_loads<NG, PITCHED>(nxt, w, r, h, ld);
  if (LAST) issue_bwd_vdo_loads<NG, PITCHED>(nxt, w, r, h, ld);
  next_phase();
  __builtin_amdgcn_sched_barrier(0);
  if (!LAST) {
#pragma unroll
    for (int g = 0; g < kParkLds; ++g) *reinterpret_cast<u32x4_t*>(unit_ptr(lds + BwdLds<TW>::park, w * kParkLds + g, lane)) = keepq[g];
  }
  if (LAST || (kParkDq && kParkLds == 0)) {
    store_rows<NG, TW, PITCHED>(turn, keepq, chunk_rsrc(sl.dq + to_k, rows, out_k), lane, out_k);
  } else if (kParkDq) {
#pragma unroll
    for (int g = kParkLds; g < NG; ++g)
      __builtin_amdgcn_raw_buffer_store_b128(keepq[g], chunk_rsrc(sl.dq + to_k, rows, out_k), r * out_k + h * (16u * NG) + 16u * g, 0, 0);
  }
  // ---- dg: the running sum of X over the tokens the gate acts on.  Inside the tile by lane shifts (lane = token),
  // across tiles through the tile totals in LDS: walking forward a token takes everything from itself to the end,
  // i.e. the totals of this and the later tiles minus what lies before it in the tile. ----
  {
    float pfx[8 * NG];  // [p][c]
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int c = 0; c < 4 * NG; ++c) pfx[4 * NG * p + c] = X[p][c];
    half_prefix_sums(pfx);
    if (r == 31) {
#pragma unroll
      for (int c = 0; c < 4 * NG; ++c) {
        const int ch = HC * h + 8 * (c >> 2) + 2 * (c & 3);
        dgtot[w * 64 + ch] = pfx[c];
        dgtot[w * 64 + ch + 1] = pfx[4 * NG + c];
      }
    }
    // the next direction's cumulative gates and tile totals are prepared here, so that one barrier serves both exchanges
    bwd_cumulate_gates<LAST, NG, TW>(ld, w, fresh_lane(), lds, G);
    lds_barrier();  // (4) tile totals of X and of the next gates visible; nobody reads q~, k~, v, do of this direction
    next_phase();
    {
      const int cl = lane < DK ? lane : 0;
      float run = 0.f;
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const float y = dgtot[t * 64 + cl];
        run += (FWD ? (t >= w) : (t < w)) ? y : 0.f;
      }
      if (SEG) {
        const float* cy = sl.carry + (FWD ? 0 : 128) + cl;
        run += s * (cy[0] + cy[64]);
      }
      offs[lane] = run;
    }
    wave_lds_sync();
    uint16_t* dg = FWD ? sl.dgf : sl.dgb;
    u32x4_t out[NG];
#pragma unroll
    for (int gq = 0; gq < NG; ++gq) {
      const f32x4_t o0 = *reinterpret_cast<const f32x4_t*>(offs + HC * h + 8 * gq);
      const f32x4_t o1 = *reinterpret_cast<const f32x4_t*>(offs + HC * h + 8 * gq + 4);
      const float o8[8] = {o0[0], o0[1], o0[2], o0[3], o1[0], o1[1], o1[2], o1[3]};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = 4 * gq + m;
        float d[2];
#pragma unroll
        for (int p = 0; p < 2; ++p)
          d[p] = FWD ? o8[2 * m + p] - before_lane(pfx[4 * NG * p + c], r) : o8[2 * m + p] + pfx[4 * NG * p + c];
        out[gq][m] = pack_bf16x2(d[0], d[1]);
      }
    }
    store_rows<NG, TW>(turn, out, chunk_rsrc(dg + tk, rows, 2 * DK), lane);
  }
}

}  // namespace

// What the segments of long sequences read besides the tensors (see bwd_direction, SEG): per (sequence, segment) the
// two directions' matrices, written by gla_backward_segment_scan_kernel.
struct BwdSegments {
  const uint16_t *sp, *rp, *rpt;
  const float* carry;
  int nseg, seg_len;
};

// PITCHED: q, k and v are read out of the rows of a stacked projection and dq, dk and dv written into the rows of its gradient, where passes over memory would
// split and gather them (`BwdPitch`: elements from row to row, heads).  Rows of 64 or 128 bytes either way; the kernel itself takes 1 to 4 % longer.  us, splitting pass,
// op, its backward and gathering pass / op and backward on rows: Dk 32, 768 sequences of 196 tokens 107 / 85, 384 66 / 55 and 64 / 54 (3 and 12 heads), 48 33 / 29, 384 of
// 100 37 / 29, 1200 of 49 44 / 33, 240 of 256 48 / 38; Dk 64, 768 of 196 149 / 113, 1800 of 128 202 / 152.
struct BwdPitch {
  long long in, out;
  int H;
};

template <int NG, bool BIDIR, bool SEG, int TW, bool PITCHED>
__device__ __forceinline__ void gla_backward_slabs(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ gf, const uint16_t* __restrict__ gb, const uint16_t* __restrict__ d_o,
    uint16_t* __restrict__ dq, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, uint16_t* __restrict__ dgf,
    uint16_t* __restrict__ dgb, int* __restrict__ flags, int nslabs, int L, float s, const BwdSegments& sg, const BwdPitch& rows) {
  extern __shared__ __align__(16) char lds[];
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // slab i: a whole sequence, or (SEG) segment i % nseg of sequence i / nseg
  auto slab_of = [&](int i) {
    size_t t0 = (size_t)i * L;
    int len = L;
    BwdSlab sl{};
    if (SEG) {
      const int seq = i / sg.nseg, seg = i - seq * sg.nseg;
      t0 = (size_t)seq * L + (size_t)seg * sg.seg_len;
      len = min(sg.seg_len, L - seg * sg.seg_len);
      sl.sp = sg.sp + (size_t)i * 2 * (16 * NG * 64);
      sl.rp = sg.rp + (size_t)i * 2 * (16 * NG * 64);
      sl.rpt = sg.rpt + (size_t)i * 2 * (16 * NG * 64);
      sl.carry = sg.carry + (size_t)i * 256;
    }
    const size_t bk = t0 * (16 * NG), bv = t0 * 64;
    sl.q = q + bk, sl.k = k + bk, sl.v = v + bv, sl.gf = gf + bk, sl.gb = BIDIR ? gb + bk : nullptr, sl.d_o = d_o + bv;
    sl.dq = dq + bk, sl.dk = dk + bk, sl.dv = dv + bv, sl.dgf = dgf + bk, sl.dgb = BIDIR ? dgb + bk : nullptr;
    if constexpr (PITCHED) {
      static_assert(!SEG, "whole sequences");
      const int b = i / rows.H, head = i - b * rows.H;
      const size_t from = (size_t)b * L * rows.in, to = (size_t)b * L * rows.out;
      sl.q = q + from + head * (16 * NG), sl.k = k + from + head * (16 * NG), sl.v = v + from + head * 64;
      sl.dq = dq + to + head * (16 * NG), sl.dk = dk + to + head * (16 * NG), sl.dv = dv + to + head * 64;
      sl.in = 2u * (unsigned)rows.in, sl.out = 2u * (unsigned)rows.out;
    }
    sl.L = len;
    return sl;
  };
  BwdLoads<NG> ld;
  f32x16_t G[2];  // cumulative gates of the direction about to run, prepared one barrier ahead of it
  if ((int)blockIdx.x < nslabs) {
    const int lane = fresh_lane(), r = lane & 31, h = lane >> 5;
    const BwdSlab s0 = slab_of(blockIdx.x);
    const BwdNext first{s0, s0.gf, s0.L};
    issue_bwd_gate_loads<NG>(first, w, r, h, ld);
    issue_bwd_qk_loads<NG, PITCHED>(first, w, r, h, ld);
    issue_bwd_vdo_loads<NG, PITCHED>(first, w, r, h, ld);
    bwd_cumulate_gates<true, NG, TW>(ld, w, lane, lds, G);
    lds_barrier();
  }
  for (int slab = blockIdx.x; slab < nslabs; slab += gridDim.x) {
    const BwdSlab sl = slab_of(slab);
    const int ntiles = (sl.L + 31) / 32;
    const int following = slab + (int)gridDim.x;
    const BwdSlab sn = slab_of(following < nslabs ? following : slab);
    const BwdNext second{sl, sl.gb, sl.L}, next_first{sn, sn.gf, following < nslabs ? sn.L : 0};
    f32x16_t dvacc[2] = {{0.f}, {0.f}};
    // a direction that is not run has neither issued the loads of the slab that follows nor prepared its gates
    const auto skip = [&] {
      const int ln = fresh_lane();
      lds_barrier();  // a wave that has left must not touch the gate totals the others still read
      issue_bwd_gate_loads<NG>(next_first, w, ln & 31, ln >> 5, ld);
      issue_bwd_qk_loads<NG, PITCHED>(next_first, w, ln & 31, ln >> 5, ld);
      issue_bwd_vdo_loads<NG, PITCHED>(next_first, w, ln & 31, ln >> 5, ld);
      bwd_cumulate_gates<true, NG, TW>(ld, w, ln, lds, G);
      lds_barrier();
    };
    bool ok = bwd_anchor<true, NG, TW>(w, lds);
    if (ok) {
      u32x4_t keepq[NG], keepk[NG];
      if constexpr (BIDIR) {
        bwd_direction<true, true, false, NG, SEG, TW, PITCHED>(sl, sl.L, ntiles, w, lds, s, dvacc, keepq, keepk, ld, second, G);
        ok = bwd_anchor<false, NG, TW>(w, lds);
        if (ok) {
          bwd_direction<false, false, true, NG, SEG, TW, PITCHED>(sl, sl.L, ntiles, w, lds, s, dvacc, keepq, keepk, ld, next_first, G);
        } else {
          skip();  // (in each branch, so that nothing of this slab's loads stays alive for it)
        }
      } else {  // the causal op: the forward direction alone, first and last at once
        bwd_direction<true, true, true, NG, SEG, TW, PITCHED>(sl, sl.L, ntiles, w, lds, s, dvacc, keepq, keepk, ld, next_first, G);
      }
    } else {
      skip();
    }
    if (w == 0 && fresh_lane() == 0) {
      if (!SEG) flags[slab] = ok ? 0 : 1;
      else if (!ok) flags[slab / sg.nseg] = 1;  // one flag per sequence, cleared by the segment scan: any segment out of range gives it away
    }
  }
}

template <int NG, bool BIDIR, bool SEG, int TW>
__global__ __launch_bounds__(64 * TW, 2) void gla_backward_mfma_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ gf, const uint16_t* __restrict__ gb, const uint16_t* __restrict__ d_o,
    uint16_t* __restrict__ dq, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, uint16_t* __restrict__ dgf,
    uint16_t* __restrict__ dgb, int* __restrict__ flags, int nslabs, int L, float s, BwdSegments sg) {
  gla_backward_slabs<NG, BIDIR, SEG, TW, false>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, nslabs, L, s, sg, BwdPitch{});
}
template <int NG, int TW>
__global__ __launch_bounds__(64 * TW, 2) void gla_backward_rows_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ gf, const uint16_t* __restrict__ gb, const uint16_t* __restrict__ d_o,
    uint16_t* __restrict__ dq, uint16_t* __restrict__ dk, uint16_t* __restrict__ dv, uint16_t* __restrict__ dgf,
    uint16_t* __restrict__ dgb, int* __restrict__ flags, int nslabs, int L, float s, BwdPitch rows) {
  gla_backward_slabs<NG, true, false, TW, true>(q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, nslabs, L, s, BwdSegments{}, rows);
}

// Links the segments of every (sequence, direction) for the backward.  Per segment s (walked in the direction's order)
// it reads the forward's state pass (contribution U_s, decay D_s) and the gradient state pass (Q_s = sum over the
// segment's tokens of (q e^{G})^T do, unscaled), and leaves
//   sp   = sqrt(D_s) S_in(s),     S_in(s') = S_out(s) = D_s S_in(s) + U_s   for the segment s' walked next,
//   rp   = sqrt(D_s) R_out(s),    R_out(s) = Q_{s'} + D_{s'} R_out(s'),  zero for the segment walked last,
//   rpt  = rp transposed,
//   carry(s) = rowsum_v(S_out(s) R_out(s)): what q dq - k dk adds up to over the segments walked after s, since a segment's
//              part, rowsum_v(S_in Q - R_out U), is the difference of two such products and R_out is zero behind the last
// (bf16 matrices in plain row-major order; carry as two partial sums per channel, over 16 accumulator lanes each).
// One workgroup of two waves per (sequence, direction, register quad cq, 16 lanes of the passes' register order).  The walks are serial
// and short, so everything is fetched into LDS in one round trip and the loops stay small: unrolled over segments in registers this
// kernel took 1 us a segment, its code being read once and cold.  The first wave walks S, the second R at the same time, each with the
// next segment's values on their way out of LDS; what needs both, the carries, comes last, from all threads.  A thread holds the four
// state elements (k channels c, c+1) x (v columns x, x+1), so that its bf16 results leave as 4-byte words.  Chunks of kScanChunk
// segments; with more than one the walks follow each other and S_out waits in `term` in between.
// us, whole backward calls, one wave after the other walk / two: 24 sequences of 2305 tokens, Dk 32 49.2 / 46.6; 3 of 5000 46.5 / 38.5, of 9000, Dk 64
// (two chunks) 93.3 / 85.3; 12 of 300 27.6 / 27.0.
constexpr int kScanChunk = 48;
constexpr int kScanSegFloats = 256 + 256 + 8;  // U or S_out, Q or R_out, decays
__global__ __launch_bounds__(128) void gla_backward_segment_scan_kernel(
    const float* __restrict__ ws_fwd, const float* __restrict__ ws_grad, float* __restrict__ term, uint16_t* __restrict__ sp,
    uint16_t* __restrict__ rp, uint16_t* __restrict__ rpt, float* __restrict__ carry, int* __restrict__ flags, int nseq, int nseg,
    int ndir, int ng, int grad_swapped) {
  extern __shared__ __align__(16) float sh[];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), t = threadIdx.x & 63;
  const int cq = blockIdx.y >> 2, quarter = blockIdx.y & 3;
  const int seq = blockIdx.x / ndir, dir = blockIdx.x % ndir, gdir = grad_swapped ? 1 - dir : dir;
  if (seq >= nseq) return;
  const int chunk = min(nseg, kScanChunk), nchunks = (nseg + chunk - 1) / chunk;
  float *F = sh, *Q = F + chunk * 256, *D = Q + chunk * 256;
  const size_t state_elems = 16 * ng * 64;
  if (blockIdx.y == 0 && threadIdx.x == 0 && dir == 0) flags[seq] = 0;
  const int m = t & 3, lane = 16 * quarter + (t >> 2), h = lane >> 5;
  const int cbase = 8 * ng * h + 8 * cq, ch0 = cbase + 2 * m;  // k channels ch0 (pk = 0), ch0 + 1 (pk = 1)
  const int v0 = 2 * cpair<4>(lane & 31);                        // v columns v0 (pv = 0), v0 + 1 (pv = 1)
  auto slot = [&](int i, int d) { return (((size_t)seq * nseg + (dir == 0 ? i : nseg - 1 - i)) * 2 + d); };  // i-th segment walked
  // lane t fetches 16 bytes (four channels) of unit (pk, pv) = t >> 4: element (pk, pv) of thread t lies at 64 (2 pk + pv) + t
  const int fetched = ((((t >> 4) * 4 + cq) * 64) + 16 * quarter + (t & 15)) * 4;
  auto fetch = [&](const float* from, int d, int i0, int n, float* to) {
    for (int i = 0; i < n; ++i) load_to_lds16(from + slot(i0 + i, d) * kGlaStateFloats + fetched, lds_offset(to + i * 256));
  };
  auto fetch_decays = [&](int i0, int n) {
    for (int i = t >> 3; i < n; i += 8) D[8 * i + (t & 7)] = ws_fwd[slot(i0 + i, dir) * kGlaStateFloats + 64 * 64 + cbase + (t & 7)];
  };
  auto kept = [&](int i) { return term + ((slot(i, dir) * ng * 4 + blockIdx.y) * 64 + t) * 4; };
  struct Step {
    float x[4], d[2];
  };
  auto step = [&](const float* from, int i) {
    Step y;
#pragma unroll
    for (int j = 0; j < 4; ++j) y.x[j] = from[256 * i + 64 * j + t];
    y.d[0] = D[8 * i + 2 * m], y.d[1] = D[8 * i + 2 * m + 1];
    return y;
  };
  float S[4] = {0.f, 0.f, 0.f, 0.f}, R[4] = {0.f, 0.f, 0.f, 0.f};
  auto walk_states = [&](int i0, int n) {
    Step next = step(F, 0);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      const Step y = next;
      next = step(F, min(i + 1, n - 1));
      uint16_t* out = sp + slot(i0 + i, dir) * state_elems + ch0 * 64 + v0;
#pragma unroll
      for (int pk = 0; pk < 2; ++pk) {
        const float rd = __builtin_amdgcn_sqrtf(y.d[pk]);
        *reinterpret_cast<uint32_t*>(out + 64 * pk) = pack_bf16x2(rd * S[2 * pk], rd * S[2 * pk + 1]);
#pragma unroll
        for (int pv = 0; pv < 2; ++pv) {
          const int x = 2 * pk + pv;
          S[x] = __builtin_fmaf(y.d[pk], S[x], y.x[x]);
          F[256 * i + 64 * x + t] = S[x];
        }
      }
      if (nchunks > 1) *reinterpret_cast<f32x4_t*>(kept(i0 + i)) = f32x4_t{S[0], S[1], S[2], S[3]};
    }
  };
  auto walk_gradients = [&](int i0, int n) {  // (R_out of a segment takes the place of its Q)
    Step next = step(Q, n - 1);
#pragma unroll 1
    for (int i = n - 1; i >= 0; --i) {
      const Step y = next;
      next = step(Q, max(i - 1, 0));
      const size_t at = slot(i0 + i, dir) * state_elems;
      const float rd[2] = {__builtin_amdgcn_sqrtf(y.d[0]), __builtin_amdgcn_sqrtf(y.d[1])};
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        *reinterpret_cast<uint32_t*>(rp + at + (ch0 + p) * 64 + v0) = pack_bf16x2(rd[p] * R[2 * p], rd[p] * R[2 * p + 1]);
        *reinterpret_cast<uint32_t*>(rpt + at + (v0 + p) * 16 * ng + ch0) = pack_bf16x2(rd[0] * R[p], rd[1] * R[2 + p]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        Q[256 * i + 64 * j + t] = R[j];
        R[j] = __builtin_fmaf(y.d[j >> 1], R[j], y.x[j]);
      }
    }
  };
  // (segment, channel 2 mm + pk): the products of the 16 lanes that hold it, in a fixed order
  auto carries = [&](int i0, int n) {
    for (int j = threadIdx.x; j < 8 * n; j += 128) {
      const int i = j >> 3, mm = (j >> 1) & 3, pk = j & 1;
      float acc = 0.f;
#pragma unroll
      for (int l = 0; l < 16; ++l) {
        const int e = 256 * i + 128 * pk + 4 * ((l + i) & 15) + mm;  // (segments start in different banks)
        acc += F[e] * Q[e] + F[e + 64] * Q[e + 64];
      }
      carry[slot(i0 + i, dir) * 128 + 64 * (quarter & 1) + cbase + (j & 7)] = acc;
    }
  };
  if (nchunks == 1) {
    if (wave == 0) fetch(ws_fwd, dir, 0, nseg, F);
    else fetch(ws_grad, gdir, 0, nseg, Q), fetch_decays(0, nseg);
    wait_vmem<0>();
    lds_barrier();
    if (wave == 0) walk_states(0, nseg);
    else walk_gradients(0, nseg);
    lds_barrier();
    carries(0, nseg);
    return;
  }
  for (int c = 0; c < nchunks; ++c) {
    const int i0 = c * chunk, n = min(chunk, nseg - i0);
    if (wave == 0) {
      fetch(ws_fwd, dir, i0, n, F);
      fetch_decays(i0, n);
      wait_vmem<0>();
      wave_lds_sync();
      walk_states(i0, n);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (what lies there has been read and written)
    }
  }
  for (int c = nchunks - 1; c >= 0; --c) {
    const int i0 = c * chunk, n = min(chunk, nseg - i0);
    lds_barrier();  // (the chunk before has been read)
    if (wave == 0) {
      for (int i = 0; i < n; ++i) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(kept(i0 + i));
#pragma unroll
        for (int j = 0; j < 4; ++j) F[256 * i + 64 * j + t] = x[j];
      }
    } else {
      fetch(ws_grad, gdir, i0, n, Q);
      fetch_decays(i0, n);
      wait_vmem<0>();
      wave_lds_sync();
      walk_gradients(i0, n);
    }
    lds_barrier();
    carries(i0, n);
  }
}

static bool seg_grid_ok(int B, int H, bool bidir) { return (long long)B * H * (bidir ? 2 : 1) <= 65535; }

bool gla_backward_mfma_supported(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir) {
  if (!(io_dtype == 1 && gate_dtype == 1 && (Dk == 64 || Dk == 32) && Dv == 64)) return false;
  return L <= 32 * kBwdTiles || seg_grid_ok(B, H, true);
}

// Long sequences: two state passes (kGlaStateFloats floats per sequence, segment and direction each), the S_in Q terms
// and the carries (fp32), then the three bf16 matrices the segments read.
static size_t seg_slots(int B, int H, int nseg) { return (size_t)B * H * nseg * 2; }
size_t gla_backward_mfma_workspace(int B, int H, int L, int Dk, int Dv) {
  if (L <= 32 * kBwdTiles || !(Dk == 64 || Dk == 32) || Dv != 64) return 0;
  return seg_slots(B, H, gla_segments(L)) * ((2 * (size_t)kGlaStateFloats + 64 * 64 + 128) * sizeof(float) + 3 * (size_t)64 * 64 * 2);
}

struct BwdLaunch {
  const void *q, *k, *v, *gf, *gb, *d_o;
  void *dq, *dk, *dv, *dgf, *dgb;
  int* flags;
  int nslabs, L;
  float s;
  BwdSegments sg;
  BwdPitch rows;  // (in = 0: head-major tensors)
  int num_cu;
  hipStream_t stream;
};
template <int NG, bool BIDIR, bool SEG, int TW>
static int launch_bwd_t(const BwdLaunch& l) {
  static_assert(kBwdTiles / TW * BwdLds<TW>::total <= 160 * 1024, "the workgroups of a CU fit its LDS");
  const int most = l.num_cu * (kBwdTiles / TW);
  const auto launch = [&](auto* kernel, bool (&done)[64], const auto& last) {
    if (!allow_lds(reinterpret_cast<const void*>(kernel), BwdLds<TW>::total, done)) return -5;
    hipLaunchKernelGGL(kernel, dim3(l.nslabs < most ? l.nslabs : most), dim3(64 * TW), BwdLds<TW>::total, l.stream,
                       (const uint16_t*)l.q, (const uint16_t*)l.k, (const uint16_t*)l.v, (const uint16_t*)l.gf, (const uint16_t*)l.gb,
                       (const uint16_t*)l.d_o, (uint16_t*)l.dq, (uint16_t*)l.dk, (uint16_t*)l.dv, (uint16_t*)l.dgf, (uint16_t*)l.dgb,
                       l.flags, l.nslabs, l.L, l.s, last);
    return hipGetLastError() == hipSuccess ? 0 : -5;
  };
  if constexpr (BIDIR && !SEG) {
    static bool done_rows[64] = {};
    if (l.rows.in) return launch(gla_backward_rows_kernel<NG, TW>, done_rows, l.rows);
  }
  static bool done[64] = {};
  return launch(gla_backward_mfma_kernel<NG, BIDIR, SEG, TW>, done, l.sg);
}
// Slabs of up to 64 and up to 128 tokens get workgroups of two and four waves, four and two of them to a CU: in one of eight, the
// waves without a tile idle and nothing runs beside the loads.  us, eight waves / as many as the slab has tiles (dword operands): Dk 64:
// 2010 slabs of 57 tokens 119 / 62, 1200 of 128 113 / 83, 3 of 49 20 / 16; Dk 32: 91 / 37, 82 / 51, 16 / 13.
// Seven waves instead of eight for 129 to 224 tokens.  Both directions at Dk 64, where the LDS of the eighth tile also holds the first
// direction's dq: 768 slabs of 129 tokens 74.6 / 71.1, of 145 77.3 / 72.9, of 180 87.1 / 81.7, of 192 88.5 / 82.9, of 196 91.4 / 87.1, 300 of 160 52.2 / 50.4,
// one of 160 26.4 / 26.2.  The rest by the wave that idles: the forward direction alone, Dk 64 768 of 129 45.4 / 42.0, of 192 52.9 / 50.1, of 210 55.8 / 53.1, 300
// of 145 30.3 / 29.5; Dk 32, both directions 768 of 160 49.7 / 48.9, 1200 of 180 83.3 / 82.1, one 18.1 / 18.0, forward 768 of 129 30.2 / 30.0, 1200 of 160 45.5 /
// 44.7.
// Three waves instead of four for 65 to 96 tokens at Dk 64, again with room for that dq: both directions 768 slabs of 70 tokens 39.0 / 36.0, 1200 55.4 /
// 51.1, 297 27.3 / 26.3, 768 of 96 41.9 / 37.8; forward alone 768 of 65 24.1 / 23.8, of 96 26.3 / 25.6, 1200 of 80 34.9 / 34.0, 300 of 65 17.5 / 16.9, one 11.6 /
// 11.5.  (Dk 32 has its dq in registers: 768 of 96 27.1 / 26.8, 1200 35.3 / 35.3; four.)
template <int NG, bool BIDIR>
static int launch_bwd(const BwdLaunch& l, bool seg, int tokens) {
  if (seg) return tokens <= 128 ? launch_bwd_t<NG, BIDIR, true, 4>(l) : launch_bwd_t<NG, BIDIR, true, 8>(l);
  if (tokens <= 64) return launch_bwd_t<NG, BIDIR, false, 2>(l);
  if constexpr (NG == 4)
    if (tokens <= 96) return launch_bwd_t<NG, BIDIR, false, 3>(l);
  if (tokens <= 128) return launch_bwd_t<NG, BIDIR, false, 4>(l);
  return tokens <= 224 ? launch_bwd_t<NG, BIDIR, false, 7>(l) : launch_bwd_t<NG, BIDIR, false, 8>(l);
}

// Where the segments of a call keep what links them: n slots, one per (sequence, segment, direction).
struct BwdRoom {
  float *fwd, *grad, *term, *carry;
  uint16_t *sp, *rp, *rpt;
  // pieces go to `scratch` (the recurrent kernel's, which runs when everything here has been read) while they fit there, else to `ws`
  bool lay_out(size_t n, int Dk, void* scratch, size_t scratch_bytes, void* ws, size_t ws_bytes) {
    bool ok = true;
    const auto take = [&](size_t bytes) -> char* {
      char* p;
      if (bytes <= scratch_bytes) p = (char*)scratch, scratch = p + bytes, scratch_bytes -= bytes;
      else if (bytes <= ws_bytes) p = (char*)ws, ws = p + bytes, ws_bytes -= bytes;
      else p = nullptr, ok = false;
      return p;
    };
    const size_t state = (size_t)Dk * 64;
    fwd = (float*)take(2 * n * kGlaStateFloats * sizeof(float));
    grad = fwd + (ok ? n * kGlaStateFloats : 0);
    term = (float*)take(n * state * sizeof(float));
    sp = (uint16_t*)take(n * state * 2);
    rp = (uint16_t*)take(n * state * 2);
    rpt = (uint16_t*)take(n * state * 2);
    carry = (float*)take(n * 128 * sizeof(float));
    return ok;
  }
};
// Segments of 128 tokens, two workgroups of four waves to a CU, or of up to 256, one of eight.  The short ones take less than half
// the time each and overlap, but double what the states cost.  us of the whole backward, long / short, at the number of long ones:
// Dk 32: 6 39 / 31, 48 44.5 / 36, 240 56.4 / 55.8, 360 92 / 76, 576 137 / 117, 384 of 256 99.8 / 101.7: always short;
// Dk 64: 6 46 / 41, 48 57 / 47 and 65 / 60, 192 71 / 76, 240 81 / 92, 576 194 / 219: short up to half a round.
static bool short_segments(int B, int H, int L, int Dk) { return Dk == 32 || (long long)B * H * gla_segments(L) <= 128; }

// flags: one int per (batch, head) sequence, written by every launch: 1 = not computed here (gates out of range)
int launch_gla_backward_mfma(const void* q, const void* k, const void* v, const void* gf, const void* gb,
                             const void* d_o, void* dq, void* dk, void* dv, void* dgf, void* dgb, int* flags,
                             void* scratch, size_t scratch_bytes, void* seg_workspace, size_t seg_bytes, int B, int H, int L,
                             int Dk, float s, long long ld_in, long long ld_out, hipStream_t stream) {
  constexpr int kMaxDevices = 64;
  static bool attr_done_dev[kMaxDevices] = {};
  static int num_cu_dev[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return -5;
  if (!attr_done_dev[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -5;
    num_cu_dev[dev] = n > 0 ? n : 256;
    attr_done_dev[dev] = true;
  }
  const bool seg = L > 32 * kBwdTiles;
  if (ld_in && (seg || !gb)) return -95;
  BwdSegments sg{};
  int nslabs = B * H;
  if (seg) {
    if (!seg_workspace || !seg_grid_ok(B, H, gb != nullptr)) return -22;
    const int ndir = gb ? 2 : 1, ng = Dk / 16;
    BwdRoom r;
    if (!(short_segments(B, H, L, Dk) && r.lay_out(seg_slots(B, H, (L + 127) / 128), Dk, scratch, scratch_bytes, seg_workspace, seg_bytes))) {
      r = BwdRoom();
      if (!r.lay_out(seg_slots(B, H, gla_segments(L)), Dk, nullptr, 0, seg_workspace, seg_bytes)) return -28;
      sg.nseg = gla_segments(L), sg.seg_len = gla_segment_len(L);
    } else {
      sg.nseg = (L + 127) / 128, sg.seg_len = 128;
    }
    // One launch for both state passes: contributions k~^T v and decays of every segment, both directions, and the gradient
    // states, the same sums over (q, do) with each token's own gate included in its weight.
    GlaArgs a{};
    a.q = q, a.k = k, a.v = v, a.g_fwd = gf, a.g_bwd = gb, a.o = const_cast<void*>(d_o), a.workspace = r.fwd;
    a.B = B, a.H = H, a.L = L, a.Dk = Dk, a.Dv = 64, a.scale = 1.f, a.out_scale = 1.f, a.io_dtype = 1, a.gate_dtype = 1;
    a.stream = stream;
    int rc;
    if (Dk == 32) {
      rc = launch_gla_states(a, sg.seg_len, sg.nseg, r.fwd, q, d_o, r.grad);
    } else {
      // The chunked kernel's state pass anchors a token at the END of its walk (the weight of token j is the decay from j to
      // the last token walked); the gradient state needs the decay from the FIRST token walked to i, i.e. the walk of
      // the other direction over the same gates: the forward gates go to the reverse waves and the reverse gates to the
      // forward waves, and slot d of that pass belongs to direction 1 - d.  (The causal op runs both directions on its
      // one gate tensor and uses the forward slot of the first pass and the reverse slot of the second.)
      if (!gb) a.g_bwd = gf;
      a.state_pass = 1, a.state_segments = sg.nseg, a.state_seg_len = sg.seg_len;
      rc = launch_gla_mfma(a);
    }
    if (rc != 0) return rc;
    static bool done[64] = {};
    if (!allow_lds(reinterpret_cast<const void*>(gla_backward_segment_scan_kernel), kScanChunk * kScanSegFloats * sizeof(float), done)) return -5;
    const int held = sg.nseg < kScanChunk ? sg.nseg : kScanChunk;
    hipLaunchKernelGGL(gla_backward_segment_scan_kernel, dim3((B * H * ndir + 7) / 8 * 8, 4 * ng), dim3(128),
                       held * kScanSegFloats * sizeof(float), stream, r.fwd, r.grad, r.term, r.sp, r.rp, r.rpt, r.carry, flags, B * H,
                       sg.nseg, ndir, ng, (int)(Dk == 64));
    sg.sp = r.sp, sg.rp = r.rp, sg.rpt = r.rpt, sg.carry = r.carry;
    nslabs = B * H * sg.nseg;
  }
  const BwdLaunch l{q, k, v, gf, gb, d_o, dq, dk, dv, dgf, dgb, flags, nslabs, L, s, sg, BwdPitch{ld_in, ld_out, H}, num_cu_dev[dev], stream};
  const int tokens = seg ? sg.seg_len : L;
  if (gb) return Dk == 64 ? launch_bwd<4, true>(l, seg, tokens) : launch_bwd<2, true>(l, seg, tokens);
  return Dk == 64 ? launch_bwd<4, false>(l, seg, tokens) : launch_bwd<2, false>(l, seg, tokens);
}

}  // namespace vig
