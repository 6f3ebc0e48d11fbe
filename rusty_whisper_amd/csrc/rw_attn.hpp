// rw_attn.hpp -- multi-head attention on gfx950 (device code).
//
// out[t_q, n_state] = concat_h softmax(q_h k_h^T / sqrt(64) + mask) v_h, as
// mha_split_kv (src/encoder.rs:48-80) computes it in f32.
//
//   k_attn_split   k and v (f32) -> f16 pairs x = hi + lo (hi = f16(x), lo =
//        f16(x - hi)), stored as the matrix cores' operands: per (head, 32 kv
//        rows) the 16 KB of ATT_BLK below (k_gemm's GEMM_KOP and GEMM_VOP
//        epilogues write the same blocks from the products that make K and V)
//   k_attn_tile    calls of more than 8 query rows: one workgroup per (32 or
//        64 query rows, head), whose 4 wavefronts split the kv blocks
//        between them and meet in LDS at the end
//   k_attn    calls of at most 8 query rows (a decoding step), or of at most 64
//        against many keys: one workgroup of two wavefronts per (32 query rows,
//        head[, kv run]); k_attn_combine merges the runs
//
// Precision.  Every product runs on v_mfma_f32_32x32x16_f16 as three f16
// products, hi*hi + hi*lo + lo*hi, accumulated in f32: each operand keeps
// 22 of f32's 24 significant bits and the dropped lo*lo term is below 2^-22
// of the product, so outputs stay within about 1e-6 (relative to the row) of
// the exact result, like the reference's f32 arithmetic.  Probabilities
// enter scaled to 2^12 or more at the row's maximum (ATT_PS), so that small
// ones keep their f16 bits: a step of 2^-24 is 2^-36 of the largest.
// Inputs must stay below f16's 65504 in magnitude (whisper's projections are
// far below it); inputs below about 1e-3 lose a few bits to f16 subnormal
// residuals.  The softmax is online (running reference score and sum per
// query row) in f32, which is the reference's max / exp / sum / divide
// reordered.
//
// Layouts inside the kernels.  The score block is computed transposed, S^T =
// K Q^T (32 kv x 32 queries): lane (h, n) then holds 16 kv entries of query n, so a
// query row's maximum and sum are in-lane plus one exchange with lane n+32.
// The output is accumulated transposed as well, O^T = V^T P^T, so the
// per-block rescale of a query column is one multiplier per lane.  P^T's
// registers feed that MFMA's B operand directly: lane half h holds kv
// 4h..4h+3 and 8+4h..8+4h+3 of each 16, and the v^T operands hold each
// 16-block of kv positions in that order (attn_vpos).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "rw_layout.hpp"

namespace rw {

constexpr int ATT_DH = 64;   // head size (every whisper model)
constexpr int ATT_KVB = 32;  // kv rows per block
constexpr int ATT_QB = 64;   // query rows a workspace's rows are padded to
constexpr int ATT_NK = 4;    // wavefronts of a k_attn_tile workgroup
constexpr int ATT_STEP_MAX = 8;   // query rows of a k_attn call at most
constexpr int ATT_ROWS_MAX = 64;  // query rows of a call that splits K and V as it loads them, at most
#ifndef ATT_MAX_SPLIT_N
#define ATT_MAX_SPLIT_N 32
#endif
constexpr int ATT_MAX_SPLIT = ATT_MAX_SPLIT_N;  // kv runs of one (query block, head) at most
static_assert(ATT_MAX_SPLIT < 128, "k_attn packs the run count into 7 bits");

// few (query block, head) workgroups -- a decoding step: split the kv
// blocks over up to ATT_MAX_SPLIT workgroups each (down to one 32-row block
// per run: each run is then one short chain of loads; the decoder step's
// cross-attention, 47 blocks per head, runs 26 splits instead of 11: 2% per
// token, 3% at 440 cached rows), merged by k_attn_combine
#ifndef ATT_SPLIT_MINBLK
#define ATT_SPLIT_MINBLK 1
#endif
inline int attn_nsplit(size_t groups, size_t nblk) {
  if (groups == 0 || groups >= 256 || nblk < 8) return 1;
  const size_t want = (512 + groups - 1) / groups, most = nblk / ATT_SPLIT_MINBLK;
  const size_t n = want < most ? want : most;
  return n < (size_t)ATT_MAX_SPLIT ? (int)n : ATT_MAX_SPLIT;
}

// Which kernel a call runs.  qt: 32-row query tiles per k_attn_tile workgroup (1
// or 2), 0: k_attn with its keys in nsplit runs.  rows: K and V are split as
// they are loaded (at most 64 rows against keys of their own).
//
// At most 8 rows run k_attn.  9 to 64 rows run k_attn_tile, where a wavefront's
// chain of a quarter of the kv blocks is short, else k_attn and its merge:
//   * splitting K and V itself a chain takes about 2 us and 1.7 per block (9 rows,
//     6 heads: 7.2 us at 8 kv blocks, 8.6 at 12, 9.8 at 14, 11.3 at 20, 20.9 at
//     47) and k_attn 8 to 9 at any length (7.9, 7.8, 8.1, 8.1, 9.0): up to
//     12 blocks;
//   * from split blocks, about 3 us and 0.7 per block (5.4 at 12, 7.4 at 24, 8.6
//     at 32, 11.3 at 47) against 7.2, 7.7, 8.1, 8.3: up to 32 blocks, and beyond
//     them where there are more than 24 (tile, head) pairs, which fill the chip
//     and make the merge long (64 rows at 47 blocks: 6 heads 12.2 against 9.4, 12
//     heads 12.3 against 11.5, 20 heads 12.4 against 12.9).
// 33 to 64 rows, two tiles a head, take at most 12 runs: with one per block the
// merge reads more than the runs save (64 rows at 47 blocks, 12 heads: 16.5 us
// with 32 runs, 12.2 with 12; 20 heads 18.0 with 26, 13.9).
// More rows run k_attn_tile: 64 per workgroup where those fill 3/4 of the 512
// workgroup places (two per CU), else 32 (k_attn_tile has both sides measured).
struct AttnRoute {
  int qt;
  bool rows;
  int nsplit;
};
constexpr size_t ATT_TILE_ROWS_BLK = 12, ATT_TILE_KV_BLK = 32, ATT_TILE_KV_PAIRS = 24;
constexpr int ATT_TWO_TILE_RUNS = 12;
inline AttnRoute attn_route(size_t t_q, size_t t_kv, size_t n_head, bool presplit, int max_split) {
  const size_t nblk = (t_kv + ATT_KVB - 1) / ATT_KVB, tiles = (t_q + 31) / 32;
  AttnRoute r{0, !presplit && t_q <= (size_t)ATT_ROWS_MAX, 1};
  if (t_q <= (size_t)ATT_ROWS_MAX) {
    int n = attn_nsplit(n_head, nblk);
    if (n > max_split) n = max_split;
    if (tiles > 1 && n > ATT_TWO_TILE_RUNS) n = ATT_TWO_TILE_RUNS;
    const bool runs = presplit ? nblk > ATT_TILE_KV_BLK && tiles * n_head <= ATT_TILE_KV_PAIRS : nblk > ATT_TILE_ROWS_BLK;
    if (t_q <= (size_t)ATT_STEP_MAX || (runs && n > 1)) {
      r.nsplit = n;
      return r;
    }
  }
  r.qt = !r.rows && (t_q + 63) / 64 * n_head >= 384 ? 2 : 1;
  return r;
}

// kv index (within a 16-block) stored at position p of the v^T operands: the
// middle quads swap (an involution)
RW_HD inline int attn_vpos(int p) {
  const int qd = (p >> 2) & 3;
  return qd == 1 ? p + 4 : qd == 2 ? p - 4 : p;
}

// K and v^T of one (head, 32 kv rows) as operands: four parts of ATT_PART
// f16 (K hi, K lo, v^T hi, v^T lo), each 4 fragments [64 lanes][8], so that a
// wavefront's load of a fragment is one contiguous 1 KB.  K's fragment s:
// lane 32 h + n holds values 16 s + 8 h .. + 7 of kv row n.  v^T's fragment
// 2 dt + s: lane 32 h + n holds value 32 dt + n of kv rows 16 s + attn_vpos(8 h
// + e), e = 0 .. 7.  (Row-major planes, whose lanes read 16-byte pieces 128
// bytes apart, held the large-v3 encoder's attention at 62 us.)
constexpr int ATT_PART = 4 * 64 * 8;
constexpr int ATT_BLK = 4 * ATT_PART;  // f16 per (head, block)

struct AttnPlanes {
  const uint16_t *kv;  // [head][tkv_pad / 32][ATT_BLK]
  int tq_pad, tkv_pad;
};

#if defined(__HIPCC__)

typedef _Float16 att_v8h __attribute__((ext_vector_type(8)));
typedef float att_v16f __attribute__((ext_vector_type(16)));

typedef float att_v2f __attribute__((ext_vector_type(2)));
typedef _Float16 att_v2h __attribute__((ext_vector_type(2)));
constexpr float ATT_LOG2E = 1.4426950408889634f;
constexpr float ATT_PS = 4096.0f;  // P's scale in its products

// x = hi + lo, both f16
__device__ inline void att_split(float x, uint16_t &hi, uint16_t &lo) {
  const _Float16 h = (_Float16)x;
  const _Float16 l = (_Float16)(x - (float)h);
  hi = __builtin_bit_cast(uint16_t, h);
  lo = __builtin_bit_cast(uint16_t, l);
}

// 8 f32 values -> the 8 hi and the 8 lo halves
struct AttSplit8 {
  uint4 hi, lo;
};
__device__ inline AttSplit8 att_split8(const float (&v)[8]) {
  uint16_t h8[8], l8[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) att_split(v[e], h8[e], l8[e]);
  return {*reinterpret_cast<const uint4 *>(h8), *reinterpret_cast<const uint4 *>(l8)};
}

// One workgroup per (head, 32-row kv block): its K rows (row-contiguous
// 32-byte reads, 128-byte runs written) and its v^T fragments (a lane gathers
// its 8 rows' value, 128-byte runs of a row per load; 1 KB runs written).
// Rows >= t_kv are zeros.  Bound by its bytes, 8 t n read and 8 t n written:
// 4.9 us for large-v3's 30.7 MB (7.1 us when v^T went through LDS to row-major
// planes).  Into blocks that the call before has just read it takes 12, likely
// because other XCDs' L2s still hold the lines it stores to (attention calls that
// take turns over 8 workspaces 48 us each, over one 55).
__global__ __launch_bounds__(256) void k_attn_split(const float *__restrict__ k, int ldk, const float *__restrict__ v,
                                                    int ldv, int t_kv, int nblk, uint16_t *__restrict__ kv) {
  const int head = blockIdx.x / nblk, blk = blockIdx.x % nblk, t = threadIdx.x;
  uint16_t *o = kv + (size_t)blockIdx.x * ATT_BLK;
  float kx[8], vx[8];
  const int c = t & 7, n = t >> 3;  // K: row n, values 8 c ..
  {
    const int row = blk * ATT_KVB + n;
    const float4 *src = reinterpret_cast<const float4 *>(k + (size_t)min(row, t_kv - 1) * ldk + head * ATT_DH + 8 * c);
    const float4 a = src[0], b = src[1];
    const bool live = row < t_kv;
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) kx[e] = live ? x[e] : 0.0f;
  }
  const int f = t >> 6, l = t & 63;  // v^T: fragment f, lane l
  {
    const float *src = v + head * ATT_DH + (f >> 1) * 32 + (l & 31);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int row = blk * ATT_KVB + 16 * (f & 1) + attn_vpos(8 * (l >> 5) + e);
      const float x = src[(size_t)min(row, t_kv - 1) * ldv];
      vx[e] = row < t_kv ? x : 0.0f;
    }
  }
  const int ko = ((c >> 1) * 64 + 32 * (c & 1) + n) * 8, vo = 2 * ATT_PART + t * 8;
  const AttSplit8 ks = att_split8(kx), vs = att_split8(vx);
  *reinterpret_cast<uint4 *>(o + ko) = ks.hi;
  *reinterpret_cast<uint4 *>(o + ATT_PART + ko) = ks.lo;
  *reinterpret_cast<uint4 *>(o + vo) = vs.hi;
  *reinterpret_cast<uint4 *>(o + ATT_PART + vo) = vs.lo;
}

// Several decoding states' one-token steps in one self-attention: plane
// "head" b * n_head + h is head h of beam b, so one k_attn launch over
// n_beams * n_head heads serves every beam (each attends to its own cache).
constexpr int ATT_MAX_BEAMS = 8;
struct BeamCaches {
  float *k[ATT_MAX_BEAMS];  // beam b's f32 key cache [n_ctx][n]
  float *v[ATT_MAX_BEAMS];  // and value cache
};

// out rows [0, t) x columns [0, cols) = 0 (attention over no keys)
__global__ __launch_bounds__(256) void k_attn_zero(float *__restrict__ out, int ld, int t, int cols) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < (size_t)t * cols) out[(idx / cols) * ld + idx % cols] = 0.0f;
}

__device__ inline att_v8h att_ld(const uint16_t *p) {
  return __builtin_bit_cast(att_v8h, *reinterpret_cast<const uint4 *>(p));
}

// c += ah bh + ah bl + al bh
__device__ inline void att_mma3(att_v8h ah, att_v8h al, att_v8h bh, att_v8h bl, att_v16f &c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, c, 0, 0, 0);
}

// One kv block's operands for one wavefront: K rows as the A operand of S^T
// (4 steps of 16 of the head's 64 values), v^T rows as the A operand of O^T
// (2 row tiles of 32 values x 2 steps of 16 kv).
struct AttK {
  att_v8h kh[4], kl[4];
};
struct AttV {
  att_v8h vh[2][2], vl[2][2];
};

// (base: the block's 4 parts plus this lane's 8 values)
__device__ inline void att_load_k(const uint16_t *base, AttK &o) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    o.kh[s] = att_ld(base + s * 512);
    o.kl[s] = att_ld(base + ATT_PART + s * 512);
  }
}

__device__ inline void att_load_v(const uint16_t *base, AttV &o) {
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      o.vh[dt][s] = att_ld(base + 2 * ATT_PART + (2 * dt + s) * 512);
      o.vl[dt][s] = att_ld(base + 3 * ATT_PART + (2 * dt + s) * 512);
    }
}

// The same K and v^T operands straight from f32 rows (kf, vf with row
// strides ldk, ldv; rows >= t_kv are zeros), for calls that do not split K
// and V into planes first: the loads (raw) and the split (att_split, the
// values k_attn_split stores) are separate, so the loads can run ahead.
struct AttKRaw {
  float4 x[4][2];
};
struct AttVRaw {
  float x[2][2][8];
};
// (last: the newest kv row, t_kv - 1, comes from there instead of kf / vf)
__device__ inline void att_load_k_raw(const float *kf, int ldk, int t_kv, int head, int blk, int h, int n,
                                      AttKRaw &o, const float *last = nullptr) {
  // lane (h, n): kv row 32 blk + n, values 8h + 16s .. + 7
  const int row = min(blk * ATT_KVB + n, t_kv - 1);
  const float *src = (last && row == t_kv - 1 ? last : kf + (size_t)row * ldk) + head * ATT_DH + 8 * h;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    o.x[s][0] = *reinterpret_cast<const float4 *>(src + 16 * s);
    o.x[s][1] = *reinterpret_cast<const float4 *>(src + 16 * s + 4);
  }
}
__device__ inline void att_split_k(const AttKRaw &x, bool live, AttK &o) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const float v[8] = {x.x[s][0].x, x.x[s][0].y, x.x[s][0].z, x.x[s][0].w,
                        x.x[s][1].x, x.x[s][1].y, x.x[s][1].z, x.x[s][1].w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint16_t hb, lb;
      att_split(live ? v[e] : 0.0f, hb, lb);
      o.kh[s][e] = __builtin_bit_cast(_Float16, hb);
      o.kl[s][e] = __builtin_bit_cast(_Float16, lb);
    }
  }
}
__device__ inline void att_load_v_raw(const float *vf, int ldv, int t_kv, int head, int blk, int h, int n,
                                      AttVRaw &o, const float *last = nullptr) {
  // lane (h, n): value d = 32 dt + n of the kv rows that the v^T plane keeps
  // at positions 32 blk + 16 s + 8 h + e (attn_vpos order within 16)
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int kv = blk * ATT_KVB + 16 * s + attn_vpos(8 * h + e), row = min(kv, t_kv - 1);
        const float x = (last && row == t_kv - 1 ? last : vf + (size_t)row * ldv)[head * ATT_DH + dt * 32 + n];
        o.x[dt][s][e] = kv < t_kv ? x : 0.0f;
      }
}
__device__ inline void att_split_v(const AttVRaw &x, AttV &o) {
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint16_t hb, lb;
        att_split(x.x[dt][s][e], hb, lb);
        o.vh[dt][s][e] = __builtin_bit_cast(_Float16, hb);
        o.vl[dt][s][e] = __builtin_bit_cast(_Float16, lb);
      }
}

// The softmax's running state of one query (a lane pair (n, n + 32) holds one):
// m, a reference score, and lsum, this lane's sum of p = 2^(log2(e) (s - m)).  m
// is the largest score seen when it was set, and moved only when a score passes it
// by more than ATT_SLACK (3.9 bits: ATT_PS p <= 2^15.9 fits f16): then the output
// and the sum are rescaled.  Any m gives the same quotient; ATT_PS p >= 2^12 at
// the row's maximum is what keeps small probabilities' f16 bits (hi + lo hold
// 2^-24 absolute, 2^-36 of the maximum): where a row's mass is on one key of little
// value, its output is made of probabilities far below the maximum, and with 2^8
// there its error was 16 times larger (a gap of 2^20: up to 4e-5 of the row).  The
// scale is a product and not 12 in the exponent, whose rounding near 12 is 2^-21 of
// every probability: rows of little spread, sums that cancel, came out at 2.2e-7 of
// their norm (100 keys; 1.2e-7 now).  s - m comes before log2(e), as a score's
// difference from one near it is exact: with log2(e) m rounded on its own, scores
// past 2^26 (|q|, |k| in the thousands) left every p at infinity or 0.  (20 heads
// at t = 1500: 42.9 us with 2^8 and log2(e) s - log2(e) m, 44.8 with the difference
// first and 12 in the exponent, 45.5 so.)  Rescaling at every new maximum moved
// some query of a tile in nearly every block (a wavefront sees 12 of them at t =
// 1500); with 3.9 bits of slack it is a few of them.
constexpr float ATT_SLACK = 3.9f / ATT_LOG2E;
constexpr float ATT_NONE = -1e30f;  // no score seen yet

// the largest score of the query's 32 kv rows (s: lane (h, n) holds query n's
// rows 8 (i / 4) + 4 h + i % 4)
__device__ inline float att_block_max(const att_v16f &s) {
  float mx = fmaxf(s[0], s[1]);
#pragma unroll
  for (int i = 2; i < 16; i += 2) mx = fmaxf(fmaxf(mx, s[i]), s[i + 1]);
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
  return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}
// does some query of the wavefront need a new m?  (the difference, which is exact
// between close scores: m + ATT_SLACK would round to more than the slack where
// scores are large)
__device__ inline bool att_moved(float m, float mx) {
  return __builtin_amdgcn_ballot_w64(mx - m > ATT_SLACK) != 0;
}
__device__ inline void att_rescale(float mx, float &m, float &lsum, att_v16f (&o)[2]) {
  const float mnew = mx - m > ATT_SLACK ? mx : m;
  const float alpha = __builtin_amdgcn_exp2f((m - mnew) * ATT_LOG2E);
  lsum *= alpha;
  o[0] *= alpha;
  o[1] *= alpha;
  m = mnew;
}
// ATT_PS p - hi, one mixed-precision FMA each (the compiler multiplies, converts
// and subtracts).  hi comes from two instructions behind the exponential, so the
// wait state that its consumers need, and that the compiler does not see here, has
// passed.
__device__ inline att_v2f att_resid(att_v2f p, att_v2h hi) {
  att_v2f r;
  const uint32_t hb = __builtin_bit_cast(uint32_t, hi);
  asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r.x) : "v"(p.x), "s"(ATT_PS), "v"(hb));
  asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r.y) : "v"(p.y), "s"(ATT_PS), "v"(hb));
  return r;
}
// scores to the P^T operands; their sum to lsum
__device__ inline void att_probs(const att_v16f &s, float m, float &lsum, att_v8h (&ph)[2], att_v8h (&pl)[2]) {
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i += 2) {
    const att_v2f p = {__builtin_amdgcn_exp2f((s[i] - m) * ATT_LOG2E),
                       __builtin_amdgcn_exp2f((s[i + 1] - m) * ATT_LOG2E)};
    s0 += p.x;
    s1 += p.y;
    // f16(p) times ATT_PS, a packed conversion and product: what f16 drops of a p
    // below 2^-14 is in the residual
    const att_v2h hi = __builtin_convertvector(p, att_v2h) * (_Float16)ATT_PS;
    const att_v2f r = att_resid(p, hi);
    const att_v2h lo = __builtin_convertvector(r, att_v2h);
    ph[i >> 3][i & 7] = hi.x, ph[i >> 3][(i & 7) + 1] = hi.y;
    pl[i >> 3][i & 7] = lo.x, pl[i >> 3][(i & 7) + 1] = lo.y;
  }
  lsum += s0 + s1;
}

// the scores of block b that query row q0 + n must not see, to -inf
__device__ inline void att_mask(att_v16f &s, int b, int h, int t_kv, bool causal, int qpos) {
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int kv = b * ATT_KVB + 8 * (i >> 2) + 4 * h + (i & 3);
    if (kv >= t_kv || (causal && kv > qpos)) s[i] = -__builtin_huge_valf();
  }
}

// XCD-aware order: workgroup id % 8 is its XCD; each XCD takes one contiguous
// range of (head, query block) in head-major order, so a head's query blocks
// share their K and v^T operands through one L2
__device__ inline int att_xcd_order(int id, int total) {
  const int per = total / 8, rem = total % 8, xcd = id % 8, slot = id / 8;
  return xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
}

// 8 values of a query row (f32, scaled by 1/8, exact) as hi and lo; rows past
// the last are zeros
__device__ inline void att_load_q(const float *__restrict__ qf, int ldq, int row, int t_q, int col, att_v8h &qh,
                                  att_v8h &ql) {
  float v[8];
  if (row < t_q) {
    const float4 *src = reinterpret_cast<const float4 *>(qf + (size_t)row * ldq + col);
    const float4 a = src[0], b = src[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.0f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    uint16_t hb, lb;
    att_split(v[e] * 0.125f, hb, lb);
    qh[e] = __builtin_bit_cast(_Float16, hb);
    ql[e] = __builtin_bit_cast(_Float16, lb);
  }
}

// Calls of more than 8 query rows.  One workgroup per (32 QT query rows,
// head); wavefront w of 4 takes kv blocks w, w + 4, ..., its operands straight
// from the split blocks (K's next block while this one's softmax runs, v^T's
// at the top of its block), with no barrier until the partial results meet in
// LDS.  A causal query row i (at absolute position t_kv - t_q + i) sees kv
// rows up to its position.
//
// Bound by the matrix cores' rate under load and the softmax beside it: with
// loads and softmax taken out, large-v3's layer (20 heads, t = 1500, 35.5
// GFLOP of f16 products) still takes 31 us, 1.15 PFLOP/s, of 45 us (two
// wavefronts of 64 queries per row group pair on 960 wavefronts took 53: one
// wavefront per SIMD, accumulators moving between register files, 16-byte
// loads).  QT = 2 keeps q's operands in LDS (232 registers, two wavefronts per
// SIMD) and loads 16 KB per 48 products; QT = 1 loads the same per 24, so it
// is for calls that 64-row tiles leave short of workgroups (each pair on one
// build, before the reference score was subtracted first): 20 heads 41 against
// 47 us, but 12 heads 34.4 against 32.9, 6 heads at t = 749 12.7 against 8.5,
// 227 rows against 1500 (20 heads) 21 against 13 us.  Eight wavefronts per
// workgroup: 46 (QT = 2) and 57 us (QT = 1).
//
// ROWS: K and V come as f32 rows (kf, vf) and are split as they are loaded, for
// calls of one or two query tiles (no split launch); the operands, and so the
// results, are the split blocks' bits.
template <int QT, bool ROWS>
__global__ __launch_bounds__(64 * ATT_NK, 2) void k_attn_tile(int t_q, int t_kv, int causal, int nqb, int total,
                                                          const float *__restrict__ qf, int ldq,
                                                          const uint16_t *__restrict__ kv, int nblk_pad,
                                                          float *__restrict__ out, int ld_out,
                                                          const float *__restrict__ kf, int ldk,
                                                          const float *__restrict__ vf, int ldv) {
  constexpr int NK = ATT_NK, QB = 32 * QT;
  constexpr bool QLDS = QT > 1;  // q's operands in LDS (64 registers' worth), else in registers
  constexpr int XLD = 36;        // floats per row of a 32-value output half in LDS
  __shared__ __align__(16) float xo[NK * QB * XLD];  // q's operands, then the partial outputs
  __shared__ float xm[NK][QB], xl[NK][QB], xinv[QB];
  static_assert(sizeof(xo) >= (size_t)QT * 8 * 1024, "q's operands");
  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = l >> 5, n = l & 31;
  const int lin = att_xcd_order(blockIdx.x, total);
  const int head = lin / nqb, q0 = (lin % nqb) * QB;
  const int off = t_kv - t_q;  // absolute position of query row 0
  const int kv_end = causal ? min(t_kv, off + q0 + QB) : t_kv;
  const int nblk = (kv_end + ATT_KVB - 1) / ATT_KVB;
  const uint16_t *base = kv + (size_t)head * nblk_pad * ATT_BLK + l * 8;

  AttK kk;
  AttV vv;
  AttKRaw kr;
  AttVRaw vr;
  auto load_k = [&](int blk) __attribute__((always_inline)) {
    if constexpr (ROWS) att_load_k_raw(kf, ldk, t_kv, head, blk, h, n, kr);
    else att_load_k(base + (size_t)blk * ATT_BLK, kk);
  };
  auto load_v = [&](int blk) __attribute__((always_inline)) {
    if constexpr (ROWS) att_load_v_raw(vf, ldv, t_kv, head, blk, h, n, vr);
    else att_load_v(base + (size_t)blk * ATT_BLK, vv);
  };
  if (wv < nblk) load_k(wv);

  // q's operands: fragment (qt, s), hi then lo
  att_v8h qh[QLDS ? 1 : 4], ql[QLDS ? 1 : 4];
  uint16_t *qs = reinterpret_cast<uint16_t *>(xo) + l * 8;
  if constexpr (QLDS) {
#pragma unroll
    for (int f = wv; f < 4 * QT; f += NK) {
      att_v8h a, b;
      att_load_q(qf, ldq, q0 + (f >> 2) * 32 + n, t_q, head * ATT_DH + 8 * h + 16 * (f & 3), a, b);
      *reinterpret_cast<uint4 *>(qs + 2 * f * 512) = __builtin_bit_cast(uint4, a);
      *reinterpret_cast<uint4 *>(qs + (2 * f + 1) * 512) = __builtin_bit_cast(uint4, b);
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      att_load_q(qf, ldq, q0 + n, t_q, head * ATT_DH + 8 * h + 16 * s, qh[s], ql[s]);
  }

  att_v16f o[QT][2];  // O^T
  float m[QT], lsum[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    o[qt][0] = (att_v16f){};
    o[qt][1] = (att_v16f){};
    m[qt] = ATT_NONE;
    lsum[qt] = 0.0f;
  }
  int b = wv;
  att_v16f s[QT];
  float mx[QT];
  // block b's scores and maxima, K's next block requested behind them
  auto scores = [&]() __attribute__((always_inline)) {
    // (an offset the compiler cannot see through: it would keep all of q's
    // operands in registers across the loop, and spill)
    int qo = l * 8;
    if constexpr (QLDS) asm volatile("" : "+v"(qo));
    if constexpr (ROWS) att_split_k(kr, b * ATT_KVB + n < t_kv, kk);
    const uint16_t *qp = reinterpret_cast<const uint16_t *>(xo) + qo;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      s[qt] = (att_v16f){};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (QLDS)
          att_mma3(kk.kh[k], kk.kl[k], att_ld(qp + 2 * (4 * qt + k) * 512), att_ld(qp + (2 * (4 * qt + k) + 1) * 512),
                   s[qt]);
        else
          att_mma3(kk.kh[k], kk.kl[k], qh[k], ql[k], s[qt]);
      }
    }
    load_k(min(b + NK, nblk - 1));
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int tq0 = q0 + qt * 32;
      if ((b + 1) * ATT_KVB > t_kv || (causal && (b + 1) * ATT_KVB - 1 > off + tq0))
        att_mask(s[qt], b, h, t_kv, causal, off + tq0 + n);
      mx[qt] = att_block_max(s[qt]);
    }
  };
  // Two loops, so that the common path has no rescale to merge with: beside
  // one the compiler copied all of O^T in every block (50 against 47 us with
  // QT = 1 at 20 heads)
  if (b < nblk) {
    load_v(b);
    scores();
    for (;;) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) att_rescale(mx[qt], m[qt], lsum[qt], o[qt]);
      bool moved;
      do {
        if constexpr (ROWS) att_split_v(vr, vv);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          att_v8h ph[2], pl[2];
          att_probs(s[qt], m[qt], lsum[qt], ph, pl);
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) att_mma3(vv.vh[dt][k], vv.vl[dt][k], ph[k], pl[k], o[qt][dt]);
        }
        b += NK;
        if (b >= nblk) break;
        load_v(b);
        scores();
        moved = false;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) moved = moved || att_moved(m[qt], mx[qt]);
      } while (!moved);
      if (b >= nblk) break;
    }
  }

  // the NK partial states meet: every wavefront's output scaled to the common
  // maximum, summed in wavefront order, divided by the common sum
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum[qt]), __float_as_uint(lsum[qt]), false, false);
    const float lt = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    if (h == 0) {
      xm[wv][qt * 32 + n] = m[qt];
      xl[wv][qt * 32 + n] = lt;
    }
  }
  __syncthreads();  // every wavefront is done with q's operands too
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float mu = ATT_NONE;
#pragma unroll
    for (int w = 0; w < NK; ++w) mu = fmaxf(mu, xm[w][qt * 32 + n]);
    if (wv == 0 && h == 0) {
      float den = 0.0f;
#pragma unroll
      for (int w = 0; w < NK; ++w) den += xl[w][qt * 32 + n] * __builtin_amdgcn_exp2f((xm[w][qt * 32 + n] - mu) * ATT_LOG2E);
      xinv[qt * 32 + n] = 1.0f / (den * ATT_PS);
    }
    const float sc = __builtin_amdgcn_exp2f((m[qt] - mu) * ATT_LOG2E);
    o[qt][0] *= sc;
    o[qt][1] *= sc;
  }
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    if (dt) __syncthreads();  // the first half has been read
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4 *>(&xo[((wv * QT + qt) * 32 + n) * XLD + 8 * g + 4 * h]) =
            make_float4(o[qt][dt][4 * g], o[qt][dt][4 * g + 1], o[qt][dt][4 * g + 2], o[qt][dt][4 * g + 3]);
    __syncthreads();
#pragma unroll
    for (int c = threadIdx.x; c < QB * 8; c += 64 * NK) {
      const int row = c >> 3, c4 = c & 7;
      float4 y = *reinterpret_cast<const float4 *>(&xo[row * XLD + 4 * c4]);
#pragma unroll
      for (int w = 1; w < NK; ++w) {
        const float4 x = *reinterpret_cast<const float4 *>(&xo[(w * QB + row) * XLD + 4 * c4]);
        y.x += x.x, y.y += x.y, y.z += x.z, y.w += x.w;
      }
      const float inv = xinv[row];
      if (q0 + row < t_q)
        *reinterpret_cast<float4 *>(out + (size_t)(q0 + row) * ld_out + head * ATT_DH + dt * 32 + 4 * c4) =
            make_float4(y.x * inv, y.y * inv, y.z * inv, y.w * inv);
    }
  }
}

// Calls of at most 8 query rows, or of at most 64 against many keys
// (attn_route).  Workgroup (blockIdx.x, blockIdx.y) = (32 query rows, head); wavefront w takes kv
// blocks w, w + 2, ...; a causal query row i (at absolute position t_kv - t_q
// + i) sees kv rows up to its position.
//
// Split kv (few query blocks, e.g. one decoding step): with part != NULL,
// workgroup z of gridDim.z takes the z-th run of the kv blocks and writes
// its unnormalized O (2^12-scaled), running maximum and sum to
// part; k_attn_combine merges the runs.
//
// The queries come as f32 rows and are scaled and split here; K and v^T as
// split blocks (P: the decoder's cross-attention keeps them).
// ROWS: K and V come as f32 rows too (kf, vf) and are split here as well (P's
// blocks are unused): a decoding step's self-attention over its cache then
// needs no split launch; the operands are the blocks' values, so the results
// are the same bits.
// The scalars and row pointers lead the arguments: the first 14 dwords
// arrive in SGPRs when the waves start (kernarg preloading), so a decoding
// step's attention requests its rows without first reading the argument
// block; the planes (P) follow.  The grid comes as arguments too (gridDim
// is read from the argument block): nx = gridDim.x, gw = causal | gridDim.z
// << 1 | gridDim.y << 8.
// (defined with the decode GEMV: a block of 8 lanes x 4 values as row i's
// activation record of block bl)
__device__ void attn_block_records(uint8_t *rec, int i, int bl, int lt, int mr, float4 x, int off, bool write);

// BEAMS (with ROWS): several beams' self-attention, one query row per
// (beam, head) plane, plane b * n_head + h; its q row is qf + b n + 64 h, its
// K and V rows beam b's caches C.k[b], C.v[b] except the newest (row
// t_kv - 1), which comes from the step's new rows kf, vf [beams][n] and is
// stored into the caches at that row (by the kv split's first run).
// rec (BEAMS, no kv split): also the output rows' activation records for
// the next product.  rec_hd = heads per beam | offset term << 8 | beams << 16.
template <bool ROWS, bool BEAMS = false>
__global__ __launch_bounds__(128) void k_attn(int t_q, int t_kv, int gw, int nx, const float *__restrict__ qf,
                                              int ldq, const float *__restrict__ kf, int ldk,
                                              const float *__restrict__ vf, int ldv, float *__restrict__ out,
                                              int ld_out, float *__restrict__ part, AttnPlanes P,
                                              uint8_t *__restrict__ rec, int rec_hd, BeamCaches C) {
  const int causal = gw & 1, gz = (gw >> 1) & 127, gy = gw >> 8;
  constexpr int QB = 32;  // query rows per workgroup
  constexpr float NEG_INF = -__builtin_huge_valf();
  __shared__ __align__(16) float xo[QB * (ATT_DH + 4)];  // partial O^T exchange, then the output tile
  __shared__ float xm[64], xl[64];
  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = l >> 5, n = l & 31;
  const int lin = att_xcd_order(blockIdx.y * nx + blockIdx.x, nx * gy);
  const int head = lin / nx, q0 = (lin % nx) * QB;
  const int off = t_kv - t_q;  // absolute position of query row 0
  const int kv_end = causal ? min(t_kv, off + q0 + QB) : t_kv;
  const int nblk_all = (kv_end + ATT_KVB - 1) / ATT_KVB;
  const int cs = (nblk_all + gz - 1) / gz;                     // blocks per split
  const int b_begin = min(nblk_all, (int)blockIdx.z * cs);
  const int nblk = min(nblk_all, b_begin + cs);               // this workgroup: blocks [b_begin, nblk)

  att_v8h qh[4], ql[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) att_load_q(qf, ldq, q0 + n, t_q, head * ATT_DH + 8 * h + 16 * s, qh[s], ql[s]);
  att_v16f o[2] = {(att_v16f){}, (att_v16f){}};  // O^T
  float m = NEG_INF, lsum = 0.0f;

  // K one block ahead; V is loaded at the top of its block and first used
  // after the scores and the softmax
  AttK cur, nxt;
  AttV vb;
  AttKRaw kr_cur, kr_nxt;  // ROWS: f32 K rows, split when their block comes
  AttVRaw vr;
  // this plane's K and V rows (BEAMS: its beam's caches and new row)
  const float *kfp = kf, *vfp = vf, *klast = nullptr, *vlast = nullptr;
  const uint16_t *base = P.kv + (size_t)head * (P.tkv_pad / ATT_KVB) * ATT_BLK + l * 8;
  int hkv = head;
  if constexpr (BEAMS) {
    const int hpb = rec_hd & 255, bb = head / hpb;
    hkv = head - bb * hpb;
    kfp = C.k[bb];
    vfp = C.v[bb];
    klast = kf + (size_t)bb * ldk;
    vlast = vf + (size_t)bb * ldv;
    if (blockIdx.z == 0) {  // the new row into the caches (read from kf / vf in this launch)
      const int t = threadIdx.x & 63;
      if (threadIdx.x < 64) C.k[bb][(size_t)(t_kv - 1) * ldk + hkv * ATT_DH + t] = klast[hkv * ATT_DH + t];
      else C.v[bb][(size_t)(t_kv - 1) * ldv + hkv * ATT_DH + t] = vlast[hkv * ATT_DH + t];
    }
  }
  if (b_begin + wv < nblk) {
    if constexpr (ROWS) att_load_k_raw(kfp, ldk, t_kv, hkv, b_begin + wv, h, n, kr_cur, klast);
    else att_load_k(base + (size_t)(b_begin + wv) * ATT_BLK, cur);
  }
  for (int b = b_begin + wv; b < nblk; b += 2) {
    if constexpr (ROWS) {
      att_load_v_raw(vfp, ldv, t_kv, hkv, b, h, n, vr, vlast);
      if (b + 2 < nblk) att_load_k_raw(kfp, ldk, t_kv, hkv, b + 2, h, n, kr_nxt, klast);
      att_split_k(kr_cur, b * ATT_KVB + n < t_kv, cur);
    } else {
      att_load_v(base + (size_t)b * ATT_BLK, vb);
      if (b + 2 < nblk) att_load_k(base + (size_t)(b + 2) * ATT_BLK, nxt);
    }
    att_v16f s = (att_v16f){};
#pragma unroll
    for (int k = 0; k < 4; ++k) att_mma3(cur.kh[k], cur.kl[k], qh[k], ql[k], s);
    if constexpr (ROWS) att_split_v(vr, vb);
    if ((b + 1) * ATT_KVB > t_kv || (causal && (b + 1) * ATT_KVB - 1 > off + q0))
      att_mask(s, b, h, t_kv, causal, off + q0 + n);
    att_v8h ph[2], pl[2];
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float mnew = fmaxf(m, mx);
    const float mu = mnew == NEG_INF ? 0.0f : mnew;  // a query with nothing visible yet
    float ps = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = __builtin_amdgcn_exp2f((s[i] - mu) * ATT_LOG2E);
      ps += p;
      // P enters the products as 2^12 p, so that small probabilities keep
      // their f16 bits; the output is divided by 2^12 lsum at the end
      const float p12 = p * ATT_PS;
      const _Float16 ph1 = (_Float16)p12;
      ph[i >> 3][i & 7] = ph1;
      pl[i >> 3][i & 7] = (_Float16)(p12 - (float)ph1);
    }
    // rescale only when some query's maximum moved
    if (__builtin_amdgcn_ballot_w64(mnew != m)) {
      const float alpha = __builtin_amdgcn_exp2f((m - mu) * ATT_LOG2E);
      lsum *= alpha;
      o[0] *= alpha;
      o[1] *= alpha;
    }
    m = mnew;
    lsum += ps;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int k = 0; k < 2; ++k) att_mma3(vb.vh[dt][k], vb.vl[dt][k], ph[k], pl[k], o[dt]);
    if constexpr (ROWS) kr_cur = kr_nxt;
    else cur = nxt;
  }

  // wavefront 1 hands its partial state to wavefront 0
  if (wv == 1) {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) xo[(dt * 16 + i) * 64 + l] = o[dt][i];
    xm[l] = m;
    xl[l] = lsum;
  }
  __syncthreads();
  if (wv == 0) {
    const float m1 = xm[l], l1 = xl[l];
    const float mm = fmaxf(m, m1);
    const float mu = mm == NEG_INF ? 0.0f : mm;
    const float s0 = __builtin_amdgcn_exp2f((m - mu) * ATT_LOG2E), s1 = __builtin_amdgcn_exp2f((m1 - mu) * ATT_LOG2E);
    float lt = lsum * s0 + l1 * s1;
    lt += __shfl_xor(lt, 32);
    const float inv = part ? 1.0f : 1.0f / (lt * ATT_PS);
    if (part && h == 0 && q0 + n < t_q) {
      const size_t pr = ((size_t)blockIdx.z * gy + head) * P.tq_pad + q0 + n;
      float *pml = part + (size_t)gz * gy * P.tq_pad * ATT_DH;
      pml[2 * pr] = mm;
      pml[2 * pr + 1] = lt;
    }
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = (o[dt][i] * s0 + xo[(dt * 16 + i) * 64 + l] * s1) * inv;
  }
  __syncthreads();
  // the output tile [32 queries][64 d] through LDS, then row-contiguous stores
  constexpr int LD = ATT_DH + 4;
  if (wv == 0) {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4 *>(&xo[n * LD + dt * 32 + 8 * g + 4 * h]) =
            make_float4(o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]);
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < QB * 16 / 128; ++it) {
    const int c = it * 128 + (int)threadIdx.x;
    const int row = c >> 4, c4 = c & 15;
    if (q0 + row < t_q) {
      float *dst = part ? part + (((size_t)blockIdx.z * gy + head) * P.tq_pad + q0 + row) * ATT_DH + 4 * c4
                        : out + (size_t)(q0 + row) * ld_out + head * ATT_DH + 4 * c4;
      *reinterpret_cast<float4 *>(dst) = *reinterpret_cast<const float4 *>(&xo[row * LD + 4 * c4]);
    }
    // the one query row is threads 0-15 of the first pass: each 8 of them
    // one 32-column block (every lane of the wavefront quantizes its values)
    if (it == 0 && rec && threadIdx.x < 64) {
      const int hpb = rec_hd & 255;
      attn_block_records(rec, head / hpb, (head % hpb) * 2 + (c4 >> 3), c4 & 7, rec_hd >> 16,
                         *reinterpret_cast<const float4 *>(&xo[row * LD + 4 * c4]), (rec_hd >> 8) & 255,
                         q0 + row < t_q && row == 0);
    }
  }
}

// Merge nsplit runs of k_attn: out = sum_z O_z e^(m_z - m) / (2^12 sum_z l_z
// e^(m_z - m)), m the largest run maximum (runs that saw nothing have
// m = -inf and weigh 0).  One thread per (query, head, d).
// (defined with the decode GEMV: one query row's block of the output as the
// next product's activation record)
__device__ void combine_records(uint8_t *rec, int row, int col, int mr, float x, int off);

// With rec: also each query row's 32-column blocks of the output as
// activation records of the next product (its offset term `rec_off`), for
// 2-8 query rows; a wavefront holds one (row, head), two blocks.
__global__ __launch_bounds__(256) void k_attn_combine(const float *__restrict__ part, int nsplit, int n_head,
                                                      int tq_pad, int t_q, float *__restrict__ out, int ld_out,
                                                      uint8_t *__restrict__ rec, int rec_off) {
  constexpr float NEG_INF = -__builtin_huge_valf();
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)t_q * n_head * ATT_DH) return;
  const int d = (int)(idx % ATT_DH);
  const int head = (int)((idx / ATT_DH) % n_head), q = (int)(idx / ((size_t)ATT_DH * n_head));
  const float *pml = part + (size_t)nsplit * n_head * tq_pad * ATT_DH;
  // every run's maximum, sum and output value requested at once (one memory
  // round trip), then folded in run order
  float mz[ATT_MAX_SPLIT], lz[ATT_MAX_SPLIT], oz[ATT_MAX_SPLIT];
#pragma unroll
  for (int z = 0; z < ATT_MAX_SPLIT; ++z) {
    mz[z] = NEG_INF, lz[z] = 0.0f, oz[z] = 0.0f;
    if (z < nsplit) {
      const size_t pr = ((size_t)z * n_head + head) * tq_pad + q;
      mz[z] = pml[2 * pr];
      lz[z] = pml[2 * pr + 1];
      oz[z] = part[pr * ATT_DH + d];
    }
  }
  float mx = NEG_INF;
#pragma unroll
  for (int z = 0; z < ATT_MAX_SPLIT; ++z) mx = fmaxf(mx, mz[z]);
  const float mu = mx == NEG_INF ? 0.0f : mx;
  float num = 0.0f, den = 0.0f;
#pragma unroll
  for (int z = 0; z < ATT_MAX_SPLIT; ++z) {
    const float w = __builtin_amdgcn_exp2f((mz[z] - mu) * ATT_LOG2E);
    if (z < nsplit && w > 0.0f) {  // a run that saw no key holds no output
      num += oz[z] * w;
      den += lz[z] * w;
    }
  }
  const float y = num / (den * ATT_PS);
  out[(size_t)q * ld_out + head * ATT_DH + d] = y;
  if (rec) combine_records(rec, q, head * ATT_DH + d, t_q, y, rec_off);  // whole wavefronts (uniform)
}

#endif  // __HIPCC__

}  // namespace rw
