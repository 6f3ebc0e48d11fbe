// rw_dec.hpp -- the small element-wise kernels of the decoder step (device
// code): the token + position embedding, a float32 layernorm (with the
// residual add of src/decoder.rs:168-170, 191-193 and mlp_block folded in
// front of it) and GELU.  The products and attention are the kernels of
// rw_kernels.hpp and rw_attn.hpp.
#pragma once
#include <stdint.h>

#include "rw_layout.hpp"

namespace rw {

#if defined(__HIPCC__)

// the token ids of a step of at most EMBED_IDS rows, passed by value: a copy of
// 4 to 32 bytes to the device was a launch of its own, 4 us and the gaps beside
// it
constexpr int EMBED_IDS = 8;
struct EmbedIds {
  int id[EMBED_IDS];
};

// x[i] = token_embedding.row_f32(tok[i]) + positional[n_past + i * pos_step]
// (src/decoder.rs:122-135): the quantized row dequantized as d * q + m (two
// roundings), then the position added.  pos_step is 1 for a prompt's
// consecutive tokens and 0 for one token of each of several beams.  One thread
// per element, blockIdx.y the token; tok NULL: the ids come in `ids`.
template <int DT>
__global__ __launch_bounds__(256) void k_embed(WeightView w, const int *__restrict__ tok, EmbedIds ids,
                                               const float *__restrict__ pos, int n_past, int pos_step,
                                               float *__restrict__ x) {
  const size_t n = (size_t)w.nb * QK, c = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  const int i = blockIdx.y, bl = (int)(c / QK);
  const int j = tok ? tok[i] : ids.id[i & (EMBED_IDS - 1)];
  const int g = j / RG, r = j % RG;
  const size_t si = sc_index(w, g, bl, r);
  const float d = h2f_exact(w.d[si]);
  const float m = has_min(DT) ? h2f_exact(w.m[si]) : 0.0f;
  x[(size_t)i * n + c] = __fadd_rn(__fadd_rn(__fmul_rn(d, (float)weight_q<DT>(w, g, bl, r, (int)(c % QK))), m),
                                   pos[(size_t)(n_past + i * pos_step) * n + c]);
}

// y = layernorm(x) row by row (src/tensor.rs:274-287): mean, mean of squared
// deviations, inv = 1 / sqrt(var + 1e-5), (x - mean) * inv * w + b; the sums
// in tree order.  One workgroup per row.  With r != NULL the residual add
// comes first: x += r (stored back), then y = layernorm(x).
constexpr int LN_REG = 8;
__global__ __launch_bounds__(256) void k_layernorm(float *__restrict__ x, int n, const float *__restrict__ w,
                                                   const float *__restrict__ b, float *__restrict__ y,
                                                   const float *__restrict__ r) {
  __shared__ float part[2][4];
  const int row = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
  float *xr = x + (size_t)row * n;
  if (r) {
    const float *rr = r + (size_t)row * n;
    for (int c = t; c < n; c += 256) xr[c] = xr[c] + rr[c];
    __syncthreads();
  }
  auto reduce = [&](float v, int slot) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o);
    if (lane == 0) part[slot][wv] = v;
    __syncthreads();
    return (part[slot][0] + part[slot][1]) + (part[slot][2] + part[slot][3]);
  };
  float *yr = y + (size_t)row * n;
  // rows of at most 256 LN_REG values stay in registers (one read of the row;
  // the same sums in the same order)
  if (n <= 256 * LN_REG) {
    float v[LN_REG], s = 0.0f;
#pragma unroll
    for (int u = 0; u < LN_REG; ++u) v[u] = t + 256 * u < n ? xr[t + 256 * u] : 0.0f;
#pragma unroll
    for (int u = 0; u < LN_REG; ++u)
      if (t + 256 * u < n) s += v[u];
    const float mean = __fdiv_rn(reduce(s, 0), (float)n);
    s = 0.0f;
#pragma unroll
    for (int u = 0; u < LN_REG; ++u)
      if (t + 256 * u < n) {
        const float d = v[u] - mean;
        s += d * d;
      }
    const float var = __fdiv_rn(reduce(s, 1), (float)n);
    const float inv = __fdiv_rn(1.0f, __fsqrt_rn(var + 1e-5f));
#pragma unroll
    for (int u = 0; u < LN_REG; ++u)
      if (t + 256 * u < n) yr[t + 256 * u] = (v[u] - mean) * inv * w[t + 256 * u] + b[t + 256 * u];
    return;
  }
  float s = 0.0f;
  for (int c = t; c < n; c += 256) s += xr[c];
  const float mean = __fdiv_rn(reduce(s, 0), (float)n);
  s = 0.0f;
  for (int c = t; c < n; c += 256) {
    const float d = xr[c] - mean;
    s += d * d;
  }
  const float var = __fdiv_rn(reduce(s, 1), (float)n);
  const float inv = __fdiv_rn(1.0f, __fsqrt_rn(var + 1e-5f));
  for (int c = t; c < n; c += 256) yr[c] = (xr[c] - mean) * inv * w[c] + b[c];
}

// h = gelu(h) (src/tensor.rs:289-305; rw_kernels.hpp's gelu)
__global__ __launch_bounds__(256) void k_gelu(float *__restrict__ h, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) h[t] = gelu(h[t]);
}

constexpr int TOPK_MAX = 16;  // candidates per row of the top-k kernels

// Block-wide reductions of one value per thread (256 threads, 4 wavefronts)
__device__ inline float block_fmax(float v, float *scratch) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v = fmaxf(v, __shfl_xor(v, o));
  __syncthreads();  // scratch may hold the previous reduction's values
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3]));
}
__device__ inline float block_fsum(float v, float *scratch) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return (scratch[0] + scratch[1]) + (scratch[2] + scratch[3]);
}
// (v, i) beats (bv, bi): larger v, or equal v and smaller i
__device__ inline bool topk_before(float v, int i, float bv, int bi) { return v > bv || (v == bv && i < bi); }

// log_softmax of each row (src/transcribe.rs:482-486: the maximum, lse =
// max + ln(sum exp(v - max)), lp = v - lse) and its top_k
// (src/transcribe.rs:672-685).  top_k scans the log-probs in id order,
// skips exactly -inf, and inserts (lp, id) ahead of every entry with an
// equal log-prob while the list has room or lp beats its last entry, then
// truncates to k.  With v* the k-th largest log-prob and g the number of
// larger ones, that keeps every entry above v*, and of the entries equal to
// v* those admitted (fewer than k entries >= v* precede them in id order)
// minus the oldest ones pushed out later: the last k - g admitted.  The
// list runs by log-prob, equal ones later id first.
// Three launches over chunks of TOPK_CHUNK logits (rows x chunks
// workgroups): k_topk_stats (each chunk's maximum and sum of exp(v - max)),
// k_topk_chunk (the row's lse from those partials, in one fixed order, then
// the chunk's first 2k - 1 entries in the order (lp desc, id asc)) and
// k_topk_merge (per row, v* and g from the chunks' picks, the admitted
// entries equal to v* in id order, and the list in the reference's order).
// A chunk holds at most g <= k - 1 entries above v*, so its first 2k - 1
// picks hold those and its first k entries equal to v*, which include every
// one of them the scan can admit: the merge is exact.
// A row holding NaN or +inf, or only -inf, has a NaN lse (as the reference
// computes it), so every log-prob is NaN; the scan then admits ids
// 0 .. k - 1, each ahead of the last, and keeps them with NaN log-probs.
// The sum runs in tree order, so lse (and every lp) can differ from the
// reference's sequential sum in its last bit.
constexpr int TOPK_CHUNK = 2048;  // logits per workgroup (8 per thread)
constexpr int TOPK_MAX_CHUNKS = 64;

__global__ __launch_bounds__(256) void k_topk_stats(const float *__restrict__ logits, int n, float *__restrict__ pm,
                                                    float *__restrict__ ps) {
  __shared__ float sf[4];
  const int c = blockIdx.x, row = blockIdx.y, nc = gridDim.x, t = threadIdx.x;
  const float *x = logits + (size_t)row * n;
  const int e0 = c * TOPK_CHUNK, e1 = min(n, e0 + TOPK_CHUNK);
  float v[TOPK_CHUNK / 256];
  float mx = -__builtin_huge_valf();
#pragma unroll
  for (int j = 0; j < TOPK_CHUNK / 256; ++j) {
    const int e = e0 + j * 256 + t;
    v[j] = e < e1 ? x[e] : -__builtin_huge_valf();
    mx = fmaxf(mx, v[j]);
  }
  mx = block_fmax(mx, sf);
  // an all -inf chunk (suppressed tokens) adds nothing; NaN, and +inf
  // (inf - inf), make the sum NaN as in the reference
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < TOPK_CHUNK / 256; ++j)
    if (e0 + j * 256 + t < e1 && v[j] != -__builtin_huge_valf()) sum += expf(v[j] - mx);
  sum = block_fsum(sum, sf);
  if (t == 0) {
    pm[(size_t)row * nc + c] = mx;
    ps[(size_t)row * nc + c] = sum;
  }
}

// A wavefront's largest value and smallest int, by DPP row moves (a lane
// without a source keeps its own value), the same in every lane.
template <int CTRL, int ROWS = 0xf>
__device__ inline int topk_dpp(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false);
}
__device__ inline float wave_fmax(float v) {
  auto up = [&](int o) __attribute__((always_inline)) { v = fmaxf(v, __int_as_float(o)); };
  up(topk_dpp<0x111>(__float_as_int(v)));       // row_shr 1, 2, 4, 8
  up(topk_dpp<0x112>(__float_as_int(v)));
  up(topk_dpp<0x114>(__float_as_int(v)));
  up(topk_dpp<0x118>(__float_as_int(v)));
  up(topk_dpp<0x142, 0xa>(__float_as_int(v)));  // row_bcast 15 into rows 1 and 3
  up(topk_dpp<0x143, 0xc>(__float_as_int(v)));  // row_bcast 31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ inline int wave_imin(int v) {
  v = min(v, topk_dpp<0x111>(v));
  v = min(v, topk_dpp<0x112>(v));
  v = min(v, topk_dpp<0x114>(v));
  v = min(v, topk_dpp<0x118>(v));
  v = min(v, topk_dpp<0x142, 0xa>(v));
  v = min(v, topk_dpp<0x143, 0xc>(v));
  return __builtin_amdgcn_readlane(v, 63);
}

// the row's lse from its chunks' (maximum, sum) pairs: the maximum of the
// maxima, then sum_c s_c exp(m_c - M) in chunk order (one chunk per lane, at
// most 64; every wavefront computes it).  A chunk of NaNs only (maximum -inf,
// sum NaN) still makes it NaN, and so does a row of -inf only, whose reference
// maximum -inf gives -inf - -inf = NaN.
__device__ inline float topk_lse(const float *pm, const float *ps, int nc) {
  const int l = threadIdx.x & 63;
  const float m = l < nc ? pm[l] : -__builtin_huge_valf(), s = l < nc ? ps[l] : 0.0f;
  const float M = wave_fmax(m);
  if (M == -__builtin_huge_valf()) return __builtin_nanf("");
  const float term = s * expf(m - M);
  const uint64_t live = __builtin_amdgcn_ballot_w64(m > -__builtin_huge_valf() || s != s);
  float S = 0.0f;
  for (int c = 0; c < nc; ++c) {
    const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(term), c));
    if (live >> c & 1) S += t;
  }
  return M + logf(S);
}

// k rounds over the values the lanes of one wavefront hold (PER each): each
// round picks the wavefront's first entry after the previous pick in the
// selection order (lp desc, id asc); picks go to (ov, oi)[0, k), padded with
// (-inf, INT32_MAX).  Returns the number picked (uniform).
template <int PER>
__device__ inline int topk_rounds(const float (&lp)[PER], const int (&id)[PER], int k, float *ov, int *oi) {
  constexpr float NEG_INF = -__builtin_huge_valf();
  const bool first = (threadIdx.x & 63) == 0;
  float pv = __builtin_huge_valf();
  int pi = -1, got = 0;
  for (int r = 0; r < k; ++r) {
    float bv = NEG_INF;
    int bi = INT32_MAX;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lp[j] > NEG_INF && topk_before(pv, pi, lp[j], id[j]) && topk_before(lp[j], id[j], bv, bi))
        bv = lp[j], bi = id[j];
    const float mv = wave_fmax(bv);
    const int mi = wave_imin(bv == mv ? bi : INT32_MAX);
    if (mi == INT32_MAX) break;  // no candidate left (uniform)
    if (first) ov[r] = mv, oi[r] = mi;
    pv = mv, pi = mi;
    got = r + 1;
  }
  if (first)
    for (int r = got; r < k; ++r) ov[r] = NEG_INF, oi[r] = INT32_MAX;
  return got;
}

// The first k entries of the values that the 256 threads hold, to (ov, oi) by
// wavefront 0 (the return value is wavefront 0's): each wavefront's first k
// into LDS without a barrier, then wavefront 0's rounds over those 4 k.  The
// entries, and their order, are the block's (a barrier-free round takes about
// 0.15 us; block-wide arg-max rounds, two barriers and 12 lane shuffles each,
// took 18 us per launch over 26 chunks of 5 rows with k = 5, and 12 us in the
// merge).
constexpr int TOPK_CAND = 2 * TOPK_MAX - 1;  // entries kept per chunk at most
template <int PER, int KMAX>
__device__ inline int topk_block(const float (&lp)[PER], const int (&id)[PER], int k, float *ov, int *oi,
                                 float (&sv)[4 * KMAX], int (&si)[4 * KMAX]) {
  constexpr int PW = (4 * KMAX + 63) / 64;
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  topk_rounds<PER>(lp, id, k, sv + wv * k, si + wv * k);
  __syncthreads();
  if (wv) return 0;
  float v[PW];
  int i[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const int e = j * 64 + l;
    v[j] = e < 4 * k ? sv[e] : -__builtin_huge_valf();
    i[j] = e < 4 * k ? si[e] : INT32_MAX;
  }
  return topk_rounds<PW>(v, i, k, ov, oi);
}

__global__ __launch_bounds__(256) void k_topk_chunk(const float *__restrict__ logits, int n, int k,
                                                    const float *__restrict__ pm, const float *__restrict__ ps,
                                                    float *__restrict__ cv, int *__restrict__ ci) {
  __shared__ float sv[4 * TOPK_CAND];
  __shared__ int si[4 * TOPK_CAND];
  const int c = blockIdx.x, row = blockIdx.y, nc = gridDim.x, t = threadIdx.x;
  const float lse = topk_lse(pm + (size_t)row * nc, ps + (size_t)row * nc, nc);
  const float *x = logits + (size_t)row * n;
  const int e0 = c * TOPK_CHUNK, e1 = min(n, e0 + TOPK_CHUNK);
  constexpr int PER = TOPK_CHUNK / 256;
  float lp[PER];
  int id[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = e0 + j * 256 + t;
    id[j] = e;
    lp[j] = e < e1 ? x[e] - lse : -__builtin_huge_valf();  // NaN stays NaN and is never picked
  }
  const int cand = 2 * k - 1;
  const size_t o = ((size_t)row * nc + c) * cand;
  topk_block<PER, TOPK_CAND>(lp, id, cand, cv + o, ci + o, sv, si);
}

// the block-wide smallest of one int per thread
__device__ inline int block_imin(int v, int *scratch) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v = min(v, __shfl_xor(v, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return min(min(scratch[0], scratch[1]), min(scratch[2], scratch[3]));
}

__global__ __launch_bounds__(256) void k_topk_merge(int nc, int k, int n, const float *__restrict__ pm,
                                                    const float *__restrict__ ps, const float *__restrict__ cv,
                                                    const int *__restrict__ ci, uint32_t *__restrict__ ids,
                                                    float *__restrict__ lps) {
  constexpr float NEG_INF = -__builtin_huge_valf();
  __shared__ float sv[4 * TOPK_MAX];
  __shared__ int si[4 * TOPK_MAX];
  __shared__ int ri[4], n_got;
  __shared__ float pick_v[TOPK_MAX];
  __shared__ int pick_i[TOPK_MAX];
  __shared__ int adm[TOPK_MAX];
  const int row = blockIdx.x, t = threadIdx.x;
  uint32_t *oid = ids + (size_t)row * k;
  float *olp = lps + (size_t)row * k;
  const float lse = topk_lse(pm + (size_t)row * nc, ps + (size_t)row * nc, nc);
  if (lse != lse) {  // every log-prob NaN: ids min(k, n) - 1 .. 0
    const int kk = min(k, n);
    if (t < k) {
      oid[t] = t < kk ? (uint32_t)(kk - 1 - t) : 0xFFFFFFFFu;
      olp[t] = t < kk ? __builtin_nanf("") : NEG_INF;
    }
    return;
  }
  constexpr int PER = (TOPK_MAX_CHUNKS * TOPK_CAND + 255) / 256;
  float lp[PER];
  int id[PER];
  const int total = nc * (2 * k - 1);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = j * 256 + t;
    lp[j] = e < total ? cv[(size_t)row * total + e] : NEG_INF;
    id[j] = e < total ? ci[(size_t)row * total + e] : INT32_MAX;
  }
  // the k first in the order (lp desc, id asc): their values are the k
  // largest log-probs, so the last is v*
  const int got0 = topk_block<PER, TOPK_MAX>(lp, id, k, pick_v, pick_i, sv, si);
  if (t == 0) n_got = got0;
  __syncthreads();
  const int got = n_got;
  int g = got, a = 0;
  if (got == k) {
    const float vs = pick_v[k - 1];
    g = 0;
    while (g < k && pick_v[g] > vs) ++g;
    // the entries equal to v* in id order, while fewer than k entries >= v*
    // precede them (i earlier ones equal to v*, plus the larger ones before)
    int prev = -1;
    for (int i = 0; i < k; ++i) {
      int best = INT32_MAX;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (lp[j] == vs && id[j] > prev && id[j] < best) best = id[j];
      best = block_imin(best, ri);
      if (best == INT32_MAX) break;  // uniform
      int before = i;
      for (int r = 0; r < g; ++r) before += pick_i[r] < best;
      if (before >= k) break;
      if (t == 0) adm[a] = best;
      ++a;
      prev = best;
    }
    __syncthreads();
  }
  if (t == 0) {
    // the entries above v* (all of them), equal log-probs later id first
    for (int x = 1; x < g; ++x)
      for (int y = x; y > 0 && pick_v[y] == pick_v[y - 1] && pick_i[y] > pick_i[y - 1]; --y) {
        const int ti = pick_i[y];
        pick_i[y] = pick_i[y - 1], pick_i[y - 1] = ti;
      }
    for (int r = 0; r < g; ++r) oid[r] = (uint32_t)pick_i[r], olp[r] = pick_v[r];
    if (got == k) {
      // then the last k - g admitted entries equal to v*, later id first
      for (int r = g; r < k; ++r) oid[r] = (uint32_t)adm[a - 1 - (r - g)], olp[r] = pick_v[k - 1];
    } else {
      for (int r = got; r < k; ++r) oid[r] = 0xFFFFFFFFu, olp[r] = NEG_INF;
    }
  }
}

#endif  // __HIPCC__

}  // namespace rw
