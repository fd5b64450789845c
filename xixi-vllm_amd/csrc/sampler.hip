// Vocab-wide sampler for gfx950: greedy argmax, temperature / top-k / top-p /
// min-p with an explicit uniform per row.  Four launch shapes share the
// arithmetic below: one 1024-thread workgroup per row (sample_kernel), the
// all-greedy argmax over several workgroups per row (greedy_segment_kernel),
// the sampled path over several workgroups per row for batches of up to
// kSegMaxBatch rows (seg_count / row_count), and for calls whose every
// top_k is at most 64 a two-launch top-k path (seg_topk / row_topk); all give
// the same ids.
//
// Greedy rows follow torch.argmax, the reference's greedy: the lowest NaN id
// if the row holds a NaN, else the largest logit at its lowest id.  Sampled
// rows drop NaN logits (the reference's softmax would turn the whole row NaN).
// Candidates are ordered by descending logit, ties by ascending id.  Every
// candidate's probability mass is an exact int64
//   q = trunc(2^40 * 2^d),  d = (l * (1/T) - x_max) * log2 e  (<= 0)
// with a fixed Taylor exp2 (explicit FMAs) shared with the C restatement of the
// oracle, so kept sets, masses and token ids are bit-identical to it.
//
// Fast path (every row whose boundary fits in LDS):
//   1. one pass: max and min keys;
//   2. one pass: q of every candidate, binned by distance below the max,
//      bucket = min(255, floor(-bs d)) with bs = 16 buckets per binary order,
//      or finer for rows spanning less than 255/16 orders (per-wave LDS
//      histograms of counts and masses, the far bucket in registers);
//   3. the buckets give the bucket holding each cut-off: top-k (by count),
//      top-p (first bucket whose inclusive mass exceeds floor(top_p * mass of
//      the top-k set)), min-p (bucket of the smallest key whose probability
//      reaches min_p of the largest); only the earliest such bucket's
//      candidates are gathered to LDS and bitonic-sorted, which gives the exact
//      boundary candidate (key, id) and the kept mass M;
//   4. one pass: inverse CDF in ascending id order, exp only for kept ids:
//      the first kept id whose inclusive mass exceeds floor(u * M).
// A boundary bucket larger than LDS falls back to an exact row-wide two-level
// (high byte, low byte) radix select over LDS histograms.
#include "xv_common.h"
#include "xv_kernels.h"
#include <math.h>

#pragma clang fp contract(off)


// Rare cases out of the way of the code most rows run through.
#define XV_LIKELY(c) __builtin_expect(!!(c), 1)
#define XV_UNLIKELY(c) __builtin_expect(!!(c), 0)

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int64_t kTieAll = 0x7fffffffffffffffll;
constexpr int kBuckets = 256;
constexpr int kMaxCand = 8192;  // candidates of one bucket sorted in LDS

XV_INLINE float sampler_exp2(float x) {
  if (!(x > -125.0f)) return 0.0f;
  float n = __builtin_rintf(x);
  float f = x - n;
  float p = 1.5252733646775596e-05f;
  p = __builtin_fmaf(p, f, 1.5403529687318951e-04f);
  p = __builtin_fmaf(p, f, 1.3333557872101665e-03f);
  p = __builtin_fmaf(p, f, 9.6181286498904228e-03f);
  p = __builtin_fmaf(p, f, 5.5504109710454941e-02f);
  p = __builtin_fmaf(p, f, 2.4022650718688965e-01f);
  p = __builtin_fmaf(p, f, 6.9314718246459961e-01f);
  p = __builtin_fmaf(p, f, 1.0f);
  return __builtin_ldexpf(p, (int)n);
}

XV_INLINE uint32_t order_key(uint32_t b) {  // 0 is reserved for NaN / padding
  if ((b & 0x7fffu) > 0x7f80u) return 0u;
  return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
}
XV_INLINE uint32_t key_to_bits(uint32_t k) { return (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu); }

// d = (l / T - x_max) * log2 e, evaluated as the oracle does
XV_INLINE float log2_ratio(uint32_t bits, float inv_t, float zmax) {
  float z = bf16_to_f32(bits) * inv_t;
  float d = z - zmax;
  return d * 1.44269502162933349609375f;
}
XV_INLINE float exp_of(uint32_t bits, float inv_t, float zmax) { return sampler_exp2(log2_ratio(bits, inv_t, zmax)); }
// e is in [0, 1] (exp2 of d <= 0; NaN gives 0), so the product converts as
// an unsigned value: the same integer, without the signed conversion's sign
// handling (about half its instructions).
XV_INLINE int64_t mass_of(float e) { return (int64_t)(uint64_t)(e * 1099511627776.0f); }
// Bucket of a candidate d below the max: floor(-d * bs), the last bucket
// holding everything further.  bs is per row (bucket_scale); any bs > 0 keeps
// the buckets monotone in the key, which is all the boundary search needs.
XV_INLINE int bucket_of(float d, float bs) {
  const float u = -d * bs;  // >= 0 for every candidate (d <= 0); NaN -> last bucket
  return u < 255.0f ? (u > 0.0f ? (int)u : 0) : 255;
}
// 16 buckets per binary order, finer when the row spans less than 255/16
// orders below its max (near-flat rows), so that the smallest candidate lands
// in the last bucket and the row spreads over all of them.
XV_INLINE float bucket_scale(float dmin) {
  return (-dmin * 16.0f >= 255.0f || !(-dmin > 1e-30f)) ? 16.0f : 255.0f / -dmin;
}

// Load the 8 logits of thread t in tile j (bits, 0xffff = NaN for padding).
XV_INLINE void load8(const bf16_t* row, int V, int base, bool vec_ok, uint32_t (&bits)[8]) {
  if (vec_ok && base + 8 <= V) {
    Vec8 v = load_vec8(row + base);
#pragma unroll
    for (int k = 0; k < 4; ++k) { bits[2 * k] = v.w[k] & 0xffffu; bits[2 * k + 1] = v.w[k] >> 16; }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) bits[k] = (base + k < V) ? (uint32_t)row[base + k] : 0xffffu;
  }
}

// The same as packed words (two ids each, the lower in the low half): half the
// registers while several vectors are in flight.
XV_INLINE void load8_words(const bf16_t* row, int V, int base, bool vec_ok, uint32_t (&w)[4]) {
  if (vec_ok && base + 8 <= V) {
    const Vec8 v = load_vec8(row + base);
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = v.w[k];
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = (base + 2 * k < V ? (uint32_t)row[base + 2 * k] : 0xffffu) |
             (base + 2 * k + 1 < V ? (uint32_t)row[base + 2 * k + 1] : 0xffffu) << 16;
  }
}
XV_INLINE uint32_t bits_of(const uint32_t (&w)[4], int k) { return (w[k >> 1] >> (16 * (k & 1))) & 0xffffu; }

// Apply f(bits, id) to every id of this thread's contiguous range
// [t*C, t*C + C), C a multiple of 8: chunks of kChunk 16-byte loads are issued
// together, so a pass over the row costs a few memory round trips, not one
// per vector.  Thread order is id order.
constexpr int kChunk = 4;  // 8 took more registers and no less time (600 rows, top-p: 643 against 605 us)
XV_INLINE int range_len(int V) { return ((V + kThreads - 1) / kThreads + 7) / 8 * 8; }
// Apply f(bits, id) to the ids of a coalesced, lane-interleaved layout: in
// step c, vector v of thread t is id 8*((c*kChunk + v)*kThreads + t).  Ids
// ascend within a thread.  Order across threads is not id order.
template <typename F>
XV_INLINE void for_each_strided(const bf16_t* row, int V, bool vec_ok, F&& f) {
  const int nvec = (V + 7) / 8;
  for (int c = 0; c * kChunk * kThreads < nvec; ++c) {
    uint32_t w[kChunk][4];
#pragma unroll
    for (int v = 0; v < kChunk; ++v) {
      const int vi = (c * kChunk + v) * kThreads + threadIdx.x;
      if (vi < nvec) load8_words(row, V, vi * 8, vec_ok, w[v]);
    }
#pragma unroll
    for (int v = 0; v < kChunk; ++v) {
      const int vi = (c * kChunk + v) * kThreads + threadIdx.x;
      if (vi < nvec)
#pragma unroll
        for (int k = 0; k < 8; ++k) f(bits_of(w[v], k), vi * 8 + k);
    }
  }
}

template <int CH = kChunk, typename F>
XV_INLINE void for_each_elem(const bf16_t* row, int V, bool vec_ok, F&& f) {
  const int C = range_len(V);
  const int i0 = threadIdx.x * C, i1 = min(V, i0 + C);
  for (int c = i0; c < i1; c += 8 * CH) {
    uint32_t w[CH][4];
#pragma unroll
    for (int v = 0; v < CH; ++v)
      if (c + 8 * v < i1) load8_words(row, V, c + 8 * v, vec_ok, w[v]);
#pragma unroll
    for (int v = 0; v < CH; ++v)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int id = c + 8 * v + k;
        if (id < i1) f(bits_of(w[v], k), id);
      }
  }
}

struct Shared {
  uint32_t red_u[kWaves];
  float red_f[kWaves];
  int64_t red_l[kWaves];
  uint32_t cnt[256];
  unsigned long long mass[256];
  // broadcast slots
  uint32_t b_key;
  int64_t b_tie;
  int64_t b_id;
  int64_t b_total;
  int b_hb;
};

// LDS of the fast path: per-wave bucket histograms, then the candidate list
struct FastShared {
  uint32_t wcnt[kWaves][kBuckets];
  unsigned long long wmass[kWaves][kBuckets];
  unsigned long long cand[kMaxCand];  // (key << 32) | (0xffffffff - id), sorted descending
  int ncand;
};

// x[lane ^ S] in registers, no LDS round trip: DPP within a 16-lane row for
// S = 1, 2 (quad_perm), 8 (row_ror:8) and 4 (row_ror:4 for lanes with bit 2
// set, row_ror:12 for the others: row_ror:n reads lane (i - n) mod 16), the
// gfx950 row-swap permutes for 16 and 32 (each result holds x[lane] in one
// half of the rows and x[lane ^ S] in the other).
template <int CTRL>
XV_INLINE uint32_t dpp_u(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, false);
}
template <int S>
XV_INLINE uint32_t xor_lane(uint32_t x) {
  const int lane = threadIdx.x & 63;
  if constexpr (S == 1) return dpp_u<0xB1>(x);
  else if constexpr (S == 2) return dpp_u<0x4E>(x);
  else if constexpr (S == 4) { const uint32_t a = dpp_u<0x124>(x), b = dpp_u<0x12C>(x); return (lane & 4) ? a : b; }
  else if constexpr (S == 8) return dpp_u<0x128>(x);
  else if constexpr (S == 16) { const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false); return (lane & 16) ? r[0] : r[1]; }
  else { static_assert(S == 32, "xor by a power of two below 64"); const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false); return (lane & 32) ? r[0] : r[1]; }
}
template <int S>
XV_INLINE unsigned long long xor_lane64(unsigned long long x) {
  return ((unsigned long long)xor_lane<S>((uint32_t)(x >> 32)) << 32) | xor_lane<S>((uint32_t)x);
}
XV_INLINE unsigned long long xor_lane64(unsigned long long x, int s) {  // s a constant after unrolling
  switch (s) {
    case 1: return xor_lane64<1>(x);
    case 2: return xor_lane64<2>(x);
    case 4: return xor_lane64<4>(x);
    case 8: return xor_lane64<8>(x);
    case 16: return xor_lane64<16>(x);
    default: return xor_lane64<32>(x);
  }
}
// Wave-wide reductions through the register permutes above (the shuffles
// they replace each took an LDS round trip, two for 64-bit values).
XV_INLINE uint32_t wave_max_u(uint32_t x) {
  x = max(x, xor_lane<1>(x));
  x = max(x, xor_lane<2>(x));
  x = max(x, xor_lane<4>(x));
  x = max(x, xor_lane<8>(x));
  x = max(x, xor_lane<16>(x));
  return max(x, xor_lane<32>(x));
}
XV_INLINE uint32_t wave_min_u(uint32_t x) {
  x = min(x, xor_lane<1>(x));
  x = min(x, xor_lane<2>(x));
  x = min(x, xor_lane<4>(x));
  x = min(x, xor_lane<8>(x));
  x = min(x, xor_lane<16>(x));
  return min(x, xor_lane<32>(x));
}
XV_INLINE float wave_maxf(float x) {
  x = fmaxf(x, __uint_as_float(xor_lane<1>(__float_as_uint(x))));
  x = fmaxf(x, __uint_as_float(xor_lane<2>(__float_as_uint(x))));
  x = fmaxf(x, __uint_as_float(xor_lane<4>(__float_as_uint(x))));
  x = fmaxf(x, __uint_as_float(xor_lane<8>(__float_as_uint(x))));
  x = fmaxf(x, __uint_as_float(xor_lane<16>(__float_as_uint(x))));
  return fmaxf(x, __uint_as_float(xor_lane<32>(__float_as_uint(x))));
}
XV_INLINE int64_t wave_min_l(int64_t x) {
#pragma unroll
  for (int sh = 1; sh < 64; sh <<= 1) {
    const int64_t y = (int64_t)xor_lane64(x, sh);
    x = y < x ? y : x;
  }
  return x;
}
XV_INLINE unsigned long long wave_max_ull(unsigned long long x) {
#pragma unroll
  for (int sh = 1; sh < 64; sh <<= 1) {
    const unsigned long long y = xor_lane64(x, sh);
    x = y > x ? y : x;
  }
  return x;
}


// x[lane - S] within the lane's 16-lane row (0 for the first S lanes of a
// row), and the cross-row broadcasts of lane 15 (into rows 1, 3) and lane 31
// (into rows 2, 3); other lanes get 0.
template <int CTRL, int ROWS>
XV_INLINE uint64_t dpp64(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, ROWS, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), CTRL, ROWS, 0xf, true);
  return ((uint64_t)hi << 32) | lo;
}
XV_INLINE int64_t wave_sum_l(int64_t x) {
  x += (int64_t)xor_lane64<1>((uint64_t)x);
  x += (int64_t)xor_lane64<2>((uint64_t)x);
  x += (int64_t)xor_lane64<4>((uint64_t)x);
  x += (int64_t)xor_lane64<8>((uint64_t)x);
  x += (int64_t)xor_lane64<16>((uint64_t)x);
  x += (int64_t)xor_lane64<32>((uint64_t)x);
  return x;
}
// Inclusive prefix sum over the wave's lanes: within rows by row_shr 1, 2, 4,
// 8, then row 1 and 3 add lane 15 of the row before, rows 2 and 3 lane 31.
XV_INLINE int64_t wave_incl_scan_l(int64_t x) {
  x += (int64_t)dpp64<0x111, 0xf>((uint64_t)x);
  x += (int64_t)dpp64<0x112, 0xf>((uint64_t)x);
  x += (int64_t)dpp64<0x114, 0xf>((uint64_t)x);
  x += (int64_t)dpp64<0x118, 0xf>((uint64_t)x);
  x += (int64_t)dpp64<0x142, 0xa>((uint64_t)x);
  x += (int64_t)dpp64<0x143, 0xc>((uint64_t)x);
  return x;
}

template <int CTRL, int ROWS>
XV_INLINE int dpp_scan_i(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, true);
}
XV_INLINE int wave_incl_scan_i(int x) {
  x += dpp_scan_i<0x111, 0xf>(x);
  x += dpp_scan_i<0x112, 0xf>(x);
  x += dpp_scan_i<0x114, 0xf>(x);
  x += dpp_scan_i<0x118, 0xf>(x);
  x += dpp_scan_i<0x142, 0xa>(x);
  x += dpp_scan_i<0x143, 0xc>(x);
  return x;
}

XV_INLINE uint32_t block_max_u(Shared& s, uint32_t x) {
  x = wave_max_u(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.red_u[w] = x;
  __syncthreads();
  uint32_t r = s.red_u[0];
  for (int i = 1; i < kWaves; ++i) r = max(r, s.red_u[i]);
  return r;
}
XV_INLINE uint32_t block_min_u(Shared& s, uint32_t x) {
  x = wave_min_u(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.red_u[w] = x;
  __syncthreads();
  uint32_t r = s.red_u[0];
  for (int i = 1; i < kWaves; ++i) r = min(r, s.red_u[i]);
  return r;
}
XV_INLINE float block_maxf(Shared& s, float x) {
  x = wave_maxf(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.red_f[w] = x;
  __syncthreads();
  float r = s.red_f[0];
  for (int i = 1; i < kWaves; ++i) r = fmaxf(r, s.red_f[i]);
  return r;
}
XV_INLINE int64_t block_sum_l(Shared& s, int64_t x) {
  x = wave_sum_l(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.red_l[w] = x;
  __syncthreads();
  int64_t r = 0;
  for (int i = 0; i < kWaves; ++i) r += s.red_l[i];
  return r;
}
// Exclusive prefix sum over the block (thread order); *total gets the block sum.
XV_INLINE int64_t block_excl_scan(Shared& s, int64_t x, int64_t* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t inc = wave_incl_scan_l(x);
  __syncthreads();
  if (lane == 63) s.red_l[w] = inc;
  __syncthreads();
  int64_t before = 0, tot = 0;
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += s.red_l[i];
    tot += s.red_l[i];
  }
  *total = tot;
  return before + inc - x;
}

struct Boundary {
  uint32_t key;  // kept: key > key, or key == key with tie index <= tie
  int64_t tie;   // kTieAll: every tie of `key` kept
};
XV_INLINE bool earlier(const Boundary& a, const Boundary& b) {
  return a.key > b.key || (a.key == b.key && a.tie < b.tie);
}

// Call f(bits, id) for every slot of a lane-interleaved layout like that of
// for_each_strided (kChunkAll vectors per step) on every lane of every wave: slots at or past V come as
// 0xffff (key 0), so f may use wave-wide operations.
constexpr int kChunkAll = 2;  // few registers: see row_count_kernel
template <typename F>
XV_INLINE void for_each_strided_all(const bf16_t* row, int V, bool vec_ok, F&& f) {
  const int nvec = (V + 7) / 8;
  for (int c = 0; c * kChunkAll * kThreads < nvec; ++c) {
    uint32_t w[kChunkAll][4];  // packed pairs, low half first
#pragma unroll
    for (int v = 0; v < kChunkAll; ++v) {
      const int base = ((c * kChunkAll + v) * kThreads + threadIdx.x) * 8;
      if (vec_ok && base + 8 <= V) {
        const Vec8 x = load_vec8(row + base);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[v][k] = x.w[k];
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          w[v][k] = (base + 2 * k < V ? (uint32_t)row[base + 2 * k] : 0xffffu) |
                    (base + 2 * k + 1 < V ? (uint32_t)row[base + 2 * k + 1] : 0xffffu) << 16;
      }
    }
#pragma unroll
    for (int v = 0; v < kChunkAll; ++v)
#pragma unroll
      for (int k = 0; k < 8; ++k)
        f((w[v][k >> 1] >> (16 * (k & 1))) & 0xffffu, ((c * kChunkAll + v) * kThreads + threadIdx.x) * 8 + k);
  }
}

// Add one count (CNT) and the mass m (MASS) to bin `bin` of the LDS
// histograms for every lane with `on`.  The lanes of each of the wave's first
// four distinct bins are summed first and added with one atomic per
// histogram: near-flat rows put nearly every candidate into two or three
// high-byte bins, where per-lane atomics to one address serialise.  Lanes of
// further bins add their own.  Called by the whole wave.
template <bool CNT, bool MASS>
XV_INLINE void hist_add(uint32_t* cnt, unsigned long long* mass, bool on, int bin, int64_t m) {
  const int lane = threadIdx.x & 63;
  bool pending = on;
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const unsigned long long todo = __ballot(pending);
    if (todo == 0ull) break;
    const int lead = __builtin_ctzll(todo);
    const int lb = __shfl(bin, lead);
    const bool mine = pending && bin == lb;
    const unsigned long long mm = __ballot(mine);
    const int64_t sm = MASS ? wave_sum_l(mine ? m : 0) : 0;
    if (lane == lead) {
      if (CNT) atomicAdd(&cnt[lb], (uint32_t)__popcll(mm));
      if (MASS) atomicAdd(&mass[lb], (unsigned long long)sm);
    }
    pending = pending && !mine;
  }
  if (pending) {
    if (CNT) atomicAdd(&cnt[bin], 1u);
    if (MASS) atomicAdd(&mass[bin], (unsigned long long)m);
  }
}

XV_INLINE void clear_hist(Shared& s) {
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += kThreads) { s.cnt[i] = 0; s.mass[i] = 0; }
  __syncthreads();
}

// Exact cut-offs by a two-level (high byte, low byte) radix select over LDS
// histograms of the whole row: the fallback when the boundary bucket of the
// fast path holds more candidates than LDS does (very flat distributions).
// Histogram passes read the row in chunks of kChunk vectors per thread (a few
// memory round trips per pass).
XV_INLINE void general_boundary(Shared& s, const bf16_t* row, int V, bool vec_ok, float inv_t, float zmax,
                                int top_k, float top_p, float min_p, bool use_k, bool use_p, bool use_m,
                                Boundary& bd_out, int64_t& id_cut_out, int64_t& M_out) {
  const int t = threadIdx.x;
  Boundary bd = {1u, kTieAll};
  if (use_k || use_p || use_m) {
    // ---- pass 2: high-byte histogram of counts and masses; min-p key ----
    clear_hist(s);
    uint32_t kmin_p = 0xffffffffu;
    for_each_strided_all(row, V, vec_ok, [&](uint32_t bits, int) {
      const uint32_t key = order_key(bits);
      const float e = exp_of(bits, inv_t, zmax);
      if (use_m && key && e >= min_p) kmin_p = min(kmin_p, key);
      hist_add<true, true>(s.cnt, s.mass, key != 0, (int)(key >> 8), mass_of(e));
    });
    kmin_p = use_m ? block_min_u(s, kmin_p) : 0u;
    __syncthreads();

    // boundary of top-k (by count), and total mass of the top-k set
    int64_t total_k = 0;
    if (t == 0) {
      int64_t tot = 0;
      for (int i = 0; i < 256; ++i) tot += (int64_t)s.mass[i];
      s.b_total = tot;
      if (use_k) {
        int64_t c = 0;
        int hb = 255;
        for (; hb > 0; --hb) {
          if (c + s.cnt[hb] > (uint32_t)(top_k - 1)) break;
          c += s.cnt[hb];
        }
        s.b_hb = hb;
        s.b_tie = c;  // count above the bin
      }
    }
    __syncthreads();
    Boundary bk = {1u, kTieAll};
    if (use_k) {
      // ---- pass 3: low-byte histogram inside the top-k high bin ----
      const int hb = s.b_hb;
      const int64_t c_above = s.b_tie;
      clear_hist(s);
      for_each_strided_all(row, V, vec_ok, [&](uint32_t bits, int) {
        const uint32_t key = order_key(bits);
        hist_add<true, false>(s.cnt, s.mass, key != 0 && (int)(key >> 8) == hb, (int)(key & 255), 0);
      });
      __syncthreads();
      if (t == 0) {
        int64_t c = c_above;
        int lb = 255;
        for (; lb > 0; --lb) {
          if (c + s.cnt[lb] > top_k - 1) break;
          c += s.cnt[lb];
        }
        s.b_key = ((uint32_t)hb << 8) | (uint32_t)lb;
        s.b_tie = (int64_t)(top_k - 1) - c;
      }
      __syncthreads();
      bk.key = s.b_key;
      bk.tie = s.b_tie;
      // mass of the top-k set: everything above the boundary key plus tie_k+1 copies
      int64_t above = 0;
      for_each_strided(row, V, vec_ok, [&](uint32_t bits, int) {
        if (order_key(bits) > bk.key) above += mass_of(exp_of(bits, inv_t, zmax));
      });
      above = block_sum_l(s, above);
      total_k = above + (bk.tie + 1) * mass_of(exp_of(key_to_bits(bk.key), inv_t, zmax));
    } else {
      total_k = s.b_total;
    }

    Boundary bp = {1u, kTieAll};
    if (use_p) {
      // ---- pass 4: first rank whose inclusive mass exceeds floor(top_p * total_k) ----
      const int64_t thr = (int64_t)floor((double)top_p * (double)total_k);
      if (use_k) {
        // pass 3 reused the histograms: rebuild the high-byte masses
        clear_hist(s);
        for_each_strided_all(row, V, vec_ok, [&](uint32_t bits, int) {
          const uint32_t key = order_key(bits);
          hist_add<false, true>(s.cnt, s.mass, key != 0, (int)(key >> 8), mass_of(exp_of(bits, inv_t, zmax)));
        });
      }
      __syncthreads();
      if (t == 0) {
        int64_t m = 0;
        int hb = 255;
        bool found = false;
        for (; hb >= 0; --hb) {
          if (m + (int64_t)s.mass[hb] > thr) { found = true; break; }
          m += (int64_t)s.mass[hb];
        }
        s.b_hb = found ? hb : -1;
        s.b_total = m;
      }
      __syncthreads();
      const int hb = s.b_hb;
      const int64_t m_above = s.b_total;
      if (hb >= 0) {
        clear_hist(s);
        for_each_strided_all(row, V, vec_ok, [&](uint32_t bits, int) {
          const uint32_t key = order_key(bits);
          const bool in = key != 0 && (int)(key >> 8) == hb;
          hist_add<false, true>(s.cnt, s.mass, in, (int)(key & 255), in ? mass_of(exp_of(bits, inv_t, zmax)) : 0);
        });
        __syncthreads();
        if (t == 0) {
          int64_t m = m_above;
          int lb = 255;
          for (; lb > 0; --lb) {
            if (m + (int64_t)s.mass[lb] > thr) break;
            m += (int64_t)s.mass[lb];
          }
          const uint32_t key = ((uint32_t)hb << 8) | (uint32_t)lb;
          const int64_t q = mass_of(exp_of(key_to_bits(key), inv_t, zmax));
          s.b_key = key;
          s.b_tie = q > 0 ? (thr - m) / q : kTieAll;
        }
        __syncthreads();
        bp.key = s.b_key;
        bp.tie = s.b_tie;
      }
    }
    bd = bk;
    if (earlier(bp, bd)) bd = bp;
    if (use_m && kmin_p != 0xffffffffu) {
      Boundary bm = {kmin_p, kTieAll};
      if (earlier(bm, bd)) bd = bm;
    }
  }

  // ---- pass 5: kept mass, and the id of the last kept tie of the boundary key ----
  // Thread t owns the contiguous ids of for_each_elem, so one block scan of the
  // per-thread tie counts ranks the ties in id order.  Every tie has the same
  // mass q.
  int64_t above = 0, nt = 0;
  for_each_elem(row, V, vec_ok, [&](uint32_t bits, int) {
    const uint32_t key = order_key(bits);
    if (key > bd.key) above += mass_of(exp_of(bits, inv_t, zmax));
    nt += key == bd.key;
  });
  int64_t ties;
  const int64_t r0 = block_excl_scan(s, nt, &ties);
  const int64_t kept_ties = bd.tie == kTieAll ? ties : min(ties, bd.tie + 1);
  const int64_t q = kept_ties ? mass_of(exp_of(key_to_bits(bd.key), inv_t, zmax)) : 0;
  const int64_t M = block_sum_l(s, above) + kept_ties * q;
  if (t == 0) s.b_id = kTieAll;
  __syncthreads();
  if (bd.tie != kTieAll && bd.tie >= r0 && bd.tie < r0 + nt) {
    int64_t r = r0;
    for_each_elem<2>(row, V, vec_ok, [&](uint32_t bits, int id) {  // one thread: few registers
      if (order_key(bits) == bd.key) {
        if (r == bd.tie) s.b_id = id;
        ++r;
      }
    });
  }
  __syncthreads();
  id_cut_out = s.b_id;
  __syncthreads();  // every thread has read b_id before it is reset
  bd_out = bd;
  M_out = M;
}

XV_INLINE int64_t block_min_l(Shared& s, int64_t x) {
  x = wave_min_l(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.red_l[w] = x;
  __syncthreads();
  int64_t r = s.red_l[0];
  for (int i = 1; i < kWaves; ++i) r = s.red_l[i] < r ? s.red_l[i] : r;
  return r;
}

XV_INLINE uint32_t cand_key(unsigned long long c) { return (uint32_t)(c >> 32); }
XV_INLINE int64_t cand_id(unsigned long long c) { return (int64_t)(0xffffffffu - (uint32_t)(c & 0xffffffffu)); }
XV_INLINE int64_t cand_mass(unsigned long long c, float inv_t, float zmax) {
  return mass_of(exp_of(key_to_bits(cand_key(c)), inv_t, zmax));
}

// Bitonic sort of fs.cand[0, n) descending (n <= kMaxCand), padding with
// zeros up to the next power of two; the padding sorts last.
XV_INLINE void sort_cand_desc(FastShared& fs, int n) {
  const int t = threadIdx.x;
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  for (int i = n + t; i < np2; i += kThreads) fs.cand[i] = 0ull;  // padding sorts last
  __syncthreads();
  for (int size = 2; size <= np2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = t; i < np2 / 2; i += kThreads) {
        const int lo = 2 * i - (i & (stride - 1));
        const int hi = lo + stride;
        const unsigned long long a = fs.cand[lo], b = fs.cand[hi];
        const bool desc = (lo & size) == 0;
        if (desc ? (a < b) : (a > b)) { fs.cand[lo] = b; fs.cand[hi] = a; }
      }
      __syncthreads();
    }
  }
}

// Gather the candidates of bucket `target` into fs.cand and bitonic-sort them
// descending (key descending, id ascending).  Returns the count; a count above
// kMaxCand means the bucket did not fit (nothing sorted).
XV_INLINE int gather_bucket(FastShared& fs, const bf16_t* row, int V, bool vec_ok, float inv_t,
                            float zmax, float bs, int target, int target_lo = -1) {
  if (target_lo < 0) target_lo = target;  // gather buckets target_lo .. target
  const int t = threadIdx.x;
  __syncthreads();
  if (t == 0) fs.ncand = 0;
  __syncthreads();
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int id) {
    const uint32_t key = order_key(bits);
    if (!key) return;
    const int bkt = bucket_of(log2_ratio(bits, inv_t, zmax), bs);
    if (bkt < target_lo || bkt > target) return;
    const int slot = atomicAdd(&fs.ncand, 1);
    if (slot < kMaxCand)
      fs.cand[slot] = ((unsigned long long)key << 32) | (unsigned long long)(0xffffffffu - (uint32_t)id);
  });
  __syncthreads();
  const int n = fs.ncand;
  if (n > kMaxCand) return n;
  sort_cand_desc(fs, n);
  return n;
}

// Sum of the masses of the first m sorted candidates.
XV_INLINE int64_t list_mass_prefix(Shared& s, const FastShared& fs, int n, int64_t m, float inv_t, float zmax) {
  const int per = (n + kThreads - 1) / kThreads;
  const int i0 = threadIdx.x * per, i1 = min(n, i0 + per);
  int64_t sum = 0;
  for (int i = i0; i < i1; ++i)
    if (i < m) sum += cand_mass(fs.cand[i], inv_t, zmax);
  return block_sum_l(s, sum);
}

// First sorted index whose inclusive mass (plus base) exceeds thr, n if none.
XV_INLINE int64_t list_first_exceed(Shared& s, const FastShared& fs, int n, int64_t base, int64_t thr, float inv_t,
                                    float zmax) {
  const int per = (n + kThreads - 1) / kThreads;
  const int i0 = threadIdx.x * per, i1 = min(n, i0 + per);
  int64_t local = 0;
  for (int i = i0; i < i1; ++i) local += cand_mass(fs.cand[i], inv_t, zmax);
  int64_t tot;
  int64_t cum = base + block_excl_scan(s, local, &tot);
  int64_t found = n;
  for (int i = i0; i < i1; ++i) {
    cum += cand_mass(fs.cand[i], inv_t, zmax);
    if (cum > thr) { found = i; break; }
  }
  return block_min_l(s, found);
}

// Number of sorted candidates with key >= kmin (a prefix of the list).
XV_INLINE int64_t list_count_ge(Shared& s, const FastShared& fs, int n, uint32_t kmin) {
  int64_t c = 0;
  for (int i = threadIdx.x; i < n; i += kThreads) c += cand_key(fs.cand[i]) >= kmin;
  return block_sum_l(s, c);
}

// Smallest key whose probability reaches min_p of the largest (0xffffffff:
// none).  Only candidates within half a binary order of the threshold need an
// exp: below that their probability is certainly under min_p.
XV_INLINE uint32_t minp_key(Shared& s, const bf16_t* row, int V, bool vec_ok, float inv_t, float zmax,
                            float min_p) {
  const float d_lo = __log2f(min_p) - 0.5f;
  uint32_t kminp = 0xffffffffu;
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int) {
    const uint32_t key = order_key(bits);
    if (!key) return;
    const float d = log2_ratio(bits, inv_t, zmax);
    if (d >= d_lo && sampler_exp2(d) >= min_p) kminp = min(kminp, key);
  });
  return block_min_u(s, kminp);
}

// Fast path with top-k: bucket counts only (no exp), then every candidate of
// the buckets up to the one holding rank k-1 is gathered and sorted; the
// top-k set, its mass, the top-p and min-p cuts all come from that list.
XV_INLINE bool topk_boundary(Shared& s, FastShared& fs, const bf16_t* row, int V, bool vec_ok,
                             float inv_t, float zmax, float bs, int top_k, float top_p, float min_p, bool use_p, bool use_m,
                             uint32_t& key_cut, int64_t& id_cut, int64_t& M, int& list_kept) {
  const int t = threadIdx.x, w = t >> 6;
  for (int i = t; i < kWaves * kBuckets; i += kThreads) (&fs.wcnt[0][0])[i] = 0u;
  __syncthreads();
  int64_t far_c = 0;
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int) {
    if (!order_key(bits)) return;
    const int bkt = bucket_of(log2_ratio(bits, inv_t, zmax), bs);
    if (bkt < kBuckets - 1) atomicAdd(&fs.wcnt[w][bkt], 1u);
    else far_c += 1;
  });
  far_c = block_sum_l(s, far_c);
  __syncthreads();
  if (t < kBuckets) {
    uint32_t c = 0;
    for (int ww = 0; ww < kWaves; ++ww) c += fs.wcnt[ww][t];
    if (t == kBuckets - 1) c += (uint32_t)far_c;
    s.cnt[t] = c;
  }
  __syncthreads();
  int bk = kBuckets;
  int64_t upto = 0;  // candidates in buckets 0..bk
  {
    int64_t c = 0;
    for (int bkt = 0; bkt < kBuckets; ++bkt) {
      c += s.cnt[bkt];
      if (c >= top_k) { bk = bkt; upto = c; break; }
    }
  }
  if (bk >= kBuckets - 1 || upto > kMaxCand) return false;  // rank k-1 far out or too many: exact row-wide path
  const uint32_t kminp = use_m ? minp_key(s, row, V, vec_ok, inv_t, zmax, min_p) : 0xffffffffu;
  const int n = gather_bucket(fs, row, V, vec_ok, inv_t, zmax, bs, bk, 0);
  if (n > kMaxCand) return false;
  const int64_t total_k = list_mass_prefix(s, fs, n, top_k, inv_t, zmax);
  int64_t jcut = (int64_t)top_k - 1;
  if (use_p) {
    const int64_t thr = (int64_t)floor((double)top_p * (double)total_k);
    jcut = min(jcut, list_first_exceed(s, fs, n, 0, thr, inv_t, zmax));
  }
  if (use_m && kminp != 0xffffffffu && kminp >= cand_key(fs.cand[n - 1]))
    jcut = min(jcut, list_count_ge(s, fs, n, kminp) - 1);
  if (jcut >= n) jcut = n - 1;
  if (jcut < 0) jcut = 0;
  const unsigned long long edge = fs.cand[jcut];
  key_cut = cand_key(edge);
  id_cut = cand_id(edge);
  M = list_mass_prefix(s, fs, n, jcut + 1, inv_t, zmax);
  list_kept = (int)jcut + 1;  // the kept set is exactly fs.cand[0, jcut]
  return true;
}

// Fast path: kept set = key > key_cut, or key == key_cut and id <= id_cut;
// M = its mass.  Returns false when a boundary bucket overflowed the list.
XV_INLINE bool fast_boundary(Shared& s, FastShared& fs, const bf16_t* row, int V, bool vec_ok,
                             float inv_t, float zmax, float bs, int top_k, float top_p, float min_p, bool use_k, bool use_p,
                             bool use_m, uint32_t& key_cut, int64_t& id_cut, int64_t& M, int& list_kept) {
  const int t = threadIdx.x, w = t >> 6;
  if (use_k) return topk_boundary(s, fs, row, V, vec_ok, inv_t, zmax, bs, top_k, top_p, min_p, use_p, use_m,
                                  key_cut, id_cut, M, list_kept);
  // ---- pass 2: every candidate's mass, binned by distance below the max ----
  for (int i = t; i < kWaves * kBuckets; i += kThreads) {
    (&fs.wcnt[0][0])[i] = 0u;
    (&fs.wmass[0][0])[i] = 0ull;
  }
  __syncthreads();
  int64_t far_c = 0, far_m = 0;
  uint32_t kminp = 0xffffffffu;
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int) {
    const uint32_t key = order_key(bits);
    if (!key) return;
    const float d = log2_ratio(bits, inv_t, zmax);
    const float e = sampler_exp2(d);
    const int64_t q = mass_of(e);
    const int bkt = bucket_of(d, bs);
    if (bkt < kBuckets - 1) {
      atomicAdd(&fs.wcnt[w][bkt], 1u);
      atomicAdd(&fs.wmass[w][bkt], (unsigned long long)q);
    } else {
      far_c += 1;
      far_m += q;
    }
    if (use_m && e >= min_p) kminp = min(kminp, key);
  });
  far_c = block_sum_l(s, far_c);
  far_m = block_sum_l(s, far_m);
  if (use_m) kminp = block_min_u(s, kminp);
  __syncthreads();
  if (t < kBuckets) {
    uint32_t c = 0;
    unsigned long long m = 0;
    for (int ww = 0; ww < kWaves; ++ww) { c += fs.wcnt[ww][t]; m += fs.wmass[ww][t]; }
    if (t == kBuckets - 1) { c += (uint32_t)far_c; m += (unsigned long long)far_m; }
    s.cnt[t] = c;
    s.mass[t] = m;
  }
  __syncthreads();
  int64_t total = 0;
  for (int bkt = 0; bkt < kBuckets; ++bkt) total += (int64_t)s.mass[bkt];
  key_cut = 1u;
  id_cut = kTieAll;
  M = total;
  if (!(use_p || use_m)) return true;

  // ---- bucket of each cut-off ----
  int bp = kBuckets;
  int64_t thr = 0, mp_before = 0;
  if (use_p) {
    thr = (int64_t)floor((double)top_p * (double)total);
    int64_t m = 0;
    for (int bkt = 0; bkt < kBuckets; ++bkt) {
      if (m + (int64_t)s.mass[bkt] > thr) { bp = bkt; mp_before = m; break; }
      m += (int64_t)s.mass[bkt];
    }
  }
  int bm = kBuckets;
  if (use_m && kminp != 0xffffffffu) bm = bucket_of(log2_ratio(key_to_bits(kminp), inv_t, zmax), bs);
  const int bf = min(bp, bm);
  if (bf >= kBuckets) return true;  // no cut-off limits the row: everything kept
  if (s.cnt[bf] > (uint32_t)kMaxCand) return false;
  const int n = gather_bucket(fs, row, V, vec_ok, inv_t, zmax, bs, bf);
  if (n > kMaxCand) return false;
  // ---- exact cut inside the boundary bucket ----
  int64_t jcut = kTieAll;
  if (bp == bf) jcut = min(jcut, list_first_exceed(s, fs, n, mp_before, thr, inv_t, zmax));
  if (bm == bf) jcut = min(jcut, list_count_ge(s, fs, n, kminp) - 1);
  if (jcut >= n) jcut = n - 1;
  if (jcut < 0) jcut = 0;
  int64_t m_before = 0;
  for (int bkt = 0; bkt < bf; ++bkt) m_before += (int64_t)s.mass[bkt];
  const unsigned long long edge = fs.cand[jcut];
  key_cut = cand_key(edge);
  id_cut = cand_id(edge);
  M = m_before + list_mass_prefix(s, fs, n, jcut + 1, inv_t, zmax);
  return true;
}

// Inverse-CDF draw over a kept set held as the sorted list fs.cand[0, n):
// re-key it as (~id << 32 | key), so that the descending sort puts ids in
// ascending order, then scan its masses.  Returns the first id whose inclusive
// mass exceeds rdraw (kTieAll: none).
XV_INLINE int64_t list_draw(Shared& s, FastShared& fs, int n, float inv_t, float zmax, int64_t rdraw) {
  const int t = threadIdx.x;
  __syncthreads();
  for (int i = t; i < n; i += kThreads) {
    const unsigned long long c = fs.cand[i];
    fs.cand[i] = ((unsigned long long)(0xffffffffu - (uint32_t)cand_id(c)) << 32) | cand_key(c);
  }
  __syncthreads();
  sort_cand_desc(fs, n);
  auto entry_mass = [&](unsigned long long c) {
    return mass_of(exp_of(key_to_bits((uint32_t)(c & 0xffffffffu)), inv_t, zmax));
  };
  const int per = (n + kThreads - 1) / kThreads;
  const int j0 = t * per, j1 = min(n, j0 + per);
  int64_t local = 0;
  for (int j = j0; j < j1; ++j) local += entry_mass(fs.cand[j]);
  int64_t tot;
  int64_t cum = block_excl_scan(s, local, &tot);
  int64_t found = kTieAll;
  for (int j = j0; j < j1; ++j) {
    cum += entry_mass(fs.cand[j]);
    if (cum > rdraw) { found = 0xffffffffu - (uint32_t)(fs.cand[j] >> 32); break; }
  }
  return block_min_l(s, found);
}

// The draw point floor(u * M), clamped to [0, M).
XV_INLINE int64_t draw_point(float u, int64_t M) {
  int64_t r = (int64_t)((double)u * (double)M);
  if (r >= M) r = M - 1;
  if (r < 0) r = 0;
  return r;
}

// The draw's answer when no candidate has mass.  A scaled row maximum z_max
// that is not finite (a largest logit of +inf or -inf, or a finite one past
// fp32's range once divided by the temperature) makes d = z - z_max NaN at
// the largest key (inf - inf), whose exp2 is 0, and -inf below it: every
// mass is 0, and the draw takes the first candidate in rank order, the
// lowest id holding the largest key.  With a finite z_max the largest logit
// has mass 2^40 and is always kept, so this is the only way the kept mass is 0.
XV_INLINE int64_t lowest_id_of_key(Shared& s, const bf16_t* row, int V, bool vec_ok, uint32_t key) {
  uint32_t first = 0xffffffffu;
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int id) {
    if (id < V && order_key(bits) == key) first = min(first, (uint32_t)id);
  });
  first = block_min_u(s, first);
  return first == 0xffffffffu ? 0 : (int64_t)first;
}

// The whole sampler for row b by one kThreads workgroup.
XV_INLINE void sample_row(Shared& s, FastShared& fs, int b, const bf16_t* __restrict__ logits, int64_t stride, int V,
                          const float* __restrict__ temps, const float* __restrict__ top_ps,
                          const int32_t* __restrict__ top_ks, const float* __restrict__ min_ps,
                          const float* __restrict__ uniforms, int flags, int64_t* __restrict__ out_ids) {
  const int t = threadIdx.x;
  const bf16_t* row = logits + (int64_t)b * stride;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  const float temp = temps ? temps[b] : 1.0f;
  const bool greedy = (flags & XV_SAMPLE_ALL_GREEDY) || temp <= 1e-5f;

  // ---- greedy (torch.argmax): the lowest NaN id if the row holds a NaN,
  // else the max value and the lowest index holding it ----
  if (greedy) {
    // one pass: the lane's max, its lowest id and its lowest NaN id, then the block's
    float fm = -INFINITY;
    uint32_t best = 0xffffffffu, nan_id = 0xffffffffu;
    for_each_strided(row, V, vec_ok, [&](uint32_t bits, int id) {
      if (!order_key(bits)) {
        if (id < V) nan_id = min(nan_id, (uint32_t)id);  // ids past V are padding
        return;
      }
      const float v = bf16_to_f32(bits);
      if (v > fm) { fm = v; best = (uint32_t)id; }  // ids ascend within a lane: keeps the lowest
    });
    nan_id = block_min_u(s, nan_id);
    const float gm = block_maxf(s, fm);
    best = block_min_u(s, fm == gm ? best : 0xffffffffu);
    if (nan_id != 0xffffffffu) best = nan_id;
    if (t == 0) out_ids[b] = best == 0xffffffffu ? 0 : (int64_t)best;
    return;
  }

  // ---- pass 1: the largest key ----
  uint32_t kmax = 0, kmin = 0xffffffffu;
  for_each_strided(row, V, vec_ok, [&](uint32_t bits, int) {
    const uint32_t key = order_key(bits);
    kmax = max(kmax, key);
    if (key) kmin = min(kmin, key);
  });
  kmax = block_max_u(s, kmax);
  kmin = block_min_u(s, kmin);
  const float inv_t = 1.0f / temp;
  const float zmax = bf16_to_f32(key_to_bits(kmax)) * inv_t;
  if (kmax && !__builtin_isfinite(zmax)) {  // no mass anywhere
    const int64_t id = lowest_id_of_key(s, row, V, vec_ok, kmax);
    if (t == 0) out_ids[b] = id;
    return;
  }
  const float bs = kmax ? bucket_scale(log2_ratio(key_to_bits(kmin), inv_t, zmax)) : 16.0f;

  const float top_p = ((flags & XV_SAMPLE_USE_TOP_P) && top_ps) ? top_ps[b] : 1.0f;
  const float min_p = ((flags & XV_SAMPLE_USE_MIN_P) && min_ps) ? min_ps[b] : 0.0f;
  const bool use_p = top_p < 1.0f;
  const bool use_m = min_p > 0.0f;
  // a min-p above 1 keeps the first candidate alone (as row_params)
  const int top_k = min_p > 1.0f ? 1 : ((flags & XV_SAMPLE_USE_TOP_K) && top_ks) ? top_ks[b] : V;
  const bool use_k = top_k > 0 && top_k < V;

  uint32_t key_cut;
  int64_t id_cut, M;
  int list_kept = 0;  // > 0: the kept set is the sorted list prefix fs.cand[0, list_kept)
  if (!fast_boundary(s, fs, row, V, vec_ok, inv_t, zmax, bs, top_k, top_p, min_p, use_k, use_p, use_m,
                     key_cut, id_cut, M, list_kept)) {
    list_kept = 0;
    Boundary bd;
    general_boundary(s, row, V, vec_ok, inv_t, zmax, top_k, top_p, min_p, use_k, use_p, use_m, bd, id_cut,
                     M);
    key_cut = bd.key;
  }

  // ---- last pass: inverse-CDF draw in ascending id order (exp for kept ids only) ----
  // Thread t owns the contiguous ids [t*C, t*C + C), C a multiple of 8, so one
  // block scan orders the whole row.
  const float u = uniforms ? uniforms[b] : 0.5f;
  const int64_t rdraw = draw_point(u, M);
  if (list_kept > 0) {
    const int64_t found = list_draw(s, fs, list_kept, inv_t, zmax, rdraw);
    if (t == 0) out_ids[b] = found == kTieAll ? 0 : found;
    return;
  }
  const int C = ((V + kThreads - 1) / kThreads + 7) / 8 * 8;
  const int i0 = t * C, i1 = min(V, i0 + C);
  auto kept_mass = [&](uint32_t bits, int id) -> int64_t {
    const uint32_t key = order_key(bits);
    const bool kept = key && (key > key_cut || (key == key_cut && (int64_t)id <= id_cut));
    return kept ? mass_of(exp_of(bits, inv_t, zmax)) : 0;
  };
  int64_t mine = 0;
  for_each_elem(row, V, vec_ok, [&](uint32_t bits, int id) { mine += kept_mass(bits, id); });
  __syncthreads();
  if (t == 0) s.b_id = -1;
  int64_t tot;
  int64_t cum = block_excl_scan(s, mine, &tot);
  if (cum <= rdraw && rdraw < cum + mine) {
    for (int i = i0; i < i1 && s.b_id < 0; i += 8) {
      uint32_t bits[8];
      load8(row, V, i, vec_ok, bits);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (i + k >= i1) break;
        cum += kept_mass(bits[k], i + k);
        if (cum > rdraw) { s.b_id = i + k; break; }
      }
    }
  }
  __syncthreads();
  if (t == 0) out_ids[b] = s.b_id >= 0 ? s.b_id : 0;
}

__global__ __launch_bounds__(kThreads) void sample_kernel(const bf16_t* __restrict__ logits, int64_t stride, int V,
                                                          const float* __restrict__ temps,
                                                          const float* __restrict__ top_ps,
                                                          const int32_t* __restrict__ top_ks,
                                                          const float* __restrict__ min_ps,
                                                          const float* __restrict__ uniforms, int flags,
                                                          int64_t* __restrict__ out_ids) {
  __shared__ Shared s;
  __shared__ FastShared fs;
  sample_row(s, fs, blockIdx.x, logits, stride, V, temps, top_ps, top_ks, min_ps, uniforms, flags, out_ids);
}

// ---------------------------------------------------------------------------
// All-greedy batches over several workgroups per row (a small batch would
// leave most CUs idle with one workgroup per row).  A lane keeps the largest
// order key of its ids (-0 folded into +0, which torch.argmax treats as equal)
// and the lowest id holding it, and its lowest NaN id, as the one-workgroup
// path does with float compares.  Each workgroup
// then folds its best into the row's 64-bit slot with one atomic max of
//   order key << 32 | (2^32 - 1 - id)      (greedy_word: NaN above every value)
// (as torch.argmax: a NaN wins, then the largest logit, among equals the lowest id) and counts
// itself in the row's arrival counter; the last workgroup of the row writes the id
// and clears both words for the next call.  Every atomic is awaited before
// the next one is issued, so the count is only bumped after the workgroup's
// max has been performed.  Atomics on one cache line serialise, so each row
// has its own line and is cut into at most 32 segments.
// A lane's greedy candidate as one word that an integer max orders like
// torch.argmax: key << 32 | (2^32 - 1 - id).  A NaN (nid >= 0, the lane's
// lowest NaN id) takes key 0xffff, above every value's order key (at most
// 0xff80, +inf); otherwise the lane's max value fm at its lowest id bid.  0
// means no candidate.
XV_INLINE unsigned long long greedy_word(float fm, int bid, int nid) {
  if (nid >= 0) return (0xffffull << 32) | (0xffffffffu - (uint32_t)nid);
  if (bid < 0) return 0ull;
  const uint32_t fb = __float_as_uint(fm) >> 16;
  return ((unsigned long long)order_key(fb == 0x8000u ? 0u : fb) << 32) | (0xffffffffu - (uint32_t)bid);
}

constexpr int kGreedyThreads = 256;
constexpr int kGreedyUnroll = 2;  // 8-id vectors per lane per step (2, 4, 6, 8, 16 measured)
constexpr int kGreedyLine = 16;  // u64 words per row: its slot, then its arrival counter, one 128-byte line

__global__ __launch_bounds__(kGreedyThreads) void greedy_segment_kernel(const bf16_t* __restrict__ logits,
                                                                        int64_t stride, int V, int seg_len,
                                                                        unsigned long long* __restrict__ slots,
                                                                        unsigned int* __restrict__ arrivals,
                                                                        int64_t* __restrict__ out_ids) {
  const int b = blockIdx.y;
  const bf16_t* row = logits + (int64_t)b * stride;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  const int beg = blockIdx.x * seg_len, end = min(V, beg + seg_len);
  // The lane's best as an order key with -0 folded into +0 (torch.argmax
  // treats them as equal), its lowest id, and its lowest NaN id.  A vector's
  // keys are computed two per packed op; only a vector whose largest key
  // beats the lane's best is searched id by id, and a vector holding a NaN
  // or padding (keys outside [0x7f, 0xff80]) goes id by id as well.
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  const u16x2 top2 = {(unsigned short)0x8000u, (unsigned short)0x8000u}, one2 = {(unsigned short)1u, (unsigned short)1u};
  uint32_t bk = 0;
  int bid = -1, nid = -1;
  constexpr int step = kGreedyThreads * 8;
  for (int i0 = beg + threadIdx.x * 8; i0 < end; i0 += kGreedyUnroll * step) {
    uint32_t w[kGreedyUnroll][4];
#pragma unroll
    for (int u = 0; u < kGreedyUnroll; ++u) {
      const int i = i0 + u * step;
      if (i < end && vec_ok && i + 8 <= end) {
        const Vec8 x = load_vec8(row + i);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[u][k] = x.w[k];
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          w[u][k] = (i + 2 * k < end ? (uint32_t)row[i + 2 * k] : 0xffffu) |
                    (i + 2 * k + 1 < end ? (uint32_t)row[i + 2 * k + 1] : 0xffffu) << 16;
      }
    }
#pragma unroll
    for (int u = 0; u < kGreedyUnroll; ++u) {
      const int i = i0 + u * step;
      if (i >= end) break;
      uint32_t kk[4];
      u16x2 hi2 = {(unsigned short)0u, (unsigned short)0u}, lo2 = {(unsigned short)0xffffu, (unsigned short)0xffffu};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        u16x2 w2 = __builtin_bit_cast(u16x2, w[u][k]);
        w2 = w2 * __builtin_elementwise_min(w2 ^ top2, one2);  // -0 (0x8000) -> +0
        const u16x2 sg = __builtin_bit_cast(u16x2, (s16x2)(__builtin_bit_cast(s16x2, w2) >> (short)15));
        const u16x2 k2 = w2 ^ (sg | top2);
        kk[k] = __builtin_bit_cast(uint32_t, k2);
        hi2 = __builtin_elementwise_max(hi2, k2);
        lo2 = __builtin_elementwise_min(lo2, k2);
      }
      const uint32_t vmax = max((uint32_t)hi2.x, (uint32_t)hi2.y), vmin = min((uint32_t)lo2.x, (uint32_t)lo2.y);
      if (vmax > 0xff80u || vmin < 0x7fu) {  // NaN or padding: id by id
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t key = (kk[k >> 1] >> (16 * (k & 1))) & 0xffffu;
          const bool real = i + k < end;
          const bool nan = real && (key > 0xff80u || key < 0x7fu);
          nid = (nid < 0 && nan) ? i + k : nid;
          const bool better = real && !nan && key > bk;
          bid = better ? i + k : bid;
          bk = better ? key : bk;
        }
      } else if (vmax > bk) {  // the lowest id holding the vector's largest key
        int first = 7;
#pragma unroll
        for (int k = 7; k >= 0; --k) first = ((kk[k >> 1] >> (16 * (k & 1))) & 0xffffu) == vmax ? k : first;
        bk = vmax;
        bid = i + first;
      }
    }
  }
  unsigned long long best = 0;
  if (nid >= 0) best = (0xffffull << 32) | (0xffffffffu - (uint32_t)nid);
  else if (bid >= 0) best = ((unsigned long long)bk << 32) | (0xffffffffu - (uint32_t)bid);
  best = wave_max_ull(best);
  __shared__ unsigned long long wbest[kGreedyThreads / 64];
  if ((threadIdx.x & 63) == 0) wbest[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kGreedyThreads / 64; ++w) best = wbest[w] > best ? wbest[w] : best;
    const unsigned int waves = gridDim.x;  // arrivals per row: one per workgroup
    // returning atomics: each result is awaited before the next is issued
    unsigned long long seen = 0;
    unsigned long long* slot = slots + (int64_t)b * kGreedyLine;
    unsigned int* arrival = arrivals + (int64_t)b * 2 * kGreedyLine;
    if (best) seen = __hip_atomic_fetch_max(slot, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (a slot never holds all ones -- keys fit 16 bits -- so the increment is 1,
    // but it depends on the max's result, which keeps the two in order)
    const unsigned int inc = seen == ~0ull ? 0u : 1u;
    const unsigned int n = __hip_atomic_fetch_add(arrival, inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (n == waves - 1) {
      const unsigned long long c = __hip_atomic_fetch_max(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      out_ids[b] = c ? (int64_t)(0xffffffffu - (uint32_t)c) : 0;  // (a row always has a candidate)
      __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(arrival, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}


// ---------------------------------------------------------------------------
// Sampled rows over several workgroups per row (batches given a workspace).
//
// A candidate's mass depends on its bf16 key alone, so exact counts per key
// replace per-id masses: the row is cut into R segments of whole 8-id vectors
// and two launches sample it (a launch boundary makes one kernel's global
// writes visible to the next, across XCDs):
//   1. seg_count:  one workgroup per segment counts its logits by value: the
//                  8192 keys of magnitudes in [2^-22, 2^10) exactly, zeros,
//                  smaller magnitudes (listed), larger ones; greedy rows take
//                  the segment's best instead;
//   2. row_count:  one workgroup per row sums the segments' counts, evaluates
//                  one exp2 per key, cuts by ranks and masses over the keys,
//                  takes each segment's kept mass from its own counts, and
//                  draws: the segment holding floor(u * M), then the id in it.
// The masses and their sums are exact integers, so cuts and draws are those
// of the one-workgroup path and the ids are identical to it.
// Top-p 0.95 at V 151936, 32 rows: 7 + 16 us, 27.9 us a call with its gaps.
// Three launches (row extremes, 256-bucket mass histograms, one workgroup per
// row gathering the cut's bucket from the whole row) took 4.7 + 13.1 + 35.6,
// 58.6 a call; 52.3 -> 20.9 us a call in a captured loop, 1 row 42.0 -> 18.0,
// 512 rows 224 -> 80, and rows whose cut bucket overflowed LDS (a spread of
// 2.5 at 256 rows) 861 -> 42.

constexpr int kSegThreads = 256;
constexpr int kSegWaves = kSegThreads / 64;
#ifndef XV_SEG_MAX
#define XV_SEG_MAX 32
#endif
#ifndef XV_SEG_CHUNK
#define XV_SEG_CHUNK 4
#endif
constexpr int kMaxSegs = XV_SEG_MAX;
constexpr int kSegChunk = XV_SEG_CHUNK;
// Rows of the multi-workgroup sampled path; larger batches take one workgroup
// per row (top-p at V 151936: 80 us at 512 rows, 605 at 600), since the
// workspace of a batch reserves 64 KB and more per row.
constexpr int kSegMaxBatch = 512;
// Segments per row of the counting path: more split the counting and the draw
// further, but the row's workgroup reads 16 KB of counts for each (32 rows of
// 151936: 4 segments 23.2 us, 8 20.7, 12 24.0, 16 24.4).  Large batches take
// fewer, about kCntTarget workgroups in all (256 rows: 512 workgroups 42.4,
// 1024 41.4, 2048 42.8).
constexpr int kCntSegs = 8;
constexpr int kCntTarget = 1024;

struct SegArgs {
  const bf16_t* logits;
  int64_t stride;
  int V, R, seg_len, flags;
  const float* temps;
  const float* top_ps;
  const int32_t* top_ks;
  const float* min_ps;
  const float* uniforms;
  int64_t* out_ids;
  unsigned long long* seg_best; // [B * R] greedy (key << 32 | ~id)
  uint32_t* seg_cnt;            // [B * R * kSegWords]
  unsigned long long* cand;     // top-k path: [B * cand_stride]
  int64_t cand_stride;          // R * kTopList
};

struct RowParams {
  bool greedy, use_k, use_p, use_m;
  int top_k;
  float temp, top_p, min_p;
};
XV_INLINE RowParams row_params(const SegArgs& a, int b) {
  RowParams p;
  p.temp = a.temps[b];
  p.greedy = p.temp <= 1e-5f;
  p.top_k = ((a.flags & XV_SAMPLE_USE_TOP_K) && a.top_ks) ? a.top_ks[b] : a.V;
  p.top_p = ((a.flags & XV_SAMPLE_USE_TOP_P) && a.top_ps) ? a.top_ps[b] : 1.0f;
  p.min_p = ((a.flags & XV_SAMPLE_USE_MIN_P) && a.min_ps) ? a.min_ps[b] : 0.0f;
  // No candidate reaches a min-p above 1 (the largest logit's ratio is
  // exactly 1), and the kept set is then the first candidate alone, as a
  // top-k of 1 keeps it.
  if (p.min_p > 1.0f) p.top_k = 1;
  p.use_k = p.top_k > 0 && p.top_k < a.V;
  p.use_p = p.top_p < 1.0f;
  p.use_m = p.min_p > 0.0f;
  return p;
}

// f(bits, id) for every id of segment [beg, end) on every lane: vector vi of
// the segment is (c * kSegChunk + v) * kThreads + t; ids ascend within a lane;
// slots of the last vector outside the segment come as 0xffff (key 0).
template <typename F>
XV_INLINE void for_seg(const bf16_t* row, bool vec_ok, int beg, int end, F&& f) {
  const int nvec = (end - beg + 7) / 8;
  for (int c = 0; c * kSegChunk * kThreads < nvec; ++c) {
    uint32_t w[kSegChunk][4];
#pragma unroll
    for (int v = 0; v < kSegChunk; ++v) {
      const int base = beg + ((c * kSegChunk + v) * kThreads + (int)threadIdx.x) * 8;
      if (base < end) load8_words(row, end, base, vec_ok, w[v]);
    }
#pragma unroll
    for (int v = 0; v < kSegChunk; ++v) {
      const int base = beg + ((c * kSegChunk + v) * kThreads + (int)threadIdx.x) * 8;
      if (base < end)
#pragma unroll
        for (int k = 0; k < 8; ++k) f(bits_of(w[v], k), base + k);
    }
  }
}

// A segment's counts in the workspace: kSegWords words, the 16-bit counts of
// the 2 * kMagBins window keys in descending order (position pos < kMagBins:
// the positive magnitude kMagLo + kMagBins - 1 - pos, past it the negative one
// kMagLo + pos - kMagBins; two to a word), then the header, then up to
// kTinyList 16-bit logits of magnitudes in (0, 2^-22) and as many of 2^10 and
// above: those that can have mass beside the segment's largest.
constexpr int kMagBins = 4096;                  // 32 octaves of 128 bf16 magnitudes
constexpr uint32_t kMagLo = (127 - 22) << 7;    // 2^-22; the window ends at 2^10
constexpr uint32_t kInfMag = 0x7f80u;
constexpr int kTinyList = 64;
constexpr int kMaxSegIds = 65528;               // a count fits 16 bits
// header words; kHFarMag and kHFirst hold 0xffff - value (a cleared word is
// "none"), kHTopMax the largest value of 2^10 and above (raw bits), kHTop the
// count of those listed
enum : int { kHPosZero = 0, kHNegZero, kHFar, kHFarMag, kHTop, kHTiny, kHFirst, kHTopMax, kHWords = 8 };
constexpr int kTopsAt = kMagBins + kHWords + kTinyList / 2;  // the list of values of 2^10 and above
constexpr int kSegWords = (kTopsAt + kTinyList / 2 + 63) / 64 * 64;
// A value this many temperatures below another has no mass beside it (2^40
// 2^d is below 1 at 27.8; the rest is rounding of d: where l / T is large
// enough for more, so is the step between bf16 values).
constexpr float kMasslessT = 28.5f;
// Window position of raw bits with m = magnitude - kMagLo < kMagBins, and back.
XV_INLINE uint32_t window_pos(uint32_t bits, uint32_t m) {
  return (bits & 0x8000u) ? (uint32_t)kMagBins + m : (uint32_t)(kMagBins - 1) - m;
}
XV_INLINE uint32_t pos_bits(int pos) {
  return pos < kMagBins ? kMagLo + (uint32_t)(kMagBins - 1 - pos) : 0x8000u | (kMagLo + (uint32_t)(pos - kMagBins));
}

// One workgroup per segment counts the segment's logits by value.  Bound by
// the LDS atomics and its two ends (clearing and writing 16 KB): 16-bit
// counts, two to a word, halve both against 32-bit ones.
__global__ __launch_bounds__(kThreads) void seg_count_kernel(SegArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t h[kSegWords];
  __shared__ unsigned long long wbest[kWaves];
  const int b = blockIdx.y, r = blockIdx.x, t = threadIdx.x, lane = t & 63;
  const bf16_t* row = a.logits + (int64_t)b * a.stride;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  const int beg = r * a.seg_len, end = min(a.V, beg + a.seg_len);
  if (a.temps[b] <= 1e-5f) {  // greedy row: the segment's best (torch.argmax: NaN, else value; lowest id)
    float fm = -INFINITY;
    int bid = -1, nid = -1;
    for_seg(row, vec_ok, beg, end, [&](uint32_t bits, int id) {
      const float v = bf16_to_f32(bits);  // NaN (and padding) never compares greater
      const bool better = v > fm;         // ids ascend within a lane: keeps the lowest
      fm = better ? v : fm;
      bid = better ? id : bid;
      nid = (nid < 0 && id < end && !order_key(bits)) ? id : nid;
    });
    unsigned long long best = wave_max_ull(greedy_word(fm, bid, nid));
    if (lane == 0) wbest[t >> 6] = best;
    __syncthreads();
    if (t < 64) {
      best = wave_max_ull(t < kWaves ? wbest[t] : 0ull);
      if (t == 0) a.seg_best[b * a.R + r] = best;
    }
    return;
  }
  uint4* h4 = reinterpret_cast<uint4*>(h);
  for (int i = t; i < kSegWords / 4; i += kThreads) h4[i] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  uint32_t* head = h + kMagBins;
  uint16_t* tiny = reinterpret_cast<uint16_t*>(head + kHWords);
  // few-valued kinds of logits count in registers: masked rows hold thousands of one of them
  uint32_t pz = 0, nz = 0, far = 0, far_mag = 0xffffu;
  for_seg(row, vec_ok, beg, end, [&](uint32_t bits, int) {
    const uint32_t mag = bits & 0x7fffu, m = mag - kMagLo;
    if (m < (uint32_t)kMagBins) {
      const uint32_t i = window_pos(bits, m);
      atomicAdd(&h[i >> 1], (i & 1) ? 0x10000u : 1u);
    } else if (mag <= kInfMag) {  // NaN (and padding) drops out
      if (mag >= kMagLo) {
        if (bits & 0x8000u) {
          ++far;
          far_mag = min(far_mag, mag);
        } else {
          head[kHTopMax] = 1u;  // found below
        }
      } else if (mag == 0u) {
        if (bits) ++nz; else ++pz;
      } else {
        const uint32_t i = atomicAdd(&head[kHTiny], 1u);
        if (i < (uint32_t)kTinyList) tiny[i] = (uint16_t)bits;
      }
    }
  });
  if (__ballot(pz | nz)) {
    pz = (uint32_t)wave_sum_l(pz);
    nz = (uint32_t)wave_sum_l(nz);
    if (lane == 0) {
      atomicAdd(&head[kHPosZero], pz);
      atomicAdd(&head[kHNegZero], nz);
    }
  }
  if (__ballot(far)) {
    far = (uint32_t)wave_sum_l(far);
    far_mag = wave_min_u(far_mag);
    if (lane == 0) {
      atomicAdd(&head[kHFar], far);
      atomicMax(&head[kHFarMag], 0xffffu - far_mag);
    }
  }
  __syncthreads();
  uint4* o = reinterpret_cast<uint4*>(a.seg_cnt + ((int64_t)b * a.R + r) * kSegWords);
  static_assert(kMagBins == 4 * kThreads && kSegWords / 4 - kThreads <= 64, "four words per thread, the rest by wave 0");
  const uint4 v = h4[t];
  o[t] = v;
  const uint32_t at = v.x ? 8 * t + (v.x & 0xffffu ? 0 : 1)
                          : v.y ? 8 * t + (v.y & 0xffffu ? 2 : 3)
                                : v.z ? 8 * t + (v.z & 0xffffu ? 4 : 5)
                                      : v.w ? 8 * t + (v.w & 0xffffu ? 6 : 7) : 0xffffu;
  const uint32_t first = wave_min_u(at);
  if (lane == 0) wbest[t >> 6] = 0xffffu - first;
  if (XV_UNLIKELY(head[kHTopMax])) {  // (uniform) the largest value of 2^10 and above, then those that can have mass beside it
    auto each_top = [&](auto&& f) {
      for_seg(row, vec_ok, beg, end, [&](uint32_t bits, int) {
        if (bits >= kMagLo + (uint32_t)kMagBins && bits <= kInfMag) f(bits);
      });
    };
    uint32_t top = 0;
    each_top([&](uint32_t bits) { top = max(top, bits); });
    top = wave_max_u(top);
    __syncthreads();  // every thread has read the flag
    if (lane == 0) atomicMax(&head[kHTopMax], top);
    __syncthreads();
    const float least = bf16_to_f32(head[kHTopMax]) - kMasslessT * a.temps[b];
    uint16_t* tops = reinterpret_cast<uint16_t*>(h + kTopsAt);
    each_top([&](uint32_t bits) {
      if (!(bf16_to_f32(bits) >= least)) return;
      const uint32_t i = atomicAdd(&head[kHTop], 1u);
      if (i < (uint32_t)kTinyList) tops[i] = (uint16_t)bits;
    });
  }
  __syncthreads();
  if (t < kSegWords / 4 - kThreads) {
    uint4 x = h4[kThreads + t];
    uint32_t f = 0;
    for (int i = 0; i < kWaves; ++i) f = max(f, (uint32_t)wbest[i]);
    if (t == kHFirst / 4) x.z = f;  // word kHFirst
    o[kThreads + t] = x;
  }
}

// List operations on at most 64 candidates held one per lane, by one wave
// (no workgroup barriers).
//
// Bitonic sort of the wave, descending; zeros (padding) sort last.
XV_INLINE unsigned long long wave_sort_desc(unsigned long long c) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int size = 2; size <= 64; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const unsigned long long o = xor_lane64(c, stride);
      const bool take_max = ((lane & size) == 0) == ((lane & stride) == 0);
      c = take_max ? (o > c ? o : c) : (o < c ? o : c);
    }
  return c;
}
// 32-bit forms of the list operations, for lists whose words order as the
// 64-bit candidate words do (a segment's key << 13 | (8191 - offset of the id
// in the segment), the row merge's key << 16 | index): each compare-exchange
// stage then moves and selects one register, not two.
XV_INLINE uint32_t xor_lane(uint32_t x, int s) {  // s a constant after unrolling
  switch (s) {
    case 1: return xor_lane<1>(x);
    case 2: return xor_lane<2>(x);
    case 4: return xor_lane<4>(x);
    case 8: return xor_lane<8>(x);
    case 16: return xor_lane<16>(x);
    default: return xor_lane<32>(x);
  }
}
XV_INLINE uint32_t wave_sort_desc32(uint32_t c) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int size = 2; size <= 64; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const uint32_t o = xor_lane(c, stride);
      const bool take_max = ((lane & size) == 0) == ((lane & stride) == 0);
      c = take_max ? max(o, c) : min(o, c);
    }
  return c;
}
template <int S>
XV_INLINE uint32_t merge_stage32(uint32_t c) {  // the larger to the lane with bit S clear
  const uint32_t o = xor_lane<S>(c);
  return (threadIdx.x & S) ? min(o, c) : max(o, c);
}
// Top 64 of two lists sorted descending (lane j holds element j of each):
// the elementwise max against the reversed second list is bitonic and holds
// the top 64; six compare-exchange stages sort it descending.  y[63 - lane]
// is row_mirror (lane i of a row reads lane 15 - i), then the row swaps.
XV_INLINE uint32_t merge_top64_32(uint32_t x, uint32_t y) {
  const uint32_t c = max(x, xor_lane<32>(xor_lane<16>(dpp_u<0x140>(y))));
  return merge_stage32<1>(merge_stage32<2>(merge_stage32<4>(merge_stage32<8>(merge_stage32<16>(merge_stage32<32>(c))))));
}

// First lane whose predicate holds, `none` if no lane's does.
XV_INLINE int64_t wave_first(bool pred, int64_t none) {
  const unsigned long long m = __ballot(pred);
  return m ? (int64_t)__builtin_ctzll(m) : none;
}

// The cut and the draw of a row's top_k list of n <= 64 candidates, sorted
// descending (lane j's candidate c, 0 past n), by one wave.  kminp: the lowest
// listed key that reaches min_p (0xffffffff: none).
XV_INLINE void row_cut_wave_list(const SegArgs& a, const RowParams& p, float inv_t, float zmax, uint32_t kminp, int b,
                                 int n, unsigned long long c) {
  const int lane = threadIdx.x & 63;
  const int64_t q = lane < n ? cand_mass(c, inv_t, zmax) : 0;
  const int64_t incl = wave_incl_scan_l(q);
  const uint32_t key = cand_key(c);
  const int64_t total_k = wave_sum_l(lane < p.top_k ? q : 0);
  int64_t jcut = (int64_t)p.top_k - 1;
  if (p.use_p) {
    const int64_t thr = (int64_t)floor((double)p.top_p * (double)total_k);
    jcut = min(jcut, wave_first(lane < n && incl > thr, n));
  }
  const uint32_t last = cand_key(__shfl(c, n - 1));
  if (p.use_m && kminp != 0xffffffffu && kminp >= last)
    jcut = min(jcut, (int64_t)__popcll(__ballot(lane < n && key >= kminp)) - 1);
  if (jcut >= n) jcut = n - 1;
  if (jcut < 0) jcut = 0;
  const int64_t m_list = wave_sum_l(lane <= jcut ? q : 0);
  // the kept list in ascending id order: re-keyed (~id << 32 | key), sorted descending
  const float u = a.uniforms ? a.uniforms[b] : 0.5f;
  const int64_t rdraw = draw_point(u, m_list);
  // no mass in the list (z_max not finite, see lowest_id_of_key): its first candidate
  const int64_t first = cand_id(__shfl(c, 0));
  int64_t fid;
  if (a.V <= (1 << 26)) {
    // 32-bit words (0x3ffffff - id) << 6 | lane, sorted descending: ids
    // ascending, each word naming the lane that holds its mass
    uint32_t e = lane <= jcut ? (0x3ffffffu - (uint32_t)cand_id(c)) << 6 | (uint32_t)lane : 0u;
    e = wave_sort_desc32(e);
    const int64_t qe = (int64_t)__shfl((long long)q, (int)(e & 63u));
    const int64_t ie = wave_incl_scan_l(lane <= jcut ? qe : 0);
    const int64_t fi = wave_first(lane <= jcut && ie > rdraw, -1);
    const uint32_t ef = __shfl(e, fi < 0 ? 0 : (int)fi);
    fid = fi < 0 ? first : (int64_t)(0x3ffffffu - (ef >> 6));
  } else {
    unsigned long long e =
        lane <= jcut ? ((unsigned long long)(0xffffffffu - (uint32_t)cand_id(c)) << 32) | cand_key(c) : 0ull;
    e = wave_sort_desc(e);
    const int64_t qe = lane <= jcut ? mass_of(exp_of(key_to_bits((uint32_t)(e & 0xffffffffu)), inv_t, zmax)) : 0;
    const int64_t ie = wave_incl_scan_l(qe);
    const int64_t fi = wave_first(lane <= jcut && ie > rdraw, -1);
    const unsigned long long ef = __shfl(e, fi < 0 ? 0 : (int)fi);
    fid = fi < 0 ? first : (int64_t)(0xffffffffu - (uint32_t)(ef >> 32));
  }
  if (lane == 0) a.out_ids[b] = fid;
}

// ---------------------------------------------------------------------------
// Top-k path, for calls whose every row has 1 <= top_k <= kTopList (the
// caller's max_top_k; greedy rows too, since a row's argmax is its first
// candidate).  The order of candidates (key descending, id ascending) does not
// depend on the temperature, so a row's top kTopList candidates are the top
// kTopList of its segments' own top kTopList lists, and they hold everything
// a top-k row's cut and draw need: the row max (the first candidate), the
// masses of the top-k set, the min-p key within it.  Two launches and one pass
// over the logits:
//   seg_topk: per segment, its top kTopList candidates, sorted, into the row's
//             list (each wave selects from its own ids, wave 0 merges);
//   row_topk: per row, a tree of pairwise merges of the sorted segment lists
//             (bitonic, in registers, one wave per merge), then the argmax
//             (greedy rows) or the cut and draw of row_cut_wave (top-k rows).
// A row that does not meet the bound runs sample_row, so ids never depend on
// the caller's claim.
constexpr int kTopList = 64;
constexpr int kTopVecs = 4;  // 8-id vectors per thread in registers: segments of up to 8192 ids


// Each wave selects the top kTopList of its own ids (vectors v * kSegThreads
// + 64 w + lane of the segment, ids ascending in (v, lane, k) order) with no
// workgroup barrier: its largest key, a wave-private LDS histogram of the
// 256 keys below it (keys further down never touch LDS), the threshold key T
// from a scan of that histogram (a bit-by-bit count over all keys when fewer
// than kTopList lie that close), then a compaction by per-lane masks into a
// 32-bit list it sorts.  Wave 0 merges the four sorted wave lists and writes
// the segment's list as 64-bit candidate words.
__global__ __launch_bounds__(kSegThreads) void seg_topk_kernel(SegArgs a) {
  static_assert(kMaxSegs * kTopList <= kMaxCand, "the segment lists fit the row's list");
  __shared__ uint32_t hist[kSegWaves][256];
  static_assert(kTopVecs * 8 * kSegThreads <= 8192, "segment offsets fit the 13 bits of a list entry");
  __shared__ uint32_t wl[kSegWaves][kTopList];
  __shared__ uint4 kst[kTopVecs][kSegThreads];  // each thread's keys, packed as in kw
  const int b = blockIdx.y, r = blockIdx.x, t = threadIdx.x, w = t >> 6, lane = t & 63;
  const bf16_t* row = a.logits + (int64_t)b * a.stride;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  const int beg = r * a.seg_len, end = min(a.V, beg + a.seg_len);
  const int nv = ((end - beg + 7) / 8 + kSegThreads - 1) / kSegThreads;  // <= kTopVecs (checked by the host)
  // Whole 16-byte vectors first, every load issued before any is used; then
  // the ids of a partial vector (at most one lane) or of an unaligned row.
  uint32_t kw[kTopVecs][4];
#pragma unroll
  for (int v = 0; v < kTopVecs; ++v) {
    const int base = beg + (v * kSegThreads + t) * 8;
#pragma unroll
    for (int k = 0; k < 4; ++k) kw[v][k] = 0xffffffffu;
    if (v < nv && vec_ok && base + 8 <= end) {
      const Vec8 y = load_vec8(row + base);
#pragma unroll
      for (int k = 0; k < 4; ++k) kw[v][k] = y.w[k];
    }
  }
#pragma unroll
  for (int v = 0; v < kTopVecs; ++v) {
    const int base = beg + (v * kSegThreads + t) * 8;
    if (v < nv && !(vec_ok && base + 8 <= end) && base < end) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        kw[v][k] = (base + 2 * k < end ? (uint32_t)row[base + 2 * k] : 0xffffu) |
                   (base + 2 * k + 1 < end ? (uint32_t)row[base + 2 * k + 1] : 0xffffu) << 16;
    }
  }
  // Order keys, two per packed 16-bit op: x ^ 0x8000 for a sign bit of 0,
  // ~x for 1 (order_key's map on non-NaN values).  Finite keys lie in
  // [0x7f, 0xff80]; NaN bits land outside, as do the padding words (0xffff
  // gives key 0).  A lane holding any such key redoes them one at a time:
  // NaN takes key 0 (dropped), except in a greedy row, which is
  // torch.argmax: its NaNs (real ids only) take key 0xffff, above every value,
  // so the list's first entry is the lowest NaN id when there is one.
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  const u16x2 top2 = {(unsigned short)0x8000u, (unsigned short)0x8000u};
  u16x2 hi2 = {(unsigned short)0u, (unsigned short)0u}, lo2 = {(unsigned short)0xffffu, (unsigned short)0xffffu};
#pragma unroll
  for (int v = 0; v < kTopVecs; ++v)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (v >= nv) {
        kw[v][k] = 0u;
        continue;
      }
      const u16x2 w2 = __builtin_bit_cast(u16x2, kw[v][k]);
      const u16x2 sg = __builtin_bit_cast(u16x2, (s16x2)(__builtin_bit_cast(s16x2, w2) >> (short)15));
      const u16x2 k2 = w2 ^ (sg | top2);
      kw[v][k] = __builtin_bit_cast(uint32_t, k2);
      hi2 = __builtin_elementwise_max(hi2, k2);
      lo2 = __builtin_elementwise_min(lo2, k2);
    }
  uint32_t kmax = max((uint32_t)hi2.x, (uint32_t)hi2.y);
  if (kmax > 0xff80u || min((uint32_t)lo2.x, (uint32_t)lo2.y) < 0x7fu) {
    const bool greedy = a.temps[b] <= 1e-5f;
    kmax = 0;
#pragma unroll
    for (int v = 0; v < kTopVecs; ++v)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t k0 = kw[v][k] & 0xffffu, k1 = kw[v][k] >> 16;
        const int id0 = beg + (v * kSegThreads + t) * 8 + 2 * k;
        if (k0 > 0xff80u || k0 < 0x7fu) k0 = greedy && v < nv && id0 < end ? 0xffffu : 0u;
        if (k1 > 0xff80u || k1 < 0x7fu) k1 = greedy && v < nv && id0 + 1 < end ? 0xffffu : 0u;
        kw[v][k] = k0 | k1 << 16;
        kmax = max(kmax, max(k0, k1));
      }
  }
  auto key_at = [&](int v, int k) { return (kw[v][k >> 1] >> (16 * (k & 1))) & 0xffffu; };
  kmax = wave_max_u(kmax);
  // count of this wave's keys >= x (wave uniform)
  auto count_ge = [&](uint32_t x) {
    int c = 0;
#pragma unroll
    for (int v = 0; v < kTopVecs; ++v)
      if (v < nv)
#pragma unroll
        for (int k = 0; k < 8; ++k) c += __popcll(__ballot(key_at(v, k) >= x));
    return c;
  };
  uint32_t T = 1;    // threshold key: every key > T is taken, and need_eq keys == T
  int need_eq = kTopList, n_eq = 0;
  if (kmax == 0) {
    T = 0xffffffffu;  // nothing but NaN: an empty list
    need_eq = 0;
  } else {
    // histogram of keys kmax - j, j = 0..255, in this wave's LDS row
    const uint32_t lo = kmax > 256u ? kmax - 255u : 1u;  // key 0 (NaN, padding) never counts
#pragma unroll
    for (int j = 0; j < 4; ++j) hist[w][lane + 64 * j] = 0u;
    // distances below kmax two at a time (no wrap: no key exceeds kmax), and
    // their byte offsets (which wrap only for distances past the range)
    const uint32_t span = kmax - lo;
    const u16x2 kmax2 = {(unsigned short)kmax, (unsigned short)kmax};
    char* const hrow = reinterpret_cast<char*>(&hist[w][0]);
#pragma unroll
    for (int v = 0; v < kTopVecs; ++v)
      if (v < nv)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u16x2 d2 = kmax2 - __builtin_bit_cast(u16x2, kw[v][j]);
          const u16x2 o2 = d2 << (unsigned short)2;
          if (d2.x <= span) atomicAdd(reinterpret_cast<uint32_t*>(hrow + o2.x), 1u);
          if (d2.y <= span) atomicAdd(reinterpret_cast<uint32_t*>(hrow + o2.y), 1u);
        }
    // lane l holds bins 4l .. 4l + 3 (keys kmax - 4l downwards)
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = hist[w][4 * lane + j];
    const int mine = (int)(h[0] + h[1] + h[2] + h[3]);
    const int incl = wave_incl_scan_i(mine);
    const int total = __shfl(incl, 63);
    if (total >= kTopList) {
      const int l = (int)wave_first(incl >= kTopList, 63);
      int above = __shfl(incl - mine, l);
      const uint32_t h0 = __shfl(h[0], l), h1 = __shfl(h[1], l), h2 = __shfl(h[2], l), h3 = __shfl(h[3], l);
      const uint32_t hh[4] = {h0, h1, h2, h3};
      int j = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (j == q && above + (int)hh[q] < kTopList) { above += (int)hh[q]; j = q + 1; }
      T = kmax - (uint32_t)(4 * l + j);
      n_eq = (int)(j == 0 ? h0 : j == 1 ? h1 : j == 2 ? h2 : h3);
      need_eq = kTopList - above;
    } else {
      // fewer than kTopList keys within 256 of the largest: the largest x
      // with count(keys >= x) >= kTopList, bit by bit (or every key)
      const int all = count_ge(1u);
      if (all <= kTopList) {  // every key: key > 0 selects them, no ranking
        T = 0;
        need_eq = 0;
      } else {
        uint32_t x = 0;
        for (int bit = 15; bit >= 0; --bit) {
          const uint32_t y = x | (1u << bit);
          if (count_ge(y) >= kTopList) x = y;
        }
        T = x;
        const int gt = count_ge(x + 1);
        need_eq = kTopList - gt;
        n_eq = count_ge(x) - gt;
      }
    }
  }
  // Compaction: keys > T, and keys == T in id order up to need_eq of them.
  // Each lane marks what it takes in a 32-bit mask (bit 4v + j: key 2j of
  // vector v, bit 16 + 4v + j: key 2j + 1), two keys per packed 16-bit
  // compare; one wave scan of the counts gives each lane its slots, and a
  // lane writes only its own candidates, reading their keys back from LDS.
  const bool rank_eq = n_eq > need_eq;
  const u16x2 one2 = {(unsigned short)1u, (unsigned short)1u};
  uint32_t take = 0;
  if (T != 0xffffffffu) {
    // without ranking every key >= T is taken (keys > 0 when T is 0)
    const uint32_t tg = rank_eq ? T : (T ? T - 1u : 0u);
    const u16x2 tg2 = {(unsigned short)tg, (unsigned short)tg};
    const u16x2 t2 = {(unsigned short)T, (unsigned short)T};
    uint32_t ne = 0, valid = 0;  // ne: keys != T
#pragma unroll
    for (int v = 0; v < kTopVecs; ++v) {
      if (v >= nv) break;
      valid |= 0x000f000fu << (4 * v);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u16x2 k2 = __builtin_bit_cast(u16x2, kw[v][j]);
        take |= __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_sub_sat(k2, tg2), one2))
                << (4 * v + j);
        if (rank_eq) ne |= __builtin_bit_cast(uint32_t, __builtin_elementwise_min(k2 ^ t2, one2)) << (4 * v + j);
      }
    }
    if (rank_eq) {
      // keys == T (T > 0 here, so never padding), ranked in id order: vector,
      // then lane, then key.  Per-vector counts in 16-bit fields of one word
      // (a wave holds at most 512 per vector), one scan for all four.
      const uint32_t eq = ~ne & valid;
      uint64_t pc = 0;
#pragma unroll
      for (int v = 0; v < kTopVecs; ++v) pc |= (uint64_t)__popc(eq & (0x000f000fu << (4 * v))) << (16 * v);
      const uint64_t inc = (uint64_t)wave_incl_scan_l((int64_t)pc);
      const uint64_t tot = (uint64_t)__shfl((long long)inc, 63);
      // first rank of each vector's keys in this lane: the wave's counts in
      // earlier vectors plus the lower lanes' in this one
      uint64_t first = inc - pc, run = 0;
#pragma unroll
      for (int v = 0; v < kTopVecs; ++v) {
        first += run << (16 * v);
        run += (tot >> (16 * v)) & 0xffffu;
      }
      for (uint32_t m = eq; m; m &= m - 1) {
        const int bit = __builtin_ctz(m), v = (bit & 15) >> 2, j = bit & 3;
        // this lane's keys == T of vector v at lower ids: pairs j' < j, and key 2j if this is 2j + 1
        const uint32_t lower = ((((1u << j) - 1u) * 0x00010001u) << (4 * v)) | ((bit >> 4) ? 1u << (bit & 15) : 0u);
        const int rank = (int)((first >> (16 * v)) & 0xffffu) + __popc(eq & lower);
        if (rank < need_eq) take |= 1u << bit;
      }
    }
  }
  // this lane's keys, for reading back by position
#pragma unroll
  for (int v = 0; v < kTopVecs; ++v)
    if (v < nv) kst[v][t] = make_uint4(kw[v][0], kw[v][1], kw[v][2], kw[v][3]);
  const int mine = __popc(take);
  const int incl = wave_incl_scan_i(mine);
  const int filled = __shfl(incl, 63);
  int slot = incl - mine;
  for (uint32_t m = take; m; m &= m - 1, ++slot) {
    const int bit = __builtin_ctz(m), v = (bit & 15) >> 2, k = 2 * (bit & 3) + (bit >> 4);
    const uint32_t key = reinterpret_cast<const unsigned short*>(&kst[v][t])[k];
    wl[w][slot] = key << 13 | (8191u - (uint32_t)((v * kSegThreads + t) * 8 + k));
  }
  uint32_t c = lane < filled ? wl[w][lane] : 0u;
  c = wave_sort_desc32(c);
  wl[w][lane] = c;
  __syncthreads();
  if (w == 0) {
    const uint32_t m = merge_top64_32(merge_top64_32(c, wl[1][lane]), merge_top64_32(wl[2][lane], wl[3][lane]));
    // back to the row's candidate word (key << 32 | ~id); 0 stays padding
    const uint32_t id = (uint32_t)beg + (8191u - (m & 8191u));
    a.cand[(int64_t)b * a.cand_stride + (int64_t)r * kTopList + lane] =
        m ? ((unsigned long long)(m >> 13) << 32) | (unsigned long long)(0xffffffffu - id) : 0ull;
  }
}

__global__ __launch_bounds__(kThreads) void row_topk_kernel(SegArgs a) {
  static_assert(kMaxSegs <= 2 * kWaves, "one merge per wave on the first level");
  __shared__ Shared s;
  __shared__ FastShared fs;
  const int b = blockIdx.x, t = threadIdx.x, w = t >> 6, lane = t & 63;
  const RowParams p = row_params(a, b);
  if (!p.greedy && !(p.use_k && p.top_k <= kTopList)) {  // outside the bound: the one-workgroup path
    sample_row(s, fs, b, a.logits, a.stride, a.V, a.temps, a.top_ps, a.top_ks, a.min_ps, a.uniforms,
               a.flags & ~XV_SAMPLE_ALL_GREEDY, a.out_ids);
    return;
  }
  const unsigned long long* list = a.cand + (int64_t)b * a.cand_stride;
  // The merges run on 32-bit words key << 16 | (0xffff - i), i the entry's
  // index r * kTopList + j in the row's lists (entry j of segment r's list):
  // lists are sorted and segments ascend in id, so for equal keys a lower i
  // is a lower id, and the words order as the candidates do.  The lists are
  // staged in fs.cand to map the merged words back.  Level 0: wave w merges
  // segment lists 2w and 2w + 1 (missing lists are empty); later levels
  // alternate between two halves of a word buffer, one barrier each.
  static_assert(kMaxSegs * kTopList <= 0x10000 && 2 * kWaves * kTopList <= kWaves * kBuckets, "word layout");
  uint32_t* ml = &fs.wcnt[0][0];
  auto word = [&](unsigned long long c, int i) { return c ? cand_key(c) << 16 | (0xffffu - (uint32_t)i) : 0u; };
  {
    const int i0 = (2 * w) * kTopList + lane, i1 = i0 + kTopList;
    const unsigned long long x = 2 * w < a.R ? list[i0] : 0ull;
    const unsigned long long y = 2 * w + 1 < a.R ? list[i1] : 0ull;
    fs.cand[i0] = x;
    fs.cand[i1] = y;
    ml[w * kTopList + lane] = merge_top64_32(word(x, i0), word(y, i1));
  }
  __syncthreads();
  int src = 0;
  for (int half = kWaves / 2; half >= 1; half >>= 1) {
    const int dst = src ^ (kWaves * kTopList);
    if (w < half)
      ml[dst + w * kTopList + lane] =
          merge_top64_32(ml[src + (2 * w) * kTopList + lane], ml[src + (2 * w + 1) * kTopList + lane]);
    src = dst;
    __syncthreads();
  }
  if (t >= 64) return;
  const uint32_t mw = ml[src + lane];
  const unsigned long long c = mw ? fs.cand[0xffffu - (mw & 0xffffu)] : 0ull;
  const int n = __popcll(__ballot(c != 0ull));
  const unsigned long long top = __shfl(c, 0);
  if (p.greedy || n == 0) {  // argmax (NaN first for greedy rows); a sampled row of NaN only: 0
    if (t == 0) a.out_ids[b] = n ? cand_id(top) : 0;
    return;
  }
  const float inv_t = 1.0f / p.temp;
  const float zmax = bf16_to_f32(key_to_bits(cand_key(top))) * inv_t;
  uint32_t kminp = 0xffffffffu;
  if (p.use_m && t < n) {
    const uint32_t key = cand_key(c);
    if (exp_of(key_to_bits(key), inv_t, zmax) >= p.min_p) kminp = key;
  }
  row_cut_wave_list(a, p, inv_t, zmax, wave_min_u(kminp), b, n, c);
}


// ---------------------------------------------------------------------------
// Per row, after seg_count: the cut and the draw from the counts.
//
// A candidate's mass depends on its key alone, so rank and mass prefixes over
// the window's positions give every cut exactly: the top-k rank, the first
// rank whose inclusive mass exceeds floor(top_p * mass), the rank of the
// lowest key that reaches min_p; the smallest of them cuts.  Between the
// positive and the negative window lie the zeros and the listed magnitudes
// below 2^-22 (`mid`: the maximum of a row shifted to 0, or of
// log-probabilities, lies there), before the positive window the listed
// values of 2^10 and above (`top`; those not listed have no mass, and nor has
// any value below them, so ranks without them give the same masses), after the
// negative one the values of -2^10 and below (`far`).  A cut in top or mid is
// found in the sorted list, the zeros of each sign counting as one key.  Rows
// the counts don't settle (more listed values than the lists hold, far values
// with mass, no value at all) run sample_row.
//
// One workgroup works alone on its CU, so the time is latency and issue, not
// bandwidth: wave w takes positions 256 w .. of each half, four per lane, so
// the dense octaves of usual rows spread over most waves; masses are held as
// doubles (integers of at most 2^40; products and sums over up to 8190 ids
// stay below 2^53, so the full-rate fp64 FMA replaces 64-bit integer products
// exactly); the masses go into an LDS table, which the draw reads instead of
// an exp2 per id.  The kernel keeps out of scratch memory: with any, its
// sixteen waves started over 3.6 us instead of 0.2, and the row took 18.8 us
// in place of 13.5 (the row loads of the one-workgroup code inside it run
// kChunk packed vectors at a time for that).
constexpr int kHalfPos = kMagBins;  // positions per half
constexpr int kCntLoads = 8;        // segments whose counts load together
static_assert(kHalfPos == 4 * kThreads, "four positions per thread and half");

struct RowCut {
  int pos;       // the cut key's position, window positions before it being kept whole; 2 * kMagBins: every one is
  int ties;      // ids of the cut key kept
  int64_t M;     // kept mass
  int n;         // rank of the cut (2^31 - 1: none)
  int in;        // the cut lies in a group, kInTop or kInMid: pos is the group's (0, kMagBins), n and M the rank and the
                 // mass before it (until `resolve` adds the group's), the cut the group's rank `ties`, or with ties 0
                 // its first rank whose inclusive mass exceeds `left`
};
enum : int { kInTop = 1, kInMid = 2 };
constexpr int kListMax = 64;  // listed values of the group a row's cut lies in: one per lane
struct RowShared {
  RowCut cut[3];  // the top-k set's end, top-p's cut, the row's cut
  int ccnt[32];        // totals of the chunks (half, wave)
  int64_t cmass[32];
  int nm[kWaves];
  unsigned long long segm[kMaxSegs];  // kept masses of the window keys before the cut's
  int64_t midq[kMaxSegs];
  int64_t topq[kMaxSegs];
  uint32_t list[kListMax];  // the group's listed values: order key << 16 | segment
  int lties[kMaxSegs];      // listed ids of the cut key
  int64_t left;
  int t0;        // the draw: the thread whose ids hold the draw point, its mass and ties before
  int tie;
  int64_t cum;
};

// Eight values per lane summed over the wave: lane l (a multiple of 8) gets
// the sum of value l / 8.  Each of the first three exchanges halves the values
// a lane still carries.
XV_INLINE int64_t wave_sum8(int64_t (&v)[8]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    v[k] = ((lane & 32) ? v[k + 4] : v[k]) + (int64_t)xor_lane64<32>((uint64_t)((lane & 32) ? v[k] : v[k + 4]));
#pragma unroll
  for (int k = 0; k < 2; ++k)
    v[k] = ((lane & 16) ? v[k + 2] : v[k]) + (int64_t)xor_lane64<16>((uint64_t)((lane & 16) ? v[k] : v[k + 2]));
  int64_t x = ((lane & 8) ? v[1] : v[0]) + (int64_t)xor_lane64<8>((uint64_t)((lane & 8) ? v[0] : v[1]));
  x += (int64_t)xor_lane64<4>((uint64_t)x);
  x += (int64_t)xor_lane64<2>((uint64_t)x);
  return x + (int64_t)xor_lane64<1>((uint64_t)x);
}

// A mass as a double: the same integer as mass_of's.
XV_INLINE double mass_d(float e) { return __builtin_trunc((double)e * 1099511627776.0); }
constexpr uint32_t kExactIds = 4095;  // ids per thread and half whose mass sum (of both halves) is exact in fp64

// Sampled row b from its segments' counts.  kRowLeft (on every thread) if the
// counts don't settle it; the largest key if no id has mass, the row's answer
// then being the lowest id that holds it.  qtab: masses of the 2 * kMagBins
// window keys by magnitude (kMagBins + magnitude for negative ones).
enum : uint32_t { kRowDone = 0, kRowLeft = 0x10000 };
XV_INLINE uint32_t row_from_counts(const SegArgs& a, const RowParams& p, RowShared& s, double* qtab, int b) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const bf16_t* row = a.logits + (int64_t)b * a.stride;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  const uint32_t* cnts = a.seg_cnt + (int64_t)b * a.R * kSegWords;
  // f(segment, its counts of this thread's positions: [half][j]): a group's
  // loads all go out before any is used (segments past R reload the last)
  auto each_group = [&](auto&& f) {
    for (int r0 = 0; r0 < a.R; r0 += kCntLoads) {
      uint2 kc[kCntLoads][2];
#pragma unroll
      for (int r = 0; r < kCntLoads; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          kc[r][h] = *reinterpret_cast<const uint2*>(cnts + (int64_t)min(r0 + r, a.R - 1) * kSegWords +
                                                     h * (kHalfPos / 2) + 2 * t);
      f(r0, kc);
    }
  };
  auto count_of = [](const uint2 (&k)[2], int h, int j) {
    return ((j < 2 ? k[h].x : k[h].y) >> (16 * (j & 1))) & 0xffffu;
  };
  const uint32_t* head = cnts + (int64_t)min(lane, a.R - 1) * kSegWords + kMagBins;
  const uint4 h0 = *reinterpret_cast<const uint4*>(head), h1 = *reinterpret_cast<const uint4*>(head + 4);
  if (t < 3) s.cut[t] = RowCut{2 * kMagBins, 0, 0, 0x7fffffff, 0};
  if (t < kMaxSegs) {
    s.segm[t] = 0ull;
    s.lties[t] = 0;
  }
  uint32_t c[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  each_group([&](int r0, const uint2 (&kc)[kCntLoads][2]) {
#pragma unroll
    for (int r = 0; r < kCntLoads; ++r)
      if (r0 + r < a.R)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) c[h][j] += count_of(kc[r], h, j);
  });
  // lane r < R: segment r's header
  const bool seg_lane = lane < a.R;
  const int first = (int)(0xffffu - wave_max_u(seg_lane ? h1.z : 0u));  // 0xffff: no window value
  const uint32_t zeros = seg_lane ? h0.x + h0.y : 0u, ntiny = seg_lane ? h1.y : 0u;
  const bool has_mid = __ballot(zeros | ntiny) != 0, has_far = __ballot(seg_lane && h0.z) != 0;
  const float inv_t = 1.0f / p.temp;
  // f(segment, its listed value on this lane, 0xffff past its list) for the
  // lists at word `at` of the segments, `count` (lane r: segment r's) long
  auto each_listed = [&](uint32_t count, int at, auto&& f) {
    for (unsigned long long m = __ballot(count != 0); m; m &= m - 1) {
      const int r = __builtin_ctzll(m);
      const int n = min((int)__shfl((int)count, r), kTinyList);
      const uint16_t* list = reinterpret_cast<const uint16_t*>(cnts + (int64_t)r * kSegWords + at);
      f(r, lane < n ? (uint32_t)list[lane] : 0xffffu);
    }
  };
  auto each_tiny = [&](auto&& f) { each_listed(ntiny, kMagBins + kHWords, f); };
  const bool has_top = __ballot(seg_lane && h1.w) != 0;
  uint32_t kmax = first < 2 * kMagBins ? order_key(pos_bits(first)) : 0u;
  if (XV_UNLIKELY(has_top)) {
    kmax = order_key(wave_max_u(seg_lane ? h1.w : 0u));
  } else if (XV_UNLIKELY(first >= kMagBins && has_mid)) {  // the largest value lies in mid
    kmax = __ballot(seg_lane && h0.x) ? 0x8000u : __ballot(seg_lane && h0.y) ? 0x7fffu : 0u;
    each_tiny([&](int, uint32_t bits) { kmax = max(kmax, order_key(bits)); });
    kmax = wave_max_u(kmax);
  }
  const uint32_t far_mag = XV_UNLIKELY(has_far) ? 0xffffu - wave_max_u(seg_lane ? h0.w : 0u) : 0u;  // its smallest
  const bool only_far = has_far && !has_top && !has_mid && first >= 2 * kMagBins;
  if (XV_UNLIKELY(only_far)) kmax = order_key(0x8000u | far_mag);
  kmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)kmax);
  const float zmax = bf16_to_f32(key_to_bits(kmax)) * inv_t;
  if (XV_UNLIKELY(kmax != 0u && !__builtin_isfinite(zmax))) return kmax;
  // All of mid has one mass where its two ends lie at the same distance from
  // the maximum: 2^-22 past a maximum of 8 is below its last place.  The lists
  // are not read then and need not be whole (half of a row's ids in (0, 2^-22),
  // 32 rows, top-k 50: 140 us with the row left to the one-workgroup path, 28 now).
  const bool one_mass = log2_ratio(kMagLo - 1u, inv_t, zmax) == log2_ratio(0x8000u | (kMagLo - 1u), inv_t, zmax);
  const bool whole = !__ballot(ntiny > (uint32_t)kTinyList);  // the lists hold every small value
  bool settled = kmax != 0u && !only_far && !__ballot(seg_lane && h1.x > (uint32_t)kTinyList) &&
                 (whole || (one_mass && (has_top || first < kMagBins)));
  int far = 0;
  if (XV_UNLIKELY(has_far)) {
    far = (int)wave_sum_l(seg_lane ? h0.z : 0u);
    const float e = exp_of(0x8000u | far_mag, inv_t, zmax);  // the largest: the others' masses are no larger
    settled = settled && mass_of(e) == 0 && !(p.use_m && e >= p.min_p);
  }
  // mid: counts and masses, lane r its segment's
  int64_t mid_q = 0;
  int mid_c = 0;
  bool mid_in = false;  // mid reaches min_p (all of it, or the row isn't settled)
  if (XV_UNLIKELY(settled && has_mid)) {
    const float ez = exp_of(0u, inv_t, zmax);
    const uint32_t equal = one_mass ? zeros + ntiny : zeros;
    int64_t mid_qr = (int64_t)equal * mass_of(ez);
    bool any_in = equal && ez >= p.min_p, any_out = equal && !(ez >= p.min_p);
    if (!one_mass)
      each_tiny([&](int r, uint32_t bits) {
        const float e = exp_of(bits, inv_t, zmax);  // (padding: 0)
        any_in |= bits != 0xffffu && e >= p.min_p;
        any_out |= bits != 0xffffu && !(e >= p.min_p);
        const int64_t q = wave_sum_l(mass_of(e));
        mid_qr += lane == r ? q : 0;
      });
    if (p.use_m) {
      mid_in = __ballot(any_in) != 0;
      settled = !(mid_in && __ballot(any_out) != 0);
    }
    mid_c = (int)wave_sum_l(zeros + ntiny);
    mid_q = wave_sum_l(mid_qr);
    if (t < a.R) s.midq[t] = mid_qr;
  }
  if (!__builtin_amdgcn_readfirstlane((int)settled)) return kRowLeft;
  // top: the listed values that have mass, their count and mass, and the rank of the last to reach min_p
  int top_c = 0, top_m = 0;
  int64_t top_q = 0;
  uint32_t top_low = 0xffffu;  // the lowest key with mass
  if (XV_UNLIKELY(has_top)) {
    const uint32_t ntop = seg_lane ? h1.x : 0u;
    int64_t top_qr = 0;
    uint32_t kmin = 0xffffu;  // the lowest key that reaches min_p
    each_listed(ntop, kTopsAt, [&](int r, uint32_t bits) {
      const float e = exp_of(bits, inv_t, zmax);  // (padding: 0)
      const int64_t m = mass_of(e);
      if (m) top_low = min(top_low, order_key(bits));
      if (m && e >= p.min_p) kmin = min(kmin, order_key(bits));
      top_c += __popcll(__ballot(m != 0));
      const int64_t q = wave_sum_l(m);
      top_qr += lane == r ? q : 0;
    });
    kmin = wave_min_u(kmin);
    each_listed(ntop, kTopsAt, [&](int, uint32_t bits) {
      top_m += __popcll(__ballot(mass_of(exp_of(bits, inv_t, zmax)) != 0 && order_key(bits) >= kmin));
    });
    top_q = wave_sum_l(top_qr);
    if (t < a.R) s.topq[t] = top_qr;
    top_low = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_min_u(top_low));
  }

  // masses; per half, the rank and mass prefixes over its positions
  int cex[2], cn[2], nm[2];  // exclusive rank prefixes, counts, ranks reaching min_p
  int64_t mex[2], ms[2];
  // top and mid: before half 0's and half 1's first position
  const int pre_c[2] = {t == 0 ? top_c : 0, t == 0 ? mid_c : 0};
  const int64_t pre_q[2] = {t == 0 ? top_q : 0, t == 0 ? mid_q : 0};
  // position pos's entry of the table
  auto tab_of = [](int pos) { return pos < kHalfPos ? kHalfPos - 1 - pos : pos; };
  {
    // one position per step of a rolled loop (the counts rotate through c[0][0])
    int n_h = pre_c[0], nm_h = t == 0 ? top_m : 0;
    int64_t m_h = pre_q[0];
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      const uint32_t ci = c[0][0];
#pragma unroll
      for (int j = 0; j < 7; ++j) c[j >> 2][j & 3] = c[(j + 1) >> 2][(j + 1) & 3];
      c[1][3] = ci;
      const int pos = (i >> 2) * kHalfPos + 4 * t + (i & 3);
      double qd = 0.0;
      if (ci) {
        const float e = exp_of(pos_bits(pos), inv_t, zmax);
        qd = mass_d(e);
        n_h += (int)ci;
        m_h += (int64_t)((uint64_t)ci * (uint64_t)qd);
        if (p.use_m && e >= p.min_p) nm_h = n_h;
      }
      qtab[tab_of(pos)] = qd;
      if (i == 3) {
        cn[0] = n_h, ms[0] = m_h, nm[0] = nm_h;
        n_h = pre_c[1], m_h = pre_q[1], nm_h = mid_in ? pre_c[1] : 0;
      }
    }
    cn[1] = n_h + (t == kThreads - 1 ? far : 0), ms[1] = m_h, nm[1] = nm_h;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int ci = 0;
    int64_t mi = 0;
    if (__ballot(cn[h] != 0)) {
      ci = wave_incl_scan_i(cn[h]);
      mi = wave_incl_scan_l(ms[h]);
    }
    cex[h] = ci - cn[h];
    mex[h] = mi - ms[h];
    if (lane == 63) {
      s.ccnt[16 * h + w] = ci;
      s.cmass[16 * h + w] = mi;
    }
  }
  // this thread's masses again, and whether some lane holds more than
  // kExactIds ids of a half (uniform in the wave)
  double q[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) q[h][j] = qtab[tab_of(h * kHalfPos + 4 * t + j)];
  bool big = false;
#pragma unroll
  for (int h = 0; h < 2; ++h) big |= c[h][0] + c[h][1] + c[h][2] + c[h][3] > kExactIds;
  big = __ballot(big) != 0;
  static_assert(kWaves == 16, "32 chunks, one per lane of half a wave");
  __syncthreads();
  int ctot;
  int64_t mtot;
  {
    const int cc = lane < 32 ? s.ccnt[lane] : 0;
    const int64_t cm = lane < 32 ? s.cmass[lane] : 0;
    const int ci = wave_incl_scan_i(cc);
    const int64_t mi = wave_incl_scan_l(cm);
    ctot = __shfl(ci, 31);
    mtot = __shfl(mi, 31);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      cex[h] += __shfl(ci - cc, 16 * h + w);
      mex[h] += __shfl(mi - cm, 16 * h + w);
    }
  }

  // rank n - 1's key, by the thread that holds it: its position, the ids of
  // the key up to the rank, and the mass through the rank
  auto locate = [&](int n, RowCut& cut) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!(cex[h] < n && n <= cex[h] + cn[h])) continue;
      int left = n - cex[h] - pre_c[h];
      int64_t m = mex[h] + pre_q[h];
      if (left <= 0) {
        cut = RowCut{h * kMagBins, n - cex[h], mex[h], cex[h], h ? kInMid : kInTop};
        continue;
      }
      int pos = 2 * kMagBins, ties = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (left > 0) {
          const bool here = left <= (int)c[h][j];
          if (here) {
            pos = h * kHalfPos + 4 * t + j;
            ties = left;
          }
          m += (int64_t)((uint64_t)(here ? left : (int)c[h][j]) * (uint64_t)q[h][j]);
          left -= (int)c[h][j];
        }
      }
      // a rank in far (left > 0 still): every window key kept, far has no mass
      cut = RowCut{pos, ties, m, n, 0};
    }
  };
  // A cut in a group: its key, by each wave for itself (every wave writes the
  // same list) from the sorted list, in mid the +0s and the -0s between the
  // positive and the negative values.  False if the lists do not hold the group.
  uint32_t in_key = 0u;  // the last resolved cut's key, where that lies in a group
  int nlist = 0;
  auto resolve = [&](RowCut& cut) -> bool {
    const int in = __builtin_amdgcn_readfirstlane(cut.in);
    if (XV_LIKELY(!in)) return true;
    if (in == kInMid && !whole) return false;
    const uint4 hz = *reinterpret_cast<const uint4*>(head);
    nlist = 0;
    each_listed(in == kInMid ? ntiny : seg_lane ? head[kHTop] : 0u, in == kInMid ? kMagBins + kHWords : kTopsAt,
                [&](int r, uint32_t bits) {
                  const bool on = bits != 0xffffu && (in == kInMid || mass_of(exp_of(bits, inv_t, zmax)) != 0);
                  const unsigned long long all = __ballot(on);
                  const int i = nlist + __popcll(all & ((1ull << lane) - 1));
                  if (on && i < kListMax) s.list[i] = order_key(bits) << 16 | (uint32_t)r;
                  nlist += __popcll(all);
                });
    if (nlist > kListMax) return false;
    __builtin_amdgcn_wave_barrier();
    const uint32_t key = wave_sort_desc32(lane < nlist ? s.list[lane] : 0u) >> 16;
    const int npz = in == kInMid ? (int)wave_sum_l(seg_lane ? hz.x : 0u) : 0;
    const int nz = in == kInMid ? npz + (int)wave_sum_l(seg_lane ? hz.y : 0u) : 0;
    const int np = __popcll(__ballot(key > 0x8000u));
    const int64_t qz = mass_of(exp_of(0u, inv_t, zmax));
    const int64_t incl = wave_incl_scan_l(key ? mass_of(exp_of(key_to_bits(key), inv_t, zmax)) : 0);
    const int64_t above = np ? __shfl(incl, np - 1) : 0;  // mass of the listed positive values
    int rank = cut.ties;
    if (rank == 0) {
      const int64_t left = s.left;
      rank = (int)wave_first(lane < np && incl > left, -1) + 1;
      if (rank == 0 && left < above + nz * qz) rank = np + 1 + (int)((left - above) / qz);
      if (rank == 0) rank = nz + 1 + (int)wave_first(lane >= np && incl + nz * qz > left, nlist - 1);
    }
    cut.n += rank;
    if (rank > np && rank <= np + nz) {
      const int i = rank - np;
      in_key = i <= npz ? 0x8000u : 0x7fffu;
      cut.ties = i <= npz ? i : i - npz;
      cut.M += above + i * qz;
    } else {
      const int j = rank <= np ? rank - 1 : rank - 1 - nz;
      in_key = __shfl(key, j);
      cut.ties = __popcll(__ballot(lane <= j && key == in_key));
      cut.M += __shfl(incl, j) + (rank <= np ? 0 : nz * qz);
    }
    in_key = (uint32_t)__builtin_amdgcn_readfirstlane((int)in_key);
    return true;
  };
  int n = ctot;
  if (p.use_k && p.top_k < n) n = p.top_k;
  int64_t base = mtot;
  if (p.use_p && n < ctot) {
    locate(n, s.cut[0]);
    __syncthreads();
    RowCut cut = s.cut[0];
    if (!__builtin_amdgcn_readfirstlane((int)resolve(cut))) return kRowLeft;
    base = cut.M;
  }
  if (p.use_p) {
    // the first rank whose inclusive mass exceeds thr (a negative thr: the first rank)
    const int64_t thr = (int64_t)floor((double)p.top_p * (double)base);
    if (thr < 0) {
      locate(1, s.cut[1]);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (!(mex[h] <= thr && thr < mex[h] + ms[h])) continue;
        int64_t left = thr - mex[h], m = mex[h];
        int k = cex[h];
        if (left < pre_q[h]) {
          s.cut[1] = RowCut{h * kMagBins, 0, m, k, h ? kInMid : kInTop};
          s.left = left;
          continue;
        }
        left -= pre_q[h];
        k += pre_c[h];
        m += pre_q[h];
        int64_t qk = 1;
        int pos = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (pos < 0) {
            const int64_t mj = (int64_t)((uint64_t)c[h][j] * (uint64_t)q[h][j]);
            if (left < mj) {
              pos = h * kHalfPos + 4 * t + j;
              qk = (int64_t)q[h][j];
            } else {
              left -= mj;
              m += mj;
              k += (int)c[h][j];
            }
          }
        }
        // left / qk, below the key's count: the double quotient is off by at most one
        int64_t i = (int64_t)((double)left / (double)qk);
        if (i * qk > left) --i;
        if ((i + 1) * qk <= left) ++i;
        s.cut[1] = RowCut{pos, (int)i + 1, m + (i + 1) * qk, k + (int)i + 1, 0};
      }
    }
  }
  int n_m = 0;
  if (p.use_m) {
#pragma unroll
    for (int h = 0; h < 2; ++h) n_m = max(n_m, nm[h] ? cex[h] + nm[h] : 0);
    n_m = (int)wave_max_u((uint32_t)n_m);
    if (lane == 0) s.nm[w] = n_m;
  }
  __syncthreads();
  RowCut cut = s.cut[1];  // no top-p: none
  if (!__builtin_amdgcn_readfirstlane((int)resolve(cut))) return kRowLeft;
  n = min(n, cut.n);
  if (p.use_m) {
    n_m = (int)wave_max_u(lane < kWaves ? (uint32_t)s.nm[lane] : 0u);
    if (n_m > 0) n = min(n, n_m);
  }
  if (n >= ctot) {
    cut = RowCut{2 * kMagBins, 0, mtot, n, 0};
  } else if (n != cut.n) {
    locate(n, s.cut[2]);
    __syncthreads();
    cut = s.cut[2];
    if (!__builtin_amdgcn_readfirstlane((int)resolve(cut))) return kRowLeft;
  }
  const int pos = __builtin_amdgcn_readfirstlane(cut.pos), cut_ties = __builtin_amdgcn_readfirstlane(cut.ties);
  const int in = __builtin_amdgcn_readfirstlane(cut.in);
  // keys above the cut's are kept whole
  const uint32_t cut_key = in ? in_key : pos < 2 * kMagBins ? order_key(pos_bits(pos)) : 0u;
  const int64_t cut_m = cut.M;
  const uint32_t cut_bits = cut_key ? key_to_bits(cut_key) : 0x10000u;  // no cut key: equals no logit
  const int64_t q_cut = mass_of(exp_of(cut_bits & 0xffffu, inv_t, zmax));

  // each segment's kept mass: its positions before the cut's, then (lane r)
  // mid and its share of the cut key's ids, the lowest ids first
  uint32_t tie_word = 0;
  if (!in && pos < 2 * kMagBins && seg_lane) tie_word = cnts[(int64_t)lane * kSegWords + (pos >> 1)];
  if (XV_UNLIKELY(in && t < nlist)) {  // (nlist <= 64)
    const uint32_t x = s.list[t], key = x >> 16;
    if (key > cut_key) atomicAdd(&s.segm[x & 0xffffu], (unsigned long long)mass_of(exp_of(key_to_bits(key), inv_t, zmax)));
    if (key == cut_key) atomicAdd(&s.lties[x & 0xffffu], 1);
  }
  bool some = false;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    double* qo = qtab + (h ? kHalfPos + 4 * t : kHalfPos - 4 - 4 * t);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      q[h][j] = h * kHalfPos + 4 * t + j < pos ? q[h][j] : 0.0;
      some |= q[h][j] != 0.0;
    }
    double2* q2 = reinterpret_cast<double2*>(qo);
    q2[0] = h ? make_double2(q[h][0], q[h][1]) : make_double2(q[h][3], q[h][2]);
    q2[1] = h ? make_double2(q[h][2], q[h][3]) : make_double2(q[h][1], q[h][0]);
  }
  if (__ballot(some)) {
    each_group([&](int r0, const uint2 (&kc)[kCntLoads][2]) {
      int64_t v[8];
      static_assert(kCntLoads == 8, "wave_sum8");
      if (!big) {
        double d[8];
#pragma unroll
        for (int r = 0; r < kCntLoads; ++r) d[r] = 0.0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (__ballot(q[h][0] + q[h][1] + q[h][2] + q[h][3] != 0.0))
#pragma unroll
            for (int r = 0; r < kCntLoads; ++r)
#pragma unroll
              for (int j = 0; j < 4; ++j) d[r] = __builtin_fma((double)count_of(kc[r], h, j), q[h][j], d[r]);
#pragma unroll
        for (int r = 0; r < kCntLoads; ++r) v[r] = (int64_t)d[r];
      } else {
#pragma unroll
        for (int r = 0; r < kCntLoads; ++r) {
          v[r] = 0;
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[r] += (int64_t)((uint64_t)count_of(kc[r], h, j) * (uint64_t)q[h][j]);
        }
      }
      const int64_t m = wave_sum8(v);
      if ((lane & 7) == 0 && r0 + (lane >> 3) < a.R) atomicAdd(&s.segm[r0 + (lane >> 3)], (unsigned long long)m);
    });
  }
  __syncthreads();
  int tie_cr = (int)((tie_word >> (16 * (pos & 1))) & 0xffffu);
  int64_t sm = seg_lane ? (int64_t)s.segm[lane] : 0;
  if (seg_lane) {
    if (in) tie_cr = s.lties[lane];
    if (XV_UNLIKELY(in == kInMid)) {
      const uint4 hz = *reinterpret_cast<const uint4*>(head);
      tie_cr += (int)(cut_key == 0x8000u ? hz.x : cut_key == 0x7fffu ? hz.y : 0u);
      sm += (int64_t)((cut_key < 0x8000u ? hz.x : 0u) + (cut_key < 0x7fffu ? hz.y : 0u)) * mass_of(exp_of(0u, inv_t, zmax));
    } else if (has_mid && pos >= kMagBins) {
      sm += s.midq[lane];
    }
    if (has_top && in != kInTop) sm += s.topq[lane];
  }
  const int tie_ex = wave_incl_scan_i(tie_cr) - tie_cr;
  const int ties_r = max(0, min(tie_cr, cut_ties - tie_ex));
  if (seg_lane) sm += ties_r * q_cut;

  // the draw: the segment holding floor(u * M), then in id order the first
  // kept id whose inclusive mass exceeds the rest.  Each thread sums a run of
  // C consecutive ids; one wave then goes through the run that holds the point.
  const float u = a.uniforms ? a.uniforms[b] : 0.5f;
  const int64_t rdraw = draw_point(u, cut_m);
  const int64_t incl = wave_incl_scan_l(sm);
  const int r = __builtin_amdgcn_readfirstlane(min((int)wave_first(seg_lane && rdraw < incl, kMaxSegs), a.R - 1));
  const int64_t rr = rdraw - (__shfl(incl, r) - __shfl(sm, r));
  const int ties = __builtin_amdgcn_readlane(ties_r, r);
  const int beg = r * a.seg_len, end = min(a.V, beg + a.seg_len);
  const int C = ((end - beg + kThreads - 1) / kThreads + 7) / 8 * 8;
  const int i0 = min(end, beg + t * C), i1 = min(end, i0 + C);
  // mass of an id before the cut key (0 for others)
  const bool mid_kept = has_mid && pos >= kMagBins;  // (of a cut in mid, the keys above it)
  const bool others = mid_kept || has_top;
  const double q_zero = mid_kept ? mass_d(exp_of(0u, inv_t, zmax)) : 0.0;
  auto id_mass = [&](uint32_t bits) -> double {
    const uint32_t mag = bits & 0x7fffu, m = mag - kMagLo;
    if (m < (uint32_t)kMagBins) return qtab[(bits >> 15) * kMagBins + m];
    if (!others) return 0.0;
    const uint32_t key = order_key(bits);
    const bool small = mag < kMagLo;
    if (!(small ? mid_kept : key >= top_low) || key <= cut_key) return 0.0;  // (far, NaN: none)
    return small && (mag == 0u || one_mass) ? q_zero : mass_d(exp_of(bits, inv_t, zmax));
  };
  double mine_d = 0.0;
  int mties = 0;
  constexpr int kVecs = 4;  // vectors in flight
  static_assert(kMaxSegIds / kThreads < (int)kExactIds, "a run's mass is exact in fp64");
  for (int i = i0; i < i1; i += 8 * kVecs) {
    uint32_t wd[kVecs][4];
#pragma unroll
    for (int v = 0; v < kVecs; ++v)
      if (i + 8 * v < i1) load8_words(row, i1, i + 8 * v, vec_ok, wd[v]);  // ids past i1: NaN
#pragma unroll
    for (int v = 0; v < kVecs; ++v)
      if (i + 8 * v < i1)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t bits = bits_of(wd[v], k);
          mine_d += id_mass(bits);
          mties += bits == cut_bits;
        }
  }
  {
    const int64_t mine = (int64_t)mine_d, mi = wave_incl_scan_l(mine);
    const int ti = wave_incl_scan_i(mties);
    if (lane == 63) {
      s.cmass[w] = mi;
      s.ccnt[w] = ti;
    }
    if (t == 0) s.t0 = -1;
    __syncthreads();
    const int64_t wm = lane < kWaves ? s.cmass[lane] : 0;
    const int wt = lane < kWaves ? s.ccnt[lane] : 0;
    const int64_t me = mi - mine + __shfl(wave_incl_scan_l(wm) - wm, w);
    const int te = ti - mties + __shfl(wave_incl_scan_i(wt) - wt, w);
    const int64_t cum = me + min(ties, te) * q_cut;
    const int64_t upto = me + mine + min(ties, te + mties) * q_cut;
    if (cum <= rr && rr < upto) {
      s.t0 = t;
      s.cum = cum;
      s.tie = te;
    }
  }
  __syncthreads();
  if (t >= 64) return kRowDone;
  const int t0 = s.t0;
  int64_t cum = s.cum;
  int te = s.tie;
  const int j0 = min(end, beg + t0 * C), j1 = min(end, j0 + C);
  for (int i = j0; t0 >= 0 && i < j1; i += 64) {
    const uint32_t bits = i + lane < j1 ? (uint32_t)row[i + lane] : 0xffffu;
    const bool tie = bits == cut_bits;
    const int rank = te + __popcll(__ballot(tie) & ((1ull << lane) - 1));
    const int64_t m = tie ? (rank < ties ? q_cut : 0) : (int64_t)id_mass(bits);
    const int64_t inc = cum + wave_incl_scan_l(m);
    const unsigned long long hit = __ballot(inc > rr);
    if (hit) {
      if (lane == 0) a.out_ids[b] = i + __builtin_ctzll(hit);
      break;
    }
    cum = __shfl(inc, 63);
    te += __popcll(__ballot(tie));
  }
  return kRowDone;
}

__global__ __launch_bounds__(kThreads) void row_count_kernel(SegArgs a) {
  __shared__ Shared s;
  __shared__ FastShared fs;
  __shared__ RowShared rs;
  static_assert(kMaxCand >= 2 * kMagBins, "the candidate list's LDS holds the mass table");
  const int b = blockIdx.x, t = threadIdx.x;
  const RowParams p = row_params(a, b);
  if (p.greedy) {  // the best of the segments' best words (torch.argmax order)
    if (t < 64) {
      const unsigned long long best = wave_max_ull(t < a.R ? a.seg_best[b * a.R + t] : 0ull);
      if (t == 0) a.out_ids[b] = best ? (int64_t)(0xffffffffu - (uint32_t)best) : 0;
    }
    return;
  }
  const uint32_t left =
      (uint32_t)__builtin_amdgcn_readfirstlane((int)row_from_counts(a, p, rs, reinterpret_cast<double*>(fs.cand), b));
  if (left != kRowDone) {
    if (left != kRowLeft) {
      const bf16_t* row = a.logits + (int64_t)b * a.stride;
      const int64_t id = lowest_id_of_key(s, row, a.V, (reinterpret_cast<uintptr_t>(row) & 15u) == 0, left);
      if (t == 0) a.out_ids[b] = id;
      return;
    }
    int rb = b;
    __asm__ volatile("" : "+s"(rb)::"memory");
    sample_row(s, fs, rb, a.logits, a.stride, a.V, a.temps, a.top_ps, a.top_ks, a.min_ps, a.uniforms,
               a.flags & ~XV_SAMPLE_ALL_GREEDY, a.out_ids);
  }
}
}  // namespace

// Workspace: one 128-byte line per row (a 64-bit slot and a 32-bit arrival
// counter) for the multi-workgroup greedy path, then the segments' counts of
// the multi-workgroup sampled path, or kTopRowBytes per row, which the top-k
// path's lists use.
namespace {
// Sets how many rows the top-k path takes: the lists of all of them (R
// kTopList 8-byte entries each) share the region of kSegMaxBatch rows.  At V
// 151936 that is 4101 rows; past it one workgroup takes a row (3450 rows 376
// us with lists, 1150 without; 4101 rows 449 and 1381).
constexpr size_t kTopRowBytes = 77936;
struct SegLayout {
  int R, seg_len;
  size_t best, cnt, total;
};
size_t align256(size_t x) { return (x + 255) / 256 * 256; }
SegLayout seg_layout(int batch, int vocab) {
  SegLayout L;
  int segs = max(1, min(kCntSegs, kCntTarget / max(batch, 1)));
  segs = max(1, min(segs, vocab / 2048));
  segs = max(segs, (vocab + kMaxSegIds - 1) / kMaxSegIds);
  L.seg_len = ((vocab + segs - 1) / segs + 7) / 8 * 8;
  L.R = (vocab + L.seg_len - 1) / L.seg_len;
  const size_t B = (size_t)max(batch, 0), BR = B * L.R;
  size_t o = 0;  // offsets within the sampled path's region
  L.best = o;  o = align256(o + BR * 8);
  L.cnt = o;   o = align256(o + BR * kSegWords * 4);
  L.total = max(o, align256(B * kTopRowBytes));
  return L;
}

// The greedy path's per-row lines, which must be zero before a call.
size_t greedy_bytes(int batch) { return align256((size_t)max(batch, 0) * kGreedyLine * 8); }
// The largest sampled-path region of any batch up to `batch`.
size_t seg_reserve(int batch, int vocab) {
  size_t r = 0;
  for (int b = 1; b <= min(batch, kSegMaxBatch); ++b) r = max(r, seg_layout(b, vocab).total);
  return r;
}
}  // namespace

// Workspace: the greedy lines at the bottom, the sampled path's region at the
// top (it ends at workspace_bytes).  A workspace of this size for B rows
// serves every call of up to B rows, greedy or sampled, in any order: the
// greedy lines [0, Bg * 128) of a call and the region a sampled call of Bs
// rows wrote at the top never overlap, since the size reserves both the lines
// of Bg rows and the largest region of any Bs <= B.
extern "C" size_t xv_sampler_workspace_size(int batch, int vocab) {
  if (batch <= 0 || vocab <= 0) return 256;
  return greedy_bytes(batch) + seg_reserve(batch, vocab);
}

extern "C" int xv_sample(const void* logits, int64_t logits_stride, int batch, int vocab,
                         const float* temperatures, const float* top_ps, const int32_t* top_ks,
                         const float* min_ps, const float* uniforms, int flags,
                         int64_t* out_ids, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (batch < 0 || vocab <= 0 || logits_stride < vocab) return (int)hipErrorInvalidValue;
  if (!(flags & XV_SAMPLE_ALL_GREEDY) && temperatures == nullptr) return (int)hipErrorInvalidValue;
  if (batch == 0) return 0;
  // All-greedy batches: several workgroups per row, about 2048 in all (1024
  // and 4096 measured slower).
  if ((flags & XV_SAMPLE_ALL_GREEDY) && workspace != nullptr &&
      workspace_bytes >= xv_sampler_workspace_size(batch, vocab) && batch <= 65535) {
    // segments of whole 8-id vectors
    const int segs = max(1, min(32, 2048 / batch));
    const int seg_len = ((vocab + segs - 1) / segs + 7) / 8 * 8;
    // one 128-byte line per row: atomics on one line serialise, so rows do not share
    unsigned long long* slots = (unsigned long long*)workspace;
    unsigned int* arrivals = (unsigned int*)(slots + 1);
    greedy_segment_kernel<<<dim3((unsigned)((vocab + seg_len - 1) / seg_len), (unsigned)batch),
                            kGreedyThreads, 0, stream>>>((const bf16_t*)logits, logits_stride, vocab, seg_len, slots,
                                                         arrivals, out_ids);
    XV_CHECK_LAUNCH();
    return 0;
  }
  // Calls whose every top_k is at most kTopList (the caller's max_top_k): the
  // two-launch top-k path, on its own segments (about 1024 workgroups, none
  // longer than the keys a thread holds) and a compact list region of
  // B * R * kTopList candidates at the top of the workspace.  It stays inside
  // the sampled region the size query reserves, so it never reaches the
  // greedy lines; batches whose lists do not fit take the paths below.
  if ((flags & XV_SAMPLE_TOP_K_LE_64) && workspace != nullptr && temperatures != nullptr &&
      workspace_bytes >= xv_sampler_workspace_size(batch, vocab)) {
    const int seg_cap = kTopVecs * 8 * kSegThreads;
    // about 1024 workgroups: one residency round (2048, as the chain, took 1.3 rounds and
    // 28.5 us at B 64 against 24.9 us)
    const int rt = max((vocab + seg_cap - 1) / seg_cap, min(kMaxSegs, max(1, 1024 / batch)));
    const int seg_len = min(seg_cap, ((vocab + rt - 1) / rt + 7) / 8 * 8);
    const int R = (vocab + seg_len - 1) / seg_len;
    const size_t region = align256((size_t)batch * R * kTopList * 8);
    if (R <= kMaxSegs && batch <= 65535 && region <= seg_reserve(batch, vocab)) {
      SegArgs a = {};
      a.logits = (const bf16_t*)logits; a.stride = logits_stride;
      a.V = vocab; a.R = R; a.seg_len = seg_len; a.flags = flags & ~XV_SAMPLE_ALL_GREEDY;
      a.temps = temperatures; a.top_ps = top_ps; a.top_ks = top_ks; a.min_ps = min_ps; a.uniforms = uniforms;
      a.out_ids = out_ids;
      a.cand = (unsigned long long*)((char*)workspace + ((workspace_bytes - region) & ~(size_t)255));
      a.cand_stride = (int64_t)R * kTopList;
      seg_topk_kernel<<<dim3((unsigned)R, (unsigned)batch), kSegThreads, 0, stream>>>(a);
      XV_CHECK_LAUNCH();
      row_topk_kernel<<<dim3((unsigned)batch), kThreads, 0, stream>>>(a);
      XV_CHECK_LAUNCH();
      return 0;
    }
  }
  // Sampled (or mixed) batches of up to kSegMaxBatch rows: several workgroups
  // per row.  Larger batches take one workgroup per row.
  if (workspace != nullptr && batch <= kSegMaxBatch && vocab <= kMaxSegs * kMaxSegIds &&
      workspace_bytes >= xv_sampler_workspace_size(batch, vocab)) {
    const SegLayout L = seg_layout(batch, vocab);
    char* w = (char*)workspace + ((workspace_bytes - L.total) & ~(size_t)255);  // region at the top
    SegArgs a = {};
    a.logits = (const bf16_t*)logits; a.stride = logits_stride;
    a.V = vocab; a.R = L.R; a.seg_len = L.seg_len; a.flags = flags & ~XV_SAMPLE_ALL_GREEDY;
    a.temps = temperatures; a.top_ps = top_ps; a.top_ks = top_ks; a.min_ps = min_ps; a.uniforms = uniforms;
    a.out_ids = out_ids;
    a.seg_best = (unsigned long long*)(w + L.best);
    a.seg_cnt = (uint32_t*)(w + L.cnt);
    seg_count_kernel<<<dim3((unsigned)L.R, (unsigned)batch), kThreads, 0, stream>>>(a);
    XV_CHECK_LAUNCH();
    row_count_kernel<<<dim3((unsigned)batch), kThreads, 0, stream>>>(a);
    XV_CHECK_LAUNCH();
    return 0;
  }
  sample_kernel<<<dim3((unsigned)batch), dim3(kThreads), 0, stream>>>(
      (const bf16_t*)logits, logits_stride, vocab, temperatures, top_ps, top_ks, min_ps, uniforms, flags, out_ids);
  XV_CHECK_LAUNCH();
  return 0;
}
