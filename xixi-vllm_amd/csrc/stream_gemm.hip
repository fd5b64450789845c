// Weight-streaming GEMMs of short batches over the [N, K] weights in place:
// out[M, N] = x[M, K] . w[N, K]^T for M <= 256 rows, bf16 operands, fp32
// accumulate, as fp32 partial sums of a K split (the input of the norm or
// q/k norm + RoPE kernel that consumes them) or as the gate/up projection
// fused with SiLU-and-mul.  Replaces, for decode batches and prompt chunks
// this short, the library GEMMs of the decoder's projections (reference
// src/compute/models/qwen3.py:50-64,108-115).
//
// What bounds it: up to about 64 rows the weights' HBM stream (Qwen3-8B
// gate_up, 201 MB, 64 rows: 34 us = 5.9 TB/s; 8 rows 31 us = 6.5 TB/s, what a
// read-only probe of the same pattern reaches), above that the loads of x
// and W through each CU together with the LDS operand reads (200 rows: 54 us).
// Three things set the rate, each measured with that probe:
// - K rotation.  Weight rows are K * 2 bytes apart, a multiple of the HBM
//   channel interleave, so workgroups that all start at K = 0 stay on the
//   same few channels: 38.7 us.  Workgroup b starts at step 5 b mod steps and
//   wraps: 32.0 us.  (The products are summed in another order per column block.)
// - No drain at the barrier.  __syncthreads waits for every LDS load in
//   flight; the loop uses s_waitcnt vmcnt(n) for the oldest stage alone and a
//   bare s_barrier: 45.4 -> 35.2 us.
// - In-order loads.  A CU's loads return in issue order, so x (from L2) waits
//   behind the W (from HBM) issued before it.  x and W of a stage are issued
//   together, x first, and travel the same ring: with x two stages deep
//   beside a deeper W ring 200 rows took 72 us instead of 54.
//
// Workgroup: WAVES = MW x KW waves over BNT 16-row tiles of w, all M rows and
// one K slice.  Per stage of KS elements it moves XT tiles of x and BNT of w
// by LDS-DMA into one of DEPTH ring slots, rows of KS * 2 bytes with their
// 16-byte pieces permuted by row (swz) so that fragment reads spread over the
// banks.  Wave (mw, kw) multiplies x tiles MTW mw .. by every w tile over its
// share of the stage's 32-element substeps; KW shares are summed through LDS at the end.
// Workgroups of one K slice differ by a multiple of `parts` in index, so an
// XCD (index mod 8) sees one slice of x and keeps it in its own L2 (Qwen3-8B
// down, 200 rows, 8 parts: 38.7 -> 30.4 us against slices spread over XCDs).
#include "xv_common.h"
#include "xv_kernels.h"

namespace {

constexpr int kModeParts = 1, kModeSiluMul = 2;
constexpr int kNt = 2;       // cache policy bits: non-temporal (each weight is read once)
constexpr int kRotate = 5;   // stages between the starting points of neighbouring column blocks

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

struct StreamArgs {
  const bf16_t* x;
  int64_t xs;
  const bf16_t* w;
  int64_t ws;
  void* out;
  int64_t os, part_stride;
  int m, kslice, inter, parts;
};

// N w fragments and NX x fragments (16 bytes per lane; tile j at j * TS from
// its address), read and waited for in one block.
#define XV_RD(i, a, j) "ds_read_b128 %" #i ", %[" #a "] offset:%[ts]*" #j "\n\t"
#define XV_RW1 XV_RD(0, wa, 0)
#define XV_RW2 XV_RW1 XV_RD(1, wa, 1)
#define XV_RW4 XV_RW2 XV_RD(2, wa, 2) XV_RD(3, wa, 3)
#define XV_RW5 XV_RW4 XV_RD(4, wa, 4)
#define XV_RW6 XV_RW5 XV_RD(5, wa, 5)
#define XV_RW8 XV_RW6 XV_RD(6, wa, 6) XV_RD(7, wa, 7)
#define XV_RW10 XV_RW8 XV_RD(8, wa, 8) XV_RD(9, wa, 9)
#define XV_OW1 "=&v"(w[0])
#define XV_OW2 XV_OW1, "=&v"(w[1])
#define XV_OW4 XV_OW2, "=&v"(w[2]), "=&v"(w[3])
#define XV_OW5 XV_OW4, "=&v"(w[4])
#define XV_OW6 XV_OW5, "=&v"(w[5])
#define XV_OW8 XV_OW6, "=&v"(w[6]), "=&v"(w[7])
#define XV_OW10 XV_OW8, "=&v"(w[8]), "=&v"(w[9])
#define XV_READ1(NW)                                                                                     \
  if constexpr (N == NW && NX == 1)                                                                      \
    __asm__ __volatile__(XV_RW##NW XV_RD(NW, xa, 0) "s_waitcnt lgkmcnt(0)"                               \
                         : XV_OW##NW, "=&v"(x[0])                                                        \
                         : [wa] "v"(wa), [xa] "v"(xa), [ts] "n"(TS)                                      \
                         : "memory")
#define XV_READ2(NW, NW1)                                                                                \
  if constexpr (N == NW && NX == 2)                                                                      \
    __asm__ __volatile__(XV_RW##NW XV_RD(NW, xa, 0) XV_RD(NW1, xa, 1) "s_waitcnt lgkmcnt(0)"             \
                         : XV_OW##NW, "=&v"(x[0]), "=&v"(x[1])                                           \
                         : [wa] "v"(wa), [xa] "v"(xa), [ts] "n"(TS)                                      \
                         : "memory")
template <int N, int NX, int TS>
XV_INLINE void read_frags(bf16x8_t (&w)[N], bf16x8_t (&x)[NX], uint32_t wa, uint32_t xa) {
  static_assert((N == 1 || N == 2 || N == 4 || N == 5 || N == 6 || N == 8 || N == 10) && (NX == 1 || NX == 2),
                "a tile count without a read block");
  XV_READ1(1);
  XV_READ1(2);
  XV_READ1(4);
  XV_READ1(5);
  XV_READ1(6);
  XV_READ1(8);
  XV_READ1(10);
  XV_READ2(1, 2);
  XV_READ2(2, 3);
  XV_READ2(4, 5);
  XV_READ2(5, 6);
  XV_READ2(6, 7);
  XV_READ2(8, 9);
  XV_READ2(10, 11);
}

// Waits until this wave's loads of its oldest stage in flight have landed;
// `rem` stages follow that one (at most D - 2 of them in flight, PER loads each).
template <int PER, int D>
XV_INLINE void wait_stage(int rem) {
  if constexpr (D <= 2) {
    __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (rem >= D - 2) __asm__ __volatile__("s_waitcnt vmcnt(%0)" ::"n"(PER * (D - 2)) : "memory");
    else wait_stage<PER, D - 1>(rem);
  }
}

XV_INLINE float round_bf16(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// 16-byte piece c of row r of a stage sits in slot c ^ swz(r): the 16 rows of
// a fragment read (one piece each) fall into 16 different slots of a
// 256-byte bank line (rows of 128 bytes: two rows per line).
template <int CH>
XV_INLINE int swz(int r) {
  return CH == 16 ? (r & 15) : ((r >> 1) & 7);
}

template <int MW, int MTW, int KW, int BNT, int KS, int XT, int DEPTH, int MODE>
__global__ __launch_bounds__(MW * KW * 64) void stream_gemm_kernel(StreamArgs a) {
  constexpr int WAVES = MW * KW;
  constexpr int CH = KS / 8;                // 16-byte pieces per row
  constexpr int ROWB = KS * 2;
  constexpr int RPU = 1024 / ROWB;          // rows per load instruction (a unit of 1 KB)
  constexpr int TS = 16 * ROWB;             // bytes of a 16-row tile
  constexpr int STAGE = (XT + BNT) * TS;    // x tiles, then w tiles
  constexpr int XU = XT * TS / 1024, UNITS = STAGE / 1024;
  constexpr int PER = (UNITS + WAVES - 1) / WAVES, EXTRA = UNITS % WAVES;  // waves below EXTRA load PER units, others one less
  constexpr int SUB = KS / 32 / KW;         // 32-element substeps of a stage per wave
  constexpr int RED = (KW - 1) * MW * BNT * MTW * 1024;
  constexpr int LDSB = DEPTH * STAGE > RED ? DEPTH * STAGE : RED;
  static_assert((CH == 8 || CH == 16) && MW * MTW >= XT && SUB >= 1 && DEPTH >= 2 && PER * (DEPTH - 2) < 64, "shape");
  static_assert(LDSB <= 160 * 1024, "LDS of a CU");
  static_assert(MODE != kModeSiluMul || BNT % 2 == 0, "gate/up tiles come in pairs");
  __shared__ __attribute__((aligned(1024))) char ring[LDSB];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, grp = lane >> 4;
  const int mw = wave % MW, kw = wave / MW;
  const bool more = EXTRA == 0 || wave < EXTRA;

  const int part = (int)blockIdx.x % a.parts, cb = (int)blockIdx.x / a.parts;
  const int64_t kbase = (int64_t)part * a.kslice;
  const int steps = a.kslice / KS;
  const char* src[PER];  // this lane's 16 bytes of unit i * WAVES + wave at the slice's first stage
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int u = min(i * WAVES + wave, UNITS - 1);
    const int row = u * RPU + lane / CH;
    const int64_t k0 = kbase + ((lane % CH) ^ swz<CH>(row)) * 8;
    if (row < XT * 16) {  // rows past M read row M - 1 (their products are never stored)
      src[i] = reinterpret_cast<const char*>(a.x + (int64_t)min(row, a.m - 1) * a.xs + k0);
    } else {
      const int wr = row - XT * 16;
      int64_t n;
      if constexpr (MODE == kModeSiluMul) {  // 8 BNT gate rows, then the matching up rows
        constexpr int H = BNT * 8;
        n = (int64_t)cb * H + (wr < H ? wr : a.inter + wr - H);
      } else {
        n = (int64_t)cb * (BNT * 16) + wr;
      }
      src[i] = reinterpret_cast<const char*>(a.w + n * a.ws + k0);
    }
  }
  const int rot = (int)(((unsigned)cb * kRotate) % (unsigned)steps);
  auto issue = [&](int s, int slot) {
    int t = s + rot;
    t = t >= steps ? t - steps : t;
    const int64_t off = (int64_t)t * ROWB;
    char* const st = ring + slot * STAGE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i == PER - 1 && EXTRA && !more) break;
      const int u = i * WAVES + wave;
      if (u < XU) __builtin_amdgcn_global_load_lds((glb_void*)(src[i] + off), (lds_void*)(st + u * 1024), 16, 0, 0);
      else __builtin_amdgcn_global_load_lds((glb_void*)(src[i] + off), (lds_void*)(st + u * 1024), 16, 0, kNt);
    }
  };
  floatx4_t acc[BNT][MTW];
#pragma unroll
  for (int i = 0; i < BNT; ++i)
#pragma unroll
    for (int q = 0; q < MTW; ++q) acc[i][q] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  const bool active = mw * MTW * 16 < a.m;
  // fragment of substep j: row r16 of a tile, piece 4 (kw SUB + j) + grp
  uint32_t fo[SUB];
#pragma unroll
  for (int j = 0; j < SUB; ++j)
    fo[j] = (uint32_t)reinterpret_cast<uintptr_t>(ring) + r16 * ROWB +
            (((4 * (kw * SUB + j) + grp) ^ swz<CH>(r16)) << 4);

  for (int s = 0; s < min(DEPTH - 1, steps); ++s) issue(s, s);
  int slot = 0, fill = DEPTH - 1;
  for (int s = 0; s < steps; ++s) {
    const int rem = steps - 1 - s;
    if (more) wait_stage<PER, DEPTH>(rem);
    else wait_stage<(PER > 1 ? PER - 1 : 1), DEPTH>(rem);
    // every wave's loads of stage s have landed, and every wave is done with stage s - 1, whose slot is filled next
    __asm__ __volatile__("s_barrier" ::: "memory");
    if (s + DEPTH - 1 < steps) issue(s + DEPTH - 1, fill);
    fill = fill == DEPTH - 1 ? 0 : fill + 1;
    if (active) {
      const uint32_t ox = slot * STAGE + mw * MTW * TS, ow = slot * STAGE + XT * TS;
#pragma unroll
      for (int j = 0; j < SUB; ++j) {
        bf16x8_t w[BNT], x[MTW];
        read_frags<BNT, MTW, TS>(w, x, fo[j] + ow, fo[j] + ox);
#pragma unroll
        for (int i = 0; i < BNT; ++i)
#pragma unroll
          for (int q = 0; q < MTW; ++q) acc[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[q], acc[i][q], 0, 0, 0);
      }
    }
    slot = slot == DEPTH - 1 ? 0 : slot + 1;
  }
  if constexpr (KW > 1) {  // sum the waves' K shares (every load has landed: the last stage waited for all)
    __syncthreads();
    floatx4_t* red = reinterpret_cast<floatx4_t*>(ring);
    if (kw > 0) {
#pragma unroll
      for (int i = 0; i < BNT; ++i)
#pragma unroll
        for (int q = 0; q < MTW; ++q) red[((((kw - 1) * MW + mw) * BNT + i) * MTW + q) * 64 + lane] = acc[i][q];
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int p = 0; p < KW - 1; ++p)
#pragma unroll
      for (int i = 0; i < BNT; ++i)
#pragma unroll
        for (int q = 0; q < MTW; ++q) acc[i][q] += red[(((p * MW + mw) * BNT + i) * MTW + q) * 64 + lane];
  }
  // acc[i][q] lane l: rows 4 (l / 16) .. +3 of w tile i (output columns), row l % 16 of x tile q
#pragma unroll
  for (int q = 0; q < MTW; ++q) {
    const int m = (mw * MTW + q) * 16 + r16;
    if (m >= a.m) continue;
    if constexpr (MODE == kModeSiluMul) {
      constexpr int H = BNT / 2;
#pragma unroll
      for (int i = 0; i < H; ++i) {
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // g and u rounded to bf16 first, as the unfused GEMM stores them
          const float gv = round_bf16(acc[i][q][e]), uv = round_bf16(acc[i + H][q][e]);
          r[e] = gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)) * uv;
        }
        const int64_t col = (int64_t)cb * (H * 16) + i * 16 + grp * 4;
        *reinterpret_cast<uint2*>(static_cast<bf16_t*>(a.out) + m * a.os + col) =
            make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]));
      }
    } else {
#pragma unroll
      for (int i = 0; i < BNT; ++i) {
        const int64_t col = (int64_t)cb * (BNT * 16) + i * 16 + grp * 4;
        *reinterpret_cast<floatx4_t*>(static_cast<float*>(a.out) + part * a.part_stride + m * a.os + col) = acc[i][q];
      }
    }
  }
}

// The most tiles per workgroup that a row class has a kernel for: with more its
// ring is too shallow, or (10) its accumulators too many.
constexpr int max_tiles(int m) { return m <= 16 ? 6 : m <= 64 ? 8 : 10; }

// The tile count and K split of one product (bnt 0: not taken).
struct StreamPlan {
  int bnt, parts;
};

// Tiles and K split of an m x n x k product (host).  256 CUs stream evenly
// when each has one workgroup, so column blocks x parts is kept within
// 224 .. 256 (gate/up, which is not split, 192 .. 256: Qwen3-8B qkv, 8 rows,
// 256 workgroups 11.3 us, 192 13.4).  A workgroup reads m x (k / parts) of x and writes m x 16 bnt
// partial sums that the consumer reads back; with 256 workgroups bnt grows
// with the split, and the two costs balance at parts^2 ~ k / (n / 16)
// (products alone, Qwen3-8B, 64 rows: down 8 parts 20.1 us, 4 parts 21.4; o 4 parts 9.6, 8 parts
// 10.1, 2 parts 10.6; 8 rows want half as many: o 2 parts 8.0, 4 parts 8.8.
// In a layer with the consumer that reads the parts, 80 to 256 rows: Qwen3-8B
// o 2 parts +1.4 .. 4.1 us, 8 parts +1.6 .. 3.9, down 4 parts +1.5 .. 4.9,
// Qwen3-32B o 8 parts +0.4 .. 3.5, down 4 parts +1.4 .. 7.5; Qwen3-0.6B's 1024
// columns take 8 parts where 4 are 0.3 to 2.0 better).
// Gate/up (no split) takes the block count nearest 256, at up to 16 rows
// blocks of two tiles whatever their number (8 rows, Qwen3-8B: 768 blocks 31.0
// us, 256 blocks 33.1).  Shapes outside these bounds are not taken: with n /
// 16 = 3200 tiles (Qwen3-32B gate/up) above 16 rows no block count fills the
// CUs evenly (400 blocks: 99 us at 32 rows, the library's 98).
StreamPlan stream_plan(int m, int n, int k, int mode) {
  const StreamPlan no{0, 0};
  if (m < 1 || m > 256 || n < 16 || k < 64 || n % 16 || (mode != kModeParts && mode != kModeSiluMul)) return no;
  const int ks = m <= 64 ? 128 : 64;
  const int tiles = n / 16;
  if (mode == kModeSiluMul) {
    if (k % ks || n % 32) return no;
    if (m <= 16) return tiles % 2 == 0 && tiles >= 256 ? StreamPlan{2, 1} : no;
    for (int bnt : {2, 4, 6, 8})  // the most workgroups up to 256
      if (tiles % bnt == 0 && tiles / bnt <= 256) return tiles / bnt >= 192 ? StreamPlan{bnt, 1} : no;
    return no;
  }
  StreamPlan best = no;
  double cost = 1e30;
  for (int parts : {1, 2, 4, 8}) {
    if (k % (parts * ks)) continue;
    const double r = (double)parts * parts * tiles / k * (m <= 16 ? 4.0 : 1.0);  // 1 at the balance
    const double c = r < 1.0 ? 1.0 / r : r;
    if (c > cost) continue;  // ties: the larger split
    for (int bnt : {1, 2, 4, 5, 6, 8, 10}) {  // the most workgroups up to 256
      if (tiles % bnt || (int64_t)tiles / bnt * parts > 256) continue;
      if ((int64_t)tiles / bnt * parts < 224 || bnt > max_tiles(m)) break;
      best = StreamPlan{bnt, parts};
      cost = c;
      break;
    }
  }
  return best;
}

// False: no such kernel.
template <int MW, int MTW, int KW, int BNT, int KS, int XT, int DEPTH>
bool launch(const StreamArgs& a, int mode, unsigned blocks, hipStream_t stream) {
  if (mode == kModeParts) {
    stream_gemm_kernel<MW, MTW, KW, BNT, KS, XT, DEPTH, kModeParts><<<blocks, MW * KW * 64, 0, stream>>>(a);
    return true;
  }
  if constexpr (BNT % 2 == 0) {
    stream_gemm_kernel<MW, MTW, KW, BNT, KS, XT, DEPTH, kModeSiluMul><<<blocks, MW * KW * 64, 0, stream>>>(a);
    return true;
  }
  return false;
}

// Waves, stage and ring depth per row class: the waves split the stage's K
// until there are two per SIMD (four at 128 and more rows, where LDS reads and
// MFMAs need the overlap: 200 rows 54 us, with half the waves 63), and the
// ring takes what fits of 160 KB.
template <int BNT>
bool launch_rows(const StreamArgs& a, int mode, unsigned blocks, hipStream_t stream) {
  if (a.m <= 16) {
    if constexpr (BNT <= max_tiles(16)) return launch<1, 1, 4, BNT, 128, 1, BNT == 1 ? 8 : BNT == 6 || BNT == 5 ? 5 : 6>(a, mode, blocks, stream);
  } else if (a.m <= 32) {
    if constexpr (BNT <= max_tiles(32)) return launch<2, 1, 4, BNT, 128, 2, BNT == 1 ? 10 : BNT == 2 ? 8 : BNT == 4 ? 6 : BNT == 5 ? 5 : 4>(a, mode, blocks, stream);
  } else if (a.m <= 64) {
    if constexpr (BNT <= max_tiles(64)) return launch<4, 1, 2, BNT, 128, 4, BNT <= 2 ? 6 : BNT == 4 ? 5 : BNT == 5 ? 4 : 3>(a, mode, blocks, stream);
  } else if (a.m <= 128) {
    return launch<8, 1, 2, BNT, 64, 8, BNT <= 2 ? 7 : BNT <= 5 ? 6 : BNT == 6 ? 5 : 4>(a, mode, blocks, stream);
  } else if constexpr (BNT == 10) {
    return launch<8, 2, 1, BNT, 64, 16, 3>(a, mode, blocks, stream);  // 20 accumulators: two waves per SIMD
  } else {
    return launch<8, 2, 2, BNT, 64, 16, BNT <= 4 ? 4 : 3>(a, mode, blocks, stream);
  }
  return false;
}

}  // namespace

extern "C" int xv_stream_gemm_parts(int m, int n, int k, int mode) { return stream_plan(m, n, k, mode).parts; }

extern "C" int xv_stream_gemm(const void* x, int64_t x_stride, const void* w, int64_t w_stride, void* out,
                              int64_t out_stride, int64_t part_stride, int m, int n, int k, int mode, int parts,
                              hipStream_t stream) {
  const StreamPlan p = stream_plan(m, n, k, mode);
  if (p.bnt == 0 || parts != p.parts) return (int)hipErrorInvalidValue;
  if (!xv_al16(x) || !xv_al16(w) || !xv_st8(x_stride) || !xv_st8(w_stride) || x_stride < k || w_stride < k)
    return (int)hipErrorInvalidValue;
  if (mode == kModeParts) {
    if (!xv_al16(out) || (out_stride & 3) || out_stride < n || (part_stride & 3) || part_stride < (int64_t)m * out_stride)
      return (int)hipErrorInvalidValue;
  } else if (((uintptr_t)out & 7u) || (out_stride & 3) || out_stride < n / 2) {
    return (int)hipErrorInvalidValue;
  }
  const StreamArgs a{(const bf16_t*)x, x_stride, (const bf16_t*)w, w_stride, out, out_stride, part_stride,
                     m, k / parts, mode == kModeSiluMul ? n / 2 : 0, parts};
  const unsigned blocks = (unsigned)(n / (16 * p.bnt) * parts);
  bool done = false;
  switch (p.bnt) {
    case 1: done = launch_rows<1>(a, mode, blocks, stream); break;
    case 2: done = launch_rows<2>(a, mode, blocks, stream); break;
    case 4: done = launch_rows<4>(a, mode, blocks, stream); break;
    case 5: done = launch_rows<5>(a, mode, blocks, stream); break;
    case 6: done = launch_rows<6>(a, mode, blocks, stream); break;
    case 8: done = launch_rows<8>(a, mode, blocks, stream); break;
    default: done = launch_rows<10>(a, mode, blocks, stream); break;
  }
  if (!done) return (int)hipErrorInvalidValue;
  XV_CHECK_LAUNCH();
  return 0;
}
