// fp32 GEMM on the 16-bit matrix cores, at fp32 accuracy:
//   Y[m, n] = sum_k X(m, k) W(n, k),  fp32 in, fp32 accumulation, fp32 out,
// for the fp32 B/C projections and their gradients (F.linear and its backward,
// mambaqc/layers/quaternion_linear.py:145-161). Each operand is a strided view with either
// k or the row index contiguous, so one entry point serves the forward (x, W), the input
// gradient (gy, W transposed) and the weight gradient (gy transposed, x transposed).
//
// Why. The fp32 matrix rate of gfx950 is 157 TFLOP/s, and hipBLASLt reaches 115-153 of them on
// these shapes; the fp16 rate is 16 times that. An fp32 value times a power of two of its row is
// split into two fp16 pieces, a = hi + lo (11 significant bits each: a is held to 2^-23 of itself,
// or to 2^-40 of its row's largest magnitude where that is more, fp16's subnormal spacing), and a
// product takes three MFMAs, hi hi + hi lo + lo hi, into one fp32 accumulator. What is dropped (lo
// lo, and what lo rounds away) is about 2^-23 of a product, random in sign, and an MFMA adds 32
// products per rounding of the accumulator where the fp32 one adds 4: the error against 64 bits is
// not larger than hipBLASLt's fp32 (tests/test_gpu_gemm_f32.py measures both).
//
//   - Row scale: 2^(14 - exponent of the row's largest |a|), so hi never overflows; taken
//     back in the epilogue with ldexp. amax holds each row's largest |a| (as fp32 bits, the
//     maximum taken on the bits, so that an inf or a NaN is the largest).
//   - Wide ranges. `small` counts a row's elements under 2^-16 of its largest, which are held to
//     less than 2^-24 of themselves, but to 2^-40 of the largest. J of them in a row of X and one
//     of W put an output off by at most 2^-40 J of the product of the rows' largest, which may be
//     all that an output is where the other operand's zeros leave nothing larger. An output (by the
//     magnitudes of its shares of k) is listed where 2^-28 K of it is less than that (2^-20 where K
//     is below 256), and computed again from the fp32 operands; every other one is so within 2^-28
//     K of those, a sixteenth of fp32's own bound for a sum of K. A row with more than one small
//     element in eight, or with an inf, is listed whole. gemm_f32_again_kernel computes both, rows
//     on the fp32 matrix cores. Of ordinary operands (normal or uniform values) about one output in
//     10^8 is listed. (A row with a NaN makes NaNs by itself.)
//   - Layout of the pieces: per row and 32 columns of k, 32 hi pieces and then 32 lo pieces
//     (128 bytes: one K step of mfma_tile.hpp's loop), columns past K zero.
//   - Blocks: an operand is split a block at a time (kBlockElems, 64 MiB of pieces), and each
//     block is multiplied while its pieces are still in the 256 MiB Infinity Cache. Long k
//     (the input gradient's) is blocked too, each block adding to the partial sums; its
//     blocks are twice as large, since each adds a pass over the partial sums and one of half the
//     rows splits the other operand again. Measured, blocks of 16 and 32 Mi elements (us): forward
//     M 2048 N 65536 K 512 518 / 600, M 4096 N 98304 K 768 1874 / 2026; input gradients
//     M 2048 N 512 K 65536 777 / 711, M 4096 N 768 K 98304 2960 / 2738, M 1024 N 1024 K 131072
//     2239 / 1436, M 600 N 384 K 98304 1327 / 598. So is a k that takes the shorter side past one
//     block (the weight gradient of many tokens), for the same reason.
//   - Few output tiles in a block (the input gradient): k is shared by `splits` workgroups per
//     tile, whose partial sums a last launch adds in order, block by block. They are at most 512
//     tiles of 128 x 128 (32 MiB) at a time, whatever the output's size.
#include <atomic>

#include "mfma_tile.hpp"

namespace mqc {
namespace {

using namespace mfma;

constexpr int kChunk = 32;                      // columns of k per 128-byte line of pieces
constexpr int64_t kBlockElems = 16 << 20;       // elements of one operand split at a time
constexpr int kCUsF = 256;

__device__ inline uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// Exponent added to a row's values before splitting: its largest magnitude lands in
// [2^14, 2^15). Zero for a row of zeros and for a row that is not finite.
__device__ inline int split_exp(float amax) {
  const uint32_t u = __float_as_uint(amax);
  if (u == 0u || u >= 0x7f800000u) return 0;
  return 15 - __builtin_amdgcn_frexp_expf(amax);
}
// An element (a zero excepted) under 2^-16 of its row's largest, by a line for the bits of |a| less
// one.
__device__ inline uint32_t small_line(float amax) {
  const uint32_t line = __float_as_uint(__builtin_amdgcn_ldexpf(0.5f, -split_exp(amax)));
  return line > 0u ? line - 1u : 0u;  // (none where even 2^-149 is held exactly)
}
// The least that a product's share of k, before its row scales, may come out as where a row has j
// small elements (nothing comes of a row of zeros).
__device__ inline float line_of(float amax, uint32_t j, float least) {
  return amax == 0.f ? -0x1p60f : least * (float)j;
}
__device__ inline bool is_small(float v, uint32_t line) { return abs_bits(v) - 1u < line; }

// What is to be computed again: rows of X and of W (counts, lists and a mark for each row listed)
// and outputs.
struct Again {
  uint32_t* rows[2];
  uint32_t* mark[2];
  uint32_t* outs;    // kMaxOuts pairs (m, n)
  uint32_t* counts;  // rows of X, rows of W, outputs
};
constexpr uint32_t kMaxOuts = 16384;
__device__ inline void list_row(const Again& g, int side, int64_t row) {
  if (atomicExch(g.mark[side] + row, 1u) == 0u)
    g.rows[side][atomicAdd(g.counts + side, 1u)] = (uint32_t)row;
}
// (Past the list's end, the row of X. Listed rows need no outputs of their own.)
__device__ inline void list_out(const Again& g, int64_t m, int64_t n) {
  if (g.mark[0][m] != 0u || g.mark[1][n] != 0u) return;
  uint32_t at = *(volatile uint32_t*)(g.counts + 2);
  if (at < kMaxOuts) at = atomicAdd(g.counts + 2, 1u);
  if (at < kMaxOuts) {
    g.outs[2 * at] = (uint32_t)m;
    g.outs[2 * at + 1] = (uint32_t)n;
  } else {
    list_row(g, 0, m);
  }
}

// v * 2^e as hi + lo, packed for two values (hi in .x, lo in .y).
__device__ inline uint2 split2(float a, float b, int e) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  a = __builtin_amdgcn_ldexpf(a, e);
  b = __builtin_amdgcn_ldexpf(b, e);
  const h2 hi = {(_Float16)a, (_Float16)b};
  const h2 lo = {(_Float16)(a - (float)hi[0]), (_Float16)(b - (float)hi[1])};
  return uint2{__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo)};
}

// Rows with k contiguous: WPR waves per row (one, or four for rows longer than a wave holds). V = 4
// where every row is 16-byte aligned. HELD: the row fits in registers (K <= 64 * WPR * V * HELD)
// and is read once; 0: it is read twice. Bound by HBM: 64 MiB of fp32 to 64 MiB of pieces in 27 us
// (5.0 TB/s, the copy rate); with one wave per row throughout, rows of 16384 took 60 us.
template <int V, int HELD, int WPR>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ A, int64_t ld,
                                                         int64_t rows, int K, int Kp,
                                                         uint16_t* __restrict__ P,
                                                         float* __restrict__ amax,
                                                         uint32_t* __restrict__ small, Again again,
                                                         int side, int64_t row0) {
  constexpr int TPR = 64 * WPR;
  constexpr int RPB = 4 / WPR;
  __shared__ uint32_t red[8];
  const int tl = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / TPR;
  if (row >= rows) return;  // (with WPR 4 a block has one row, so no wave leaves a barrier)
  const float* a = A + row * ld;
  char* p = (char*)P + row * (int64_t)Kp * 4;
  float v[HELD ? HELD : 1][V];
  uint32_t m = 0;
  auto load = [&](int k, float (&o)[V]) {
    if constexpr (V == 4) {
      const float4 f = k < K ? *(const float4*)(a + k) : float4{0.f, 0.f, 0.f, 0.f};
      o[0] = f.x; o[1] = f.y; o[2] = f.z; o[3] = f.w;
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = k + i < K ? a[k + i] : 0.f;
    }
  };
  auto top = [&](const float (&o)[V]) {
#pragma unroll
    for (int i = 0; i < V; ++i) m = m > abs_bits(o[i]) ? m : abs_bits(o[i]);
  };
  auto store = [&](int k, const float (&o)[V], int e) {
    if (k >= Kp) return;
    char* q = p + (k / kChunk) * 128 + (k % kChunk) * 2;
    const uint2 s0 = split2(o[0], o[1], e);
    if constexpr (V == 4) {
      const uint2 s1 = split2(o[2], o[3], e);
      *(uint2*)q = uint2{s0.x, s1.x};
      *(uint2*)(q + 64) = uint2{s0.y, s1.y};
    } else {
      *(uint32_t*)q = s0.x;
      *(uint32_t*)(q + 64) = s0.y;
    }
  };
  if constexpr (HELD > 0) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) load((i * TPR + tl) * V, v[i]);
#pragma unroll
    for (int i = 0; i < HELD; ++i) top(v[i]);
  } else {
    for (int k = tl * V; k < K; k += TPR * V) {
      load(k, v[0]);
      top(v[0]);
    }
  }
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)m, s);
    m = m > o ? m : o;
  }
  if constexpr (WPR > 1) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WPR; ++w) m = m > red[w] ? m : red[w];
  }
  const float am = __uint_as_float(m);
  const uint32_t line = small_line(am);
  const int e = split_exp(am);
  // (Lane 0 of a wave, which is active while any lane is, counts all of them.)
  uint32_t seen = 0;
  auto look = [&](const float (&o)[V]) {
#pragma unroll
    for (int i = 0; i < V; ++i) seen += __popcll(__ballot(is_small(o[i], line)));
  };
  if constexpr (HELD > 0) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) store((i * TPR + tl) * V, v[i], e);
#pragma unroll
    for (int i = 0; i < HELD; ++i) look(v[i]);
  } else {
    for (int k = tl * V; k < Kp; k += TPR * V) {
      load(k, v[0]);
      store(k, v[0], e);
      look(v[0]);
    }
  }
  if constexpr (WPR > 1) {
    if ((threadIdx.x & 63) == 0) red[4 + (threadIdx.x >> 6)] = seen;
    __syncthreads();
    seen = red[4] + red[5] + red[6] + red[7];
  }
  if (tl == 0) {
    amax[row] = am;
    small[row] = seen;
    if (m == 0x7f800000u || (m < 0x7f800000u && seen > (uint32_t)K / 8u))
      list_row(again, side, row0 + row);
  }
}

// Rows contiguous (the matrix [K, rows] with row stride ld): the largest magnitude of every
// column, over strips of kStrip rows of k, then the pieces through an LDS transpose.
constexpr int kStrip = 64;
__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

__global__ __launch_bounds__(256) void col_max_kernel(const float* __restrict__ A, int64_t ld,
                                                      int64_t rows, int K, uint32_t* __restrict__ amax) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= rows) return;
  const int k0 = (int)blockIdx.y * kStrip;
  const int k1 = k0 + kStrip < K ? k0 + kStrip : K;
  uint32_t m = 0;
#pragma unroll 16
  for (int k = k0; k < k1; ++k) {
    const uint32_t b = abs_bits(A[(int64_t)k * ld + c]);
    m = m > b ? m : b;
  }
  atomicMax(amax + c, m);
}

// 64 k x 64 rows per workgroup: read with consecutive lanes on consecutive rows, written as
// 256 contiguous bytes (two lines of pieces) per row.
constexpr int kTrT = 64;
__global__ __launch_bounds__(256) void split_cols_kernel(const float* __restrict__ A, int64_t ld,
                                                         int64_t rows, int K, int Kp,
                                                         uint16_t* __restrict__ P,
                                                         const float* __restrict__ amax,
                                                         uint32_t* __restrict__ small, Again again,
                                                         int side, int64_t row0) {
  __shared__ float t[kTrT][kTrT + 1];
  const int64_t c0 = (int64_t)blockIdx.x * kTrT;
  const int k0 = (int)blockIdx.y * kTrT;
  const int cl = threadIdx.x & 63;
  const int kl = threadIdx.x >> 6;
  const int64_t c = c0 + cl < rows ? c0 + cl : rows - 1;
#pragma unroll
  for (int i = 0; i < kTrT / 4; ++i) {
    const int k = k0 + i * 4 + kl;
    t[i * 4 + kl][cl] = k < K ? A[(int64_t)k * ld + c] : 0.f;
  }
  __syncthreads();
  // Four lanes per row and line of pieces, 8 k each.
  const int depth = K - k0 < kTrT ? K - k0 : kTrT;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int item = i * 256 + (int)threadIdx.x;
    const int part = item & 3, line = (item >> 2) & 1, r = item >> 3;
    const int kk = line * kChunk + part * 8;
    const float am = amax[c0 + r < rows ? c0 + r : rows - 1];
    const uint32_t under = small_line(am);
    uint32_t seen = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) seen += is_small(t[kk + j][r], under) ? 1u : 0u;
    // (The row's eight lanes.)
    seen += __shfl_xor(seen, 1);
    seen += __shfl_xor(seen, 2);
    seen += __shfl_xor(seen, 4);
    if (c0 + r < rows && (item & 7) == 0 && am <= __uint_as_float(0x7f800000u)) {
      if (seen > 0) atomicAdd(small + c0 + r, seen);
      if (seen * 8 > (uint32_t)depth || am == __uint_as_float(0x7f800000u))
        list_row(again, side, row0 + c0 + r);
    }
    if (c0 + r < rows && k0 + line * kChunk < Kp) {
      const int e = split_exp(am);
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint2 s = split2(t[kk + 2 * j][r], t[kk + 2 * j + 1][r], e);
        hi[j] = s.x;
        lo[j] = s.y;
      }
      char* q = (char*)P + (c0 + r) * (int64_t)Kp * 4 + (k0 / kChunk + line) * 128 + part * 16;
      *(uint4*)q = uint4{hi[0], hi[1], hi[2], hi[3]};
      *(uint4*)(q + 64) = uint4{lo[0], lo[1], lo[2], lo[3]};
    }
  }
}

struct GemmF32Args {
  const uint16_t* xp;   // pieces [M][Kp]
  const uint16_t* wp;   // pieces [N][Kp]
  const float* xmax;    // [M]
  const float* wmax;    // [N]
  const uint32_t* xsmall;  // counts, the same
  const uint32_t* wsmall;
  float least;          // of an output (before the row scales) per small element
  float* out;           // Y, or the partial sums [splits][M][ldo]
  int64_t ldo, split_stride;
  int M, N, K, Kp, splits;
  int accumulate;       // add to out
  Again again;
  int64_t m0, n0;       // the block's first rows
};

// One TW x TX tile of Y (TW along N) over one share of k. MFMA-bound (three MFMAs per 32 k
// of each 16 x 16 block): M 1024, N 16384, K 1024 (one tile per CU) takes 90 us, 382 TFLOP/s
// of fp32 products or 1.15 PFLOP/s of MFMAs, the rate of the same K loop on plain 16-bit
// operands; with both operands' splitting the whole N 131072 product runs at 300 TFLOP/s
// (915 us, hipBLASLt's fp32 1940 us; 12 us of it clearing the lists and looking at them, empty).
template <typename Cfg>
__global__ __launch_bounds__(Cfg::kThreads) void gemm_f32_kernel(GemmF32Args a) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rl = lane & 15, q = lane >> 4;
  const int mt = (a.M + Cfg::TX - 1) / Cfg::TX;
  const int nt = (a.N + Cfg::TW - 1) / Cfg::TW;
  // M tiles fastest, then N, then the shares of k; each XCD a contiguous range, so the M
  // tiles of a W tile read it through one L2.
  const int n = (int)gridDim.x, lin = (int)blockIdx.x;
  const int logical = n % kXCDs ? lin : (lin % kXCDs) * (n / kXCDs) + lin / kXCDs;
  const int z = logical / (mt * nt);
  const int tile = logical - z * (mt * nt);
  const int m0 = tile % mt * Cfg::TX;
  const int n0 = tile / mt * Cfg::TW;
  const int steps = a.Kp / kChunk;
  const int s_lo = (int)((int64_t)steps * z / a.splits);
  const int s_hi = (int)((int64_t)steps * (z + 1) / a.splits);
  const int ldk = a.Kp * 2;  // 16-bit pieces per row
  floatx4 acc[Cfg::WB][Cfg::XB];
#pragma unroll
  for (int i = 0; i < Cfg::WB; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::XB; ++j) acc[i][j] = (floatx4){};
  // Rows past the matrix read its last row; their results are not stored.
  auto rows_of = [&](const uint16_t* base, int r0, int count) {
    return [=](int g, int k0, int i, uint32_t& voff, const DmaLane& dl) -> const void* {
      const int gb = r0 + g < count ? r0 + g : count - 1;
      const int r = r0 + g + dl.lrow < count ? r0 + g + dl.lrow : count - 1;
      voff = (uint32_t)((r - gb) * ldk * 2) + dl.cb(i);
      return base + ((int64_t)gb * ldk + s_lo * kBK + k0);
    };
  };
  // (A short last block of k may leave a share empty.)
  if (s_hi > s_lo)
    tile_kloop_cfg<Cfg, _Float16, true>((s_hi - s_lo) * kBK, lds, acc, rows_of(a.wp, n0, a.N),
                                        rows_of(a.xp, m0, a.M));

  // The tile's row exponents and lines through LDS, W's rows and then X's, one per thread.
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();
  static_assert(Cfg::kThreads == Cfg::TW + Cfg::TX, "a row of the tile each");
  {
    const int t = (int)threadIdx.x;
    const bool of_w = t < Cfg::TW;
    const int r0 = of_w ? n0 + t : m0 + t - Cfg::TW, count = of_w ? a.N : a.M;
    const int r = r0 < count ? r0 : count - 1;
    const float am = of_w ? a.wmax[r] : a.xmax[r];
    const uint32_t j = of_w ? a.wsmall[r] : a.xsmall[r];
    ((int*)lds)[t] = split_exp(am);
    ((float*)lds)[Cfg::kThreads + t] = line_of(am, j, a.least);
  }
  __syncthreads();
  float* out = a.out + z * a.split_stride;
  const int wn = wave / Cfg::NW_X, wm = wave % Cfg::NW_X;
  const int nt0 = wn * (Cfg::TW / Cfg::NW_W) + 4 * q;   // of the tile
  const int mt0 = wm * (Cfg::TX / Cfg::NW_X) + rl;
  const bool vec = (a.ldo & 3) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int nb = 0; nb < Cfg::WB; ++nb) {
    const int nn = n0 + nt0 + nb * 16;
    const int4 we4 = *(const int4*)(lds + (nt0 + nb * 16) * 4);
    const float4 wj4 = *(const float4*)(lds + (Cfg::kThreads + nt0 + nb * 16) * 4);
    const int we[4] = {we4.x, we4.y, we4.z, we4.w};
    const float wj[4] = {wj4.x, wj4.y, wj4.z, wj4.w};
#pragma unroll
    for (int mb = 0; mb < Cfg::XB; ++mb) {
      const int mt_ = Cfg::TW + mt0 + mb * 16;
      const int m = m0 + mt0 + mb * 16;
      if (m >= a.M || nn >= a.N) continue;
      const int xe = ((const int*)lds)[mt_];
      const float xj = ((const float*)lds)[Cfg::kThreads + mt_];
      float v[4];
      bool small = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = __builtin_amdgcn_ldexpf(acc[nb][mb][i], -(xe + we[i]));
        small |= fabsf(acc[nb][mb][i]) < xj + wj[i];
      }
      if (small) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nn + i < a.N && fabsf(acc[nb][mb][i]) < xj + wj[i])
            list_out(a.again, a.m0 + m, a.n0 + nn + i);
      }
      float* o = out + (int64_t)m * a.ldo + nn;
      if (vec && nn + 4 <= a.N) {
        floatx4 r = {v[0], v[1], v[2], v[3]};
        if (a.accumulate) r += *(const floatx4*)o;
        *(floatx4*)o = r;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nn + i < a.N) o[i] = a.accumulate ? o[i] + v[i] : v[i];
      }
    }
  }
}

// A block of Y (+)= the sum of its partial sums, in order of k, and the listing of its outputs, by
// the partial sums' magnitudes (over all blocks of k that they hold: `blocks` of row maxima and
// counts, `step` words apart).
struct SumArgs {
  const float* part;
  int64_t stride;
  int splits;
  float* Y;
  int64_t ldy;
  int N;
  int64_t total;
  int accumulate;
  const float* xmax;
  const float* wmax;
  int64_t to_small;   // words from a row's maximum to its count
  int blocks;
  int64_t step;
  float least;
  Again again;
  int64_t m0, n0;
};
__global__ __launch_bounds__(256) void sum_splits_kernel(SumArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.total) return;
  const int64_t m = i / a.N, n = i - m * a.N;
  float line = 0.f;
  for (int b = 0; b < a.blocks; ++b) {
    const float* xm = a.xmax + b * a.step + m;
    const float* wm = a.wmax + b * a.step + n;
    const float l = line_of(*xm, *(const uint32_t*)(xm + a.to_small), a.least) +
                    line_of(*wm, *(const uint32_t*)(wm + a.to_small), a.least);
    if (l > 0.f) line += __builtin_amdgcn_ldexpf(l, -(split_exp(*xm) + split_exp(*wm)));
  }
  float* y = a.Y + m * a.ldy + n;
  float s = a.part[i], t = fabsf(s);
  for (int z = 1; z < a.splits; ++z) {
    const float p = a.part[z * a.stride + i];
    s += p;
    t += fabsf(p);
  }
  *y = a.accumulate ? *y + s : s;
  if (t < line) list_out(a.again, a.m0 + m, a.n0 + n);
}

// The listed rows' outputs again, from the operands: row by row of X with all of W, and the other
// way round, in tiles of 32 listed rows by 64 rows of the other operand. Short lists (a row or
// two): a workgroup's 8 waves share a tile's k and add their parts in order through LDS. Long ones:
// each wave has a tile of its own (all rows of X at M 1024, N 131072, K 1024 3.1 ms, 90 TFLOP/s).
// Fragments are read straight from the operands (rows of 64 bytes or more, through L2), two steps
// of 16 k ahead. Then the listed outputs, one wave to each, or all of the workgroup's where k is
// long.
constexpr int kRowsThreads = 512;
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kRowsL = 32, kRowsO = 64;  // listed rows and others per tile
constexpr unsigned kRowsGrid = 512;
struct AgainArgs {
  const float* A[2];   // the operand whose rows are listed: X, then W
  int64_t sr[2], sk[2];
  int n[2];            // rows of X and of W
  Again again;
  float* Y;
  int64_t ldy;
  int K;
};

// acc += 32 rows by 64 over the steps of 16 k from s_lo to s_hi; lp and op are this lane's rows. V:
// k contiguous in both, in whole aligned fours.
template <bool V>
__device__ inline void again_product(const float* const (&lp)[2], const float* const (&op)[4],
                                     int64_t lsk, int64_t osk, int K, int s_lo, int s_hi, int kq,
                                     floatx4 (&acc)[2][4]) {
  if (s_lo >= s_hi) return;
  floatx4 lf[2][2], of[2][4];
  // Four k of this lane's row in a step. Past the end the last k again, which is not used.
  auto get = [&](const float* p, int64_t sk, int s) {
    const int k = (s < s_hi ? s : s_hi - 1) * 16 + 4 * kq;
    floatx4 v;
    if constexpr (V) {
      v = *(const floatx4*)(p + (k < K ? k : K - 4));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = p[(int64_t)(k + i < K ? k + i : K - 1) * sk];
    }
    return v;
  };
  auto fetch = [&](int buf, int s) {
#pragma unroll
    for (int i = 0; i < 2; ++i) lf[buf][i] = get(lp[i], lsk, s);
#pragma unroll
    for (int i = 0; i < 4; ++i) of[buf][i] = get(op[i], osk, s);
  };
  fetch(0, s_lo);
  fetch(1, s_lo + 1);
  for (int s0 = s_lo; s0 < s_hi; s0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k0 = (s0 + u) * 16 + 4 * kq;
      floatx4 lc[2], oc[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool in = s0 + u < s_hi && k0 + k < K;
#pragma unroll
        for (int i = 0; i < 2; ++i) lc[i][k] = in ? lf[u][i][k] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) oc[i][k] = in ? of[u][i][k] : 0.f;
      }
      fetch(u, s0 + u + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(oc[j][k], lc[i][k], acc[i][j], 0, 0, 0);
    }
  }
}

__global__ __launch_bounds__(kRowsThreads) void gemm_f32_again_kernel(AgainArgs a) {
  __shared__ floatx4 red[kRowsWaves][8][64];
  const int lane = threadIdx.x & 63, rl = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int steps = (a.K + 15) / 16;
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {
    const int count = (int)a.again.counts[side];
    const int others = (a.n[1 - side] + kRowsO - 1) / kRowsO;
    const int listed = (count + kRowsL - 1) / kRowsL;
    const int64_t tiles = (int64_t)listed * others;
    const bool own = tiles >= (int64_t)kRowsGrid * kRowsWaves;
    const int s_lo = own ? 0 : (int)((int64_t)steps * wave / kRowsWaves);
    const int s_hi = own ? steps : (int)((int64_t)steps * (wave + 1) / kRowsWaves);
    // The shorter axis fastest, a contiguous range of tiles to an XCD, so the longer operand is
    // read once.
    const int64_t group = (blockIdx.x % kXCDs) * (kRowsGrid / kXCDs) + blockIdx.x / kXCDs;
    const int64_t first = own ? group * kRowsWaves + wave : group;
    const int64_t stride = own ? kRowsGrid * kRowsWaves : kRowsGrid;
    const float* L = a.A[side];
    const float* O = a.A[1 - side];
    const int64_t lsk = a.sk[side], osr = a.sr[1 - side], osk = a.sk[1 - side];
    const bool lvec = lsk == 1 && a.sr[side] % 4 == 0 && a.K % 4 == 0 && ((uintptr_t)L & 15) == 0;
    const bool ovec = osk == 1 && osr % 4 == 0 && a.K % 4 == 0 && ((uintptr_t)O & 15) == 0;
#pragma unroll 1
    for (int64_t tile = first; tile < tiles; tile += stride) {
      const int l0 = (int)(listed < others ? tile % listed : tile / others) * kRowsL;
      const int o0 = (int)(listed < others ? tile / listed : tile % others) * kRowsO;
      const float* lp[2];
      const float* op[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int j = l0 + i * 16 + rl < count ? l0 + i * 16 + rl : count - 1;
        lp[i] = L + (int64_t)a.again.rows[side][j] * a.sr[side];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = o0 + i * 16 + rl < a.n[1 - side] ? o0 + i * 16 + rl : a.n[1 - side] - 1;
        op[i] = O + (int64_t)r * osr;
      }
      floatx4 acc[2][4];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (lvec && ovec)
        again_product<true>(lp, op, lsk, osk, a.K, s_lo, s_hi, kq, acc);
      else
        again_product<false>(lp, op, lsk, osk, a.K, s_lo, s_hi, kq, acc);
      // Four consecutive others from o on of listed row j.
      auto put = [&](int j, int o, const floatx4& v) {
        if (j >= count) return;
        const int64_t row = a.again.rows[side][j];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (o + e < a.n[1 - side]) {
            // (What both lists hold is written with the rows of X.)
            if (side == 0)
              a.Y[row * a.ldy + o + e] = v[e];
            else if (a.again.mark[0][o + e] == 0u)
              a.Y[(int64_t)(o + e) * a.ldy + row] = v[e];
          }
      };
      if (own) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) put(l0 + i * 16 + rl, o0 + j * 16 + 4 * kq, acc[i][j]);
        continue;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) red[wave][i * 4 + j][lane] = acc[i][j];
      __syncthreads();
      floatx4 v = red[0][wave][lane];
#pragma unroll
      for (int w = 1; w < kRowsWaves; ++w) v += red[w][wave][lane];
      put(l0 + (wave >> 2) * 16 + rl, o0 + (wave & 3) * 16 + 4 * kq, v);
    }
  }
  // Listed outputs.
  const uint32_t listed = a.again.counts[2];
  const int outs = (int)(listed < kMaxOuts ? listed : kMaxOuts);
  const int per = a.K > 4096 ? kRowsWaves : 1;  // waves to an output
  const int slot = wave / per, part = wave % per, at_once = kRowsWaves / per;
  float* sums = (float*)red;
#pragma unroll 1
  for (int i0 = (int)blockIdx.x * at_once; i0 < outs; i0 += (int)kRowsGrid * at_once) {
    const int i = i0 + slot < outs ? i0 + slot : outs - 1;
    const int64_t m = a.again.outs[2 * i], n = a.again.outs[2 * i + 1];
    const float* x = a.A[0] + m * a.sr[0];
    const float* w = a.A[1] + n * a.sr[1];
    float sum = 0.f;
#pragma unroll 8
    for (int k = part * 64 + lane; k < a.K; k += per * 64)
      sum = fmaf(x[(int64_t)k * a.sk[0]], w[(int64_t)k * a.sk[1]], sum);
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) sum += __shfl_xor(sum, s);
    __syncthreads();
    if (lane == 0) sums[wave] = sum;
    __syncthreads();
    // (A listed row's were written above, maybe by another workgroup.)
    if (lane == 0 && part == 0 && i0 + slot < outs && a.again.mark[0][m] == 0u &&
        a.again.mark[1][n] == 0u) {
      for (int p = 1; p < per; ++p) sum += sums[wave + p];
      a.Y[m * a.ldy + n] = sum;
    }
  }
}

using Big = Tile256;
using Small = TileCfg<128, 128, 2, 2>;

// How one call runs: block sizes (rows of X, rows of W, columns of k), the tile and the
// shares of k per tile.
struct Plan {
  int64_t mb, nb, kb;
  bool big;
  int splits;
};

inline int64_t up(int64_t v, int64_t to) { return (v + to - 1) / to * to; }
inline int64_t padk(int64_t k) { return up(k, kChunk); }

Plan plan(int64_t M, int64_t N, int64_t K) {
  Plan p;
  // k is blocked where it is the long axis (both operands are then read along it) or the shorter
  // side does not fit one block: by 2 kBlockElems / longest, or 8192 where that is less and the
  // shorter side fits (each block of k passes over the output once more).
  p.kb = K;
  int64_t elems = kBlockElems;
  const int64_t longest = M > N ? M : N, shortest = M > N ? N : M;
  if ((K > longest && K * longest > 2 * kBlockElems) || K * shortest > kBlockElems) {
    int64_t by_short = kBlockElems / up(shortest, 256) / 256 * 256;
    if (by_short > 8192) by_short = 8192;
    p.kb = 2 * kBlockElems / longest;
    if (p.kb < by_short) p.kb = by_short;
    // (Of equal length, or the last one's launches would be mostly overhead.)
    const int64_t blocks = p.kb > 0 ? (K + p.kb - 1) / p.kb : K;
    p.kb = up((K + blocks - 1) / blocks, 256);
    if (p.kb > K) p.kb = K;
  }
  if (K > longest) elems = 2 * kBlockElems;
  auto rows = [&](int64_t r) {
    int64_t most = elems / padk(p.kb) / 256 * 256;
    if (most < 256) most = 256;
    return r < most ? r : most;
  };
  p.mb = rows(M);
  p.nb = rows(N);
  // A block of the longer operand in whole rounds of one 256 x 256 tile per CU, where it has
  // that many.
  auto rounds = [&](int64_t& blk, int64_t total, int64_t other) {
    if (blk >= total) return;
    int64_t g = kCUsF;
    for (int64_t o = (other + 255) / 256; g > 1 && o % 2 == 0; o /= 2) g /= 2;
    if (blk / 256 >= g) blk = blk / 256 / g * g * 256;
  };
  rounds(p.nb, N, p.mb);
  rounds(p.mb, M, p.nb);
  const int64_t t256 = ((p.mb + 255) / 256) * ((p.nb + 255) / 256);
  const int64_t t128 = ((p.mb + 127) / 128) * ((p.nb + 127) / 128);
  // The 128 x 128 tile where one side is short or rows of X would be padding (M 273 N 73728 K 384
  // 167 / 136 us; padding of W's rows costs less than the smaller tile does, M 30720 N 320 K 534
  // 104 / 114), or the 256 x 256 tiles would leave CUs idle.
  p.big = p.mb > 128 && p.nb > 128 && up(p.mb, 256) * 8 <= up(p.mb, 128) * 9 &&
          t256 >= kCUsF * 3 / 4;
  const int64_t tiles = p.big ? t256 : t128;
  const int64_t slots = p.big ? kCUsF : 2 * kCUsF;  // workgroups resident at once
  const int64_t steps = padk(p.kb) / kChunk;
  int64_t z = 1;
  if (tiles * 2 <= slots) {
    z = slots / tiles;
    if (z > steps / 8) z = steps / 8;
    if (z > 64) z = 64;
    if (z < 1) z = 1;
  }
  p.splits = (int)z;
  return p;
}

// Row maxima of every block that a call splits, in order, and after them the rows' counts of small
// elements: one word each per row of each.
int64_t row_words(const Plan& p, int64_t M, int64_t N, int64_t K) {
  const int64_t kblocks = (K + p.kb - 1) / p.kb, mblocks = (M + p.mb - 1) / p.mb;
  return up(2 * kblocks * (M + N * (p.nb < N ? mblocks : 1)), 64);
}

// After them, the marks of X's and W's rows and the three counts (these and the words above start
// from zero); then the lists of rows and of outputs.
int64_t mark_words(int64_t M, int64_t N) { return up(M + N + 3, 64); }
int64_t list_words(int64_t M, int64_t N) { return up(M + N, 64) + 2 * kMaxOuts; }

int64_t f32_workspace(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const Plan p = plan(M, N, K);
  const int64_t kp = padk(p.kb);
  int64_t b = up(p.mb * kp * 4, 256) + up(p.nb * kp * 4, 256) + row_words(p, M, N, K) * 4 +
              (mark_words(M, N) + list_words(M, N)) * 4;
  if (p.splits > 1) b += p.splits * p.mb * p.nb * 4;
  return b;
}

// Pieces of rows [0, rows) and columns [0, K) of a view with element
// (r, k) at A[r * sr + k * sk], the rows' maxima and counts, and rows listed from row0 on.
int split_operand(const float* A, int64_t sr, int64_t sk, int64_t rows, int64_t K, uint16_t* P,
                  float* amax, uint32_t* small, const Again& again, int side, int64_t row0, hipStream_t s) {
  const int Kp = (int)padk(K);
  if (sk == 1) {
    const unsigned g4 = (unsigned)((rows + 3) / 4), g1 = (unsigned)rows;
    const bool v4 = sr % 4 == 0 && K % 4 == 0 && aligned(A, 16);
    if (v4 && K <= 1024)
      split_rows_kernel<4, 4, 1><<<g4, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax, small,
                                                     again, side, row0);
    else if (v4 && K <= 2048)
      split_rows_kernel<4, 8, 1><<<g4, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax, small,
                                                     again, side, row0);
    else if (v4 && K <= 16384)
      split_rows_kernel<4, 16, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax, small,
                                                     again, side, row0);
    else if (v4)
      split_rows_kernel<4, 0, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax, small,
                                                     again, side, row0);
    else
      split_rows_kernel<2, 0, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax, small,
                                                     again, side, row0);
    return launch_status();
  }
  col_max_kernel<<<dim3((unsigned)((rows + 255) / 256), (unsigned)((K + kStrip - 1) / kStrip)), 256, 0,
                   s>>>(A, sk, rows, (int)K, (uint32_t*)amax);
  split_cols_kernel<<<dim3((unsigned)((rows + kTrT - 1) / kTrT), (unsigned)((K + kTrT - 1) / kTrT)), 256,
                      0, s>>>(A, sk, rows, (int)K, Kp, P, amax, small, again, side, row0);
  return launch_status();
}

constexpr int kMaxDevices = 64;
std::atomic<bool> g_f32_attr_set[kMaxDevices];

}  // namespace
}  // namespace mqc

using namespace mqc;

extern "C" {

int64_t mqc_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return MQC_E_SHAPE;
  if (M > (1LL << 30) || N > (1LL << 30) || K > (1LL << 30)) return MQC_E_LIMIT;
  return f32_workspace(M, N, K);
}

int mqc_gemm_f32(const float* X, int64_t x_row, int64_t x_col, const float* W, int64_t w_row,
                 int64_t w_col, float* Y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  if (M < 0 || N < 0 || K < 0) return MQC_E_SHAPE;
  if (M == 0 || N == 0) return MQC_OK;
  if (K == 0 || ldy < N) return MQC_E_SHAPE;
  if (x_row < 0 || x_col < 0 || w_row < 0 || w_col < 0 || (x_row != 1 && x_col != 1) ||
      (w_row != 1 && w_col != 1))
    return MQC_E_SHAPE;
  if (!X || !W || !Y || !workspace) return MQC_E_NULL;
  if (!aligned(X, 4) || !aligned(W, 4) || !aligned(Y, 4) || !aligned(workspace, 256))
    return MQC_E_ALIGN;
  if (M > (1LL << 30) || N > (1LL << 30) || K > (1LL << 30)) return MQC_E_LIMIT;
  const Plan p = plan(M, N, K);
  const int64_t kp = padk(p.kb);
  // 32-bit lane offsets inside an 8-row group of pieces, and 16-bit grid rows.
  if (kp * 4 * 8 >= (1LL << 31) || (p.kb + kStrip - 1) / kStrip > 65535 ||
      (p.mb + 255) / 256 * ((p.nb + 255) / 256) * 4 * p.splits > 0x7fffffffLL)
    return MQC_E_LIMIT;
  if (workspace_bytes < f32_workspace(M, N, K)) return MQC_E_SPACE;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return MQC_E_LIMIT;
  if (!g_f32_attr_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute((const void*)gemm_f32_kernel<Big>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, Big::kStagesBytes);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)gemm_f32_kernel<Small>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, Small::kStagesBytes);
    if (e != hipSuccess) return (int)e;
    g_f32_attr_set[dev].store(true, std::memory_order_release);
  }
  hipStream_t s = (hipStream_t)stream;
  char* w = (char*)workspace;
  uint16_t* xp = (uint16_t*)w;
  w += up(p.mb * kp * 4, 256);
  uint16_t* wp = (uint16_t*)w;
  w += up(p.nb * kp * 4, 256);
  uint32_t* next_max = (uint32_t*)w;
  const int64_t words = row_words(p, M, N, K);
  w += words * 4;
  uint32_t* marks = (uint32_t*)w;
  const int64_t marked = mark_words(M, N);
  w += marked * 4;
  uint32_t* lists = (uint32_t*)w;
  w += list_words(M, N) * 4;
  float* part = (float*)w;
  float *xmax = nullptr, *wmax = nullptr;
  const int64_t to_small = words / 2;
  const Again again{{lists, lists + M}, {marks, marks + M}, lists + up(M + N, 64), marks + M + N};
  // (A small element is off by 2^-25 of a piece, times 2^15 at most: 2^-28 K of this.)
  const float least = K > 256 ? 0x1p18f / (float)K : 0x1p10f;
  // (The maxima over columns are taken by atomics, from zero.)
  const bool by_col = x_col != 1 || w_col != 1;
  const int64_t zeros = marked + (by_col ? words : 0);
  fill_zero_kernel<<<(unsigned)((zeros + 255) / 256), 256, 0, s>>>(
      by_col ? next_max : marks, zeros);
  int st = launch_status();
  if (st != MQC_OK) return st;
  for (int64_t k0 = 0; k0 < K; k0 += p.kb) {
    const int64_t kn = K - k0 < p.kb ? K - k0 : p.kb;
    for (int64_t m0 = 0; m0 < M; m0 += p.mb) {
      const int64_t mn = M - m0 < p.mb ? M - m0 : p.mb;
      const float* Xb = X + m0 * x_row + k0 * x_col;
      xmax = (float*)next_max;
      next_max += mn;
      st = split_operand(Xb, x_row, x_col, mn, kn, xp, xmax, (uint32_t*)xmax + to_small, again, 0, m0,
                         s);
      if (st != MQC_OK) return st;
      for (int64_t n0 = 0; n0 < N; n0 += p.nb) {
        const int64_t nn = N - n0 < p.nb ? N - n0 : p.nb;
        const float* Wb = W + n0 * w_row + k0 * w_col;
        // (The pieces of a W that fits one block outlive the blocks of X.)
        if (m0 == 0 || p.nb < N) {
          wmax = (float*)next_max;
          next_max += nn;
          st = split_operand(Wb, w_row, w_col, nn, kn, wp, wmax, (uint32_t*)wmax + to_small, again, 1,
                             n0, s);
          if (st != MQC_OK) return st;
        }
        GemmF32Args a{};
        a.xp = xp; a.wp = wp; a.xmax = xmax; a.wmax = wmax;
        a.xsmall = (uint32_t*)xmax + to_small; a.wsmall = (uint32_t*)wmax + to_small;
        a.M = (int)mn; a.N = (int)nn; a.K = (int)kn; a.Kp = (int)padk(kn);
        a.splits = p.splits;
        a.least = p.splits > 1 ? 0.f : least;
        a.again = again; a.m0 = m0; a.n0 = n0;
        float* const Yb = Y + m0 * ldy + n0;
        // (One block of the output keeps its partial sums over the blocks of k.)
        const bool keeps = p.mb >= M && p.nb >= N;
        a.accumulate = k0 > 0 && (p.splits == 1 || keeps);
        if (p.splits > 1) {
          a.out = part;
          a.ldo = nn;
          a.split_stride = p.mb * p.nb;
        } else {
          a.out = Yb;
          a.ldo = ldy;
        }
        const int t = p.big ? 256 : 128;
        const unsigned grid = (unsigned)((mn + t - 1) / t * ((nn + t - 1) / t) * p.splits);
        if (p.big)
          gemm_f32_kernel<Big><<<grid, Big::kThreads, Big::kStagesBytes, s>>>(a);
        else
          gemm_f32_kernel<Small><<<grid, Small::kThreads, Small::kStagesBytes, s>>>(a);
        if (p.splits > 1 && (!keeps || k0 + kn == K)) {
          SumArgs u{};
          u.part = part; u.stride = a.split_stride; u.splits = p.splits;
          u.Y = Yb; u.ldy = ldy; u.N = (int)nn; u.total = mn * nn;
          u.accumulate = k0 > 0 && !keeps;
          // (Every block of k has the M + N words of one block of X and of W.)
          const int64_t before = keeps ? k0 / p.kb * (M + N) : 0;
          u.xmax = xmax - before; u.wmax = wmax - before; u.to_small = to_small;
          u.blocks = keeps ? (int)(k0 / p.kb) + 1 : 1;
          u.step = M + N; u.least = least;
          u.again = again; u.m0 = m0; u.n0 = n0;
          sum_splits_kernel<<<(unsigned)((mn * nn + 255) / 256), 256, 0, s>>>(u);
        }
        st = launch_status();
        if (st != MQC_OK) return st;
      }
    }
  }
  AgainArgs r{};
  r.A[0] = X; r.sr[0] = x_row; r.sk[0] = x_col; r.n[0] = (int)M;
  r.A[1] = W; r.sr[1] = w_row; r.sk[1] = w_col; r.n[1] = (int)N;
  r.again = again; r.Y = Y; r.ldy = ldy; r.K = (int)K;
  gemm_f32_again_kernel<<<kRowsGrid, kRowsThreads, 0, s>>>(r);
  return launch_status();
}

}  // extern "C"
