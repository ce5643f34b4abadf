// fp32 GEMM on the 16-bit matrix cores, at fp32 accuracy:
//   Y[m, n] = sum_k X(m, k) W(n, k),  fp32 in, fp32 accumulation, fp32 out,
// for the fp32 B/C projections and their gradients (F.linear and its backward,
// mambaqc/layers/quaternion_linear.py:145-161). Each operand is a strided view with either
// k or the row index contiguous, so one entry point serves the forward (x, W), the input
// gradient (gy, W transposed) and the weight gradient (gy transposed, x transposed).
//
// Why. The fp32 matrix rate of gfx950 is 157 TFLOP/s, and hipBLASLt reaches 115-153 of them
// on these shapes; the fp16 rate is 16 times that. An fp32 value times a power of two of its row is split into two fp16
// pieces, a = hi + lo (11 significant bits each, lo exact to 2^-24 of the value's
// binade or 2^-40 of the row's largest magnitude), and a product takes three MFMAs, hi hi + hi lo + lo hi, into one fp32
// accumulator. What is dropped (lo lo, and what lo rounds away) is about 2^-24 of a product,
// random in sign, and an MFMA adds 32 products per rounding of the accumulator where the
// fp32 one adds 4: the error against 64 bits is not larger than hipBLASLt's fp32
// (tests/test_gpu_gemm_f32.py measures both).
//
//   - Row scale: 2^(14 - exponent of the row's largest |a|), so hi never overflows; taken
//     back in the epilogue with ldexp. amax holds each row's largest |a| (as fp32 bits, the
//     maximum taken on the bits, so that an inf or a NaN is the largest).
//   - Rows with a NaN or an inf: their amax says so; a NaN row's outputs are NaN, and those of a
//     row with an inf are computed in the epilogue from the fp32 operands with a plain fp32 loop.
//   - Layout of the pieces: per row and 32 columns of k, 32 hi pieces and then 32 lo pieces
//     (128 bytes: one K step of mfma_tile.hpp's loop), columns past K zero.
//   - Blocks: an operand is split a block at a time (kBlockElems, 64 MiB of pieces), and each
//     block is multiplied while its pieces are still in the 256 MiB Infinity Cache. Long k
//     (the input gradient's) is blocked too, each block adding to the partial sums; its
//     blocks are twice as large, since each adds a pass over the partial sums. Measured, blocks of
//     16 and 32 Mi elements (us): forward M 2048 N 65536 K 512 518 / 600, M 4096 N 98304
//     K 768 1874 / 2026; input gradients of the two 781 / 711 and 2890 / 2679. So is a k that
//     takes the shorter side past one block (the weight gradient of many tokens): that side would
//     otherwise be split again for every block of the longer one.
//   - Few output tiles in a block (the input gradient): k is shared by `splits` workgroups per
//     tile, whose partial sums a last launch adds in order, block by block. They are at most 512 tiles
//     of 128 x 128 (32 MiB) at a time, whatever the output's size.
#include <atomic>

#include "mfma_tile.hpp"

namespace mqc {
namespace {

using namespace mfma;

constexpr int kChunk = 32;                      // columns of k per 128-byte line of pieces
constexpr int64_t kBlockElems = 16 << 20;       // elements of one operand split at a time
constexpr int kCUsF = 256;

// Exponent added to a row's values before splitting: its largest magnitude lands in
// [2^14, 2^15). Zero for a row of zeros (and for a row that is not finite, which the
// epilogue does not take from the pieces).
__device__ inline int split_exp(float amax) {
  const uint32_t u = __float_as_uint(amax);
  if (u == 0u || u >= 0x7f800000u) return 0;
  return 15 - __builtin_amdgcn_frexp_expf(amax);
}
__device__ inline bool not_finite(float amax) { return __float_as_uint(amax) >= 0x7f800000u; }

__device__ inline uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// v * 2^e as hi + lo, packed for two values (hi in .x, lo in .y).
__device__ inline uint2 split2(float a, float b, int e) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  a = __builtin_amdgcn_ldexpf(a, e);
  b = __builtin_amdgcn_ldexpf(b, e);
  const h2 hi = {(_Float16)a, (_Float16)b};
  const h2 lo = {(_Float16)(a - (float)hi[0]), (_Float16)(b - (float)hi[1])};
  return uint2{__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo)};
}

// Rows with k contiguous: WPR waves per row (one, or four for rows longer than a wave holds).
// V = 4 where every row is 16-byte aligned. HELD: the row fits in registers (K <= 64 * WPR *
// V * HELD) and is read once; 0: it is read twice. Bound by HBM: 64 MiB of fp32 to 64 MiB of pieces in
// 27 us (5.0 TB/s, the copy rate); with one wave per row throughout, rows of 16384 took 60 us.
template <int V, int HELD, int WPR>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ A, int64_t ld,
                                                         int64_t rows, int K, int Kp,
                                                         uint16_t* __restrict__ P,
                                                         float* __restrict__ amax) {
  constexpr int TPR = 64 * WPR;
  constexpr int RPB = 4 / WPR;
  __shared__ uint32_t red[4];
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
  const int e = split_exp(am);
  if (tl == 0) amax[row] = am;
  if constexpr (HELD > 0) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) store((i * TPR + tl) * V, v[i], e);
  } else {
    for (int k = tl * V; k < Kp; k += TPR * V) {
      load(k, v[0]);
      store(k, v[0], e);
    }
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
                                                         const float* __restrict__ amax) {
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
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int item = i * 256 + (int)threadIdx.x;
    const int part = item & 3, line = (item >> 2) & 1, r = item >> 3;
    const int kk = line * kChunk + part * 8;
    if (c0 + r < rows && k0 + line * kChunk < Kp) {
      const int e = split_exp(amax[c0 + r]);
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
  const float* X;       // the operands themselves, for rows that are not finite
  const float* W;
  int64_t xm, xk, wn, wk;
  float* out;           // Y, or the partial sums [splits][M][ldo]
  int64_t ldo, split_stride;
  int M, N, K, Kp, splits;
  int accumulate;       // add to out
};

// One TW x TX tile of Y (TW along N) over one share of k. MFMA-bound (three MFMAs per 32 k
// of each 16 x 16 block): M 1024, N 16384, K 1024 (one tile per CU) takes 90 us, 382 TFLOP/s
// of fp32 products or 1.15 PFLOP/s of MFMAs, the rate of the same K loop on plain 16-bit
// operands; with both operands' splitting the whole N 131072 product runs at 288 TFLOP/s
// (954 us, hipBLASLt's fp32 1935 us).
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

  float* out = a.out + z * a.split_stride;
  const int wn = wave / Cfg::NW_X, wm = wave % Cfg::NW_X;
  const int nbase = n0 + wn * (Cfg::TW / Cfg::NW_W) + 4 * q;
  const int mbase = m0 + wm * (Cfg::TX / Cfg::NW_X) + rl;
  const bool vec = (a.ldo & 3) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int nb = 0; nb < Cfg::WB; ++nb) {
    const int nn = nbase + nb * 16;
    float wm4[4];
    int we[4];
    bool bad_w = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wm4[i] = a.wmax[nn + i < a.N ? nn + i : a.N - 1];
      we[i] = split_exp(wm4[i]);
      bad_w |= not_finite(wm4[i]);
    }
#pragma unroll
    for (int mb = 0; mb < Cfg::XB; ++mb) {
      const int m = mbase + mb * 16;
      if (m >= a.M || nn >= a.N) continue;
      const float xm1 = a.xmax[m];
      const int xe = split_exp(xm1);
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_ldexpf(acc[nb][mb][i], -(xe + we[i]));
      if (bad_w || not_finite(xm1)) {
        // A row with a NaN has nothing but NaNs in its outputs; one with an inf takes the plain
        // fp32 sum of this share of k.
        const int k1 = s_hi * kChunk < a.K ? s_hi * kChunk : a.K;
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
          if (nn + i >= a.N) break;
          const float wmax = i == 0 ? wm4[0] : i == 1 ? wm4[1] : i == 2 ? wm4[2] : wm4[3];
          if (!(not_finite(xm1) || not_finite(wmax))) continue;
          float sum = 0.f;
          if (xm1 != xm1 || wmax != wmax) {
            sum = __uint_as_float(0x7fc00000u);
          } else {
#pragma unroll 1
            for (int k = s_lo * kChunk; k < k1; ++k)
              sum = fmaf(a.X[m * a.xm + k * a.xk], a.W[(nn + i) * a.wn + k * a.wk], sum);
          }
          v[0] = i == 0 ? sum : v[0];
          v[1] = i == 1 ? sum : v[1];
          v[2] = i == 2 ? sum : v[2];
          v[3] = i == 3 ? sum : v[3];
        }
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

// A block of Y (+)= the sum of its partial sums, rows of N, in order of k.
__global__ __launch_bounds__(256) void sum_splits_kernel(const float* __restrict__ part,
                                                         int64_t stride, int splits,
                                                         float* __restrict__ Y, int64_t ldy, int N,
                                                         int64_t total, int accumulate) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  float* y = Y + i / N * ldy + i % N;
  float s = part[i];
  for (int z = 1; z < splits; ++z) s += part[z * stride + i];
  *y = accumulate ? *y + s : s;
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
  // side does not fit one block: by 2 kBlockElems / longest, or 8192 where that is less and the shorter
  // side fits (each block of k passes over the output once more).
  p.kb = K;
  const int64_t longest = M > N ? M : N, shortest = M > N ? N : M;
  if ((K > longest && K * longest > 2 * kBlockElems) || K * shortest > kBlockElems) {
    int64_t by_short = kBlockElems / up(shortest, 256) / 256 * 256;
    if (by_short > 8192) by_short = 8192;
    p.kb = 2 * kBlockElems / longest;
    if (p.kb < by_short) p.kb = by_short;
    p.kb = up(p.kb > 0 ? p.kb : 1, 256);
    if (p.kb > K) p.kb = K;
  }
  auto rows = [&](int64_t r) {
    int64_t most = kBlockElems / padk(p.kb) / 256 * 256;
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
  // The 128 x 128 tile where one side is short (a 256-row tile would be mostly padding) or
  // the 256 x 256 tiles would leave CUs idle.
  p.big = p.mb > 128 && p.nb > 128 && t256 >= kCUsF * 3 / 4;
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

// Row maxima of every block that a call splits, in order: one word per row of each.
int64_t max_words(const Plan& p, int64_t M, int64_t N, int64_t K) {
  const int64_t kblocks = (K + p.kb - 1) / p.kb, mblocks = (M + p.mb - 1) / p.mb;
  return up(kblocks * (M + N * (p.nb < N ? mblocks : 1)), 64);
}

int64_t f32_workspace(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const Plan p = plan(M, N, K);
  const int64_t kp = padk(p.kb);
  int64_t b = up(p.mb * kp * 4, 256) + up(p.nb * kp * 4, 256) + max_words(p, M, N, K) * 4;
  if (p.splits > 1) b += p.splits * p.mb * p.nb * 4;
  return b;
}

// Pieces and row maxima of rows [0, rows) and columns [0, K) of a view with element
// (r, k) at A[r * sr + k * sk].
int split_operand(const float* A, int64_t sr, int64_t sk, int64_t rows, int64_t K, uint16_t* P,
                  float* amax, hipStream_t s) {
  const int Kp = (int)padk(K);
  if (sk == 1) {
    const unsigned g4 = (unsigned)((rows + 3) / 4), g1 = (unsigned)rows;
    const bool v4 = sr % 4 == 0 && K % 4 == 0 && aligned(A, 16);
    if (v4 && K <= 1024)
      split_rows_kernel<4, 4, 1><<<g4, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax);
    else if (v4 && K <= 2048)
      split_rows_kernel<4, 8, 1><<<g4, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax);
    else if (v4 && K <= 16384)
      split_rows_kernel<4, 16, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax);
    else if (v4)
      split_rows_kernel<4, 0, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax);
    else
      split_rows_kernel<2, 0, 4><<<g1, 256, 0, s>>>(A, sr, rows, (int)K, Kp, P, amax);
    return launch_status();
  }
  col_max_kernel<<<dim3((unsigned)((rows + 255) / 256), (unsigned)((K + kStrip - 1) / kStrip)), 256, 0,
                   s>>>(A, sk, rows, (int)K, (uint32_t*)amax);
  split_cols_kernel<<<dim3((unsigned)((rows + kTrT - 1) / kTrT), (unsigned)((K + kTrT - 1) / kTrT)), 256,
                      0, s>>>(A, sk, rows, (int)K, Kp, P, amax);
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
  float* next_max = (float*)w;
  const int64_t words = max_words(p, M, N, K);
  w += words * 4;
  float* part = (float*)w;
  float *xmax = nullptr, *wmax = nullptr;
  // (The maxima over columns are taken by atomics, from zero.)
  if (x_col != 1 || w_col != 1) {
    fill_zero_kernel<<<(unsigned)((words + 255) / 256), 256, 0, s>>>((uint32_t*)next_max, words);
    const int st = launch_status();
    if (st != MQC_OK) return st;
  }
  for (int64_t k0 = 0; k0 < K; k0 += p.kb) {
    const int64_t kn = K - k0 < p.kb ? K - k0 : p.kb;
    for (int64_t m0 = 0; m0 < M; m0 += p.mb) {
      const int64_t mn = M - m0 < p.mb ? M - m0 : p.mb;
      const float* Xb = X + m0 * x_row + k0 * x_col;
      xmax = next_max;
      next_max += mn;
      int st = split_operand(Xb, x_row, x_col, mn, kn, xp, xmax, s);
      if (st != MQC_OK) return st;
      for (int64_t n0 = 0; n0 < N; n0 += p.nb) {
        const int64_t nn = N - n0 < p.nb ? N - n0 : p.nb;
        const float* Wb = W + n0 * w_row + k0 * w_col;
        // (The pieces of a W that fits one block outlive the blocks of X.)
        if (m0 == 0 || p.nb < N) {
          wmax = next_max;
          next_max += nn;
          st = split_operand(Wb, w_row, w_col, nn, kn, wp, wmax, s);
          if (st != MQC_OK) return st;
        }
        GemmF32Args a{};
        a.xp = xp; a.wp = wp; a.xmax = xmax; a.wmax = wmax;
        a.X = Xb; a.W = Wb; a.xm = x_row; a.xk = x_col; a.wn = w_row; a.wk = w_col;
        a.M = (int)mn; a.N = (int)nn; a.K = (int)kn; a.Kp = (int)padk(kn);
        a.splits = p.splits;
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
        if (p.splits > 1 && (!keeps || k0 + kn == K))
          sum_splits_kernel<<<(unsigned)((mn * nn + 255) / 256), 256, 0, s>>>(
              part, a.split_stride, p.splits, Yb, ldy, (int)nn, mn * nn, k0 > 0 && !keeps);
        st = launch_status();
        if (st != MQC_OK) return st;
      }
    }
  }
  return MQC_OK;
}

}  // extern "C"
