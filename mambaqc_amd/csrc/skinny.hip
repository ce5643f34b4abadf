// Skinny GEMM for the projections of the recurrent decode step (bf16 / fp16):
//   Y[M, N] = X[M, K] . W[N, K]^T (+ bias[N]),  M <= 16 rows, fp32 accumulation,
// the nn.Linear / F.linear layout of mambaqc/layers/quaternion_linear.py:145-172
// and of the block's nn.Linear layers (models/quaternion_mamba2_block.py:78-122)
// at the few token rows of one decode step. One launch can take up to four
// weights that share X (dt_proj, gate_proj, B_proj and C_proj), and the decode
// step's element-wise neighbours run inside the products (SK_CONV, SK_NORM_GATE):
// a step of a block is four launches, [in_proj + conv], [dt, gate, B, C], the SSM
// step and [LayerNorm + out_proj + gate].
//
// A decode step reads every weight once and does almost no arithmetic, so each
// projection is a read of W at HBM speed, and the small ones are a launch each.
// The product runs on the MFMA unit, which leaves the VALU idle and needs no
// cross-lane reductions:
//   - one wave per tile of 16 weight rows; per K step of 32 it issues one
//     v_mfma_f32_16x16x32 with W's 16 rows as the B operand (lane l holds 8
//     consecutive k of row l % 16, straight from HBM, 16 bytes per lane) and
//     X as the A operand (row l % 16 from LDS; lanes past M hold zeros);
//   - K steps are loaded in groups of 8 (8 KB per wave in flight), with enough
//     waves per CU (small register and LDS footprint) to cover HBM latency;
//   - the 16 x 16 result lands as rows 4 (l / 16) + i of column l % 16; the
//     lanes holding rows < M add the bias and store them.
// X (M x K, at most 64 KB) is copied to LDS once per workgroup, rows padded by
// 16 bytes so the A reads of different rows fall on different banks. Rows of W
// past N are clamped onto row N - 1 for the loads and never stored.
//
// Weights with few rows would leave most CUs idle with one wave per tile, so
// then 4, 8 or 16 waves share each tile's K (see skinny_launch).
//
// Weights with many rows, at most 8 token rows and K a multiple of 64 take the
// wide mode instead (skinny_wide_kernel): a tile reads each weight row as 64
// bytes per instruction (half a 128-byte line), while the wide mode's load
// instructions read 8 whole lines each and keep all of a row group's lines in
// flight; its products run on the VALU as dot2 instructions.
//
// Measured on MI355X at 4 rows (bf16): a pair of [1024 x 1024] weights in one
// launch 6.3 us, where hipBLASLt takes about 6.6 us per weight; [131072 x 1024]
// pairs (the small preset's B/C) 95-98 us in tiles against 99.7 us for two
// calls. The wide mode, same box, pairs at 4 rows unless noted, against tiles
// and hipBLASLt: [131072 x 1024] 87-90 / 100-102 / 114-115 us; the base
// preset's [393216 x 1536] 386-392 / 424-425 / 427 us (6.2 TB/s), at 1 row
// 369-371 / 414-419 / 436, at 8 rows 415-416 / 455-457 / 452-458;
// [524288 x 2048] 688-690 / 746 / 878-888 us. Decode steps of 4 tokens with
// every projection here: base preset 5.73 -> 5.30 ms eager and 5.68-5.73 ->
// 5.29-5.30 ms as a HIP graph against the B/C pair on hipBLASLt (same box;
// earlier, moving the other projections here took 5.89 -> 5.72 ms), small
// preset 2.05 -> 1.37 ms eager and 1.27 -> 1.09 ms as a graph.
#include <atomic>

#include "ssm_scan.hpp"

namespace mqc {
namespace {

typedef __bf16 skbf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 skf16x8 __attribute__((ext_vector_type(8)));
typedef float skfloatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int sku32x4 __attribute__((ext_vector_type(4)));

constexpr int kSkThreads = 256;
constexpr int kSkWaves = kSkThreads / 64;
constexpr int kSkMaxRows = 16;
constexpr int kSkStep = 32;  // K per MFMA
constexpr int kSkGroup = 8;  // K steps loaded together
constexpr int64_t kSkMaxLds = 64 << 10;  // X in LDS, plus the split modes' partial tiles
constexpr int kSkBlocksPerCU = 8;
constexpr int kSkCUs = 256;  // MI355X compute units

template <typename T> struct SkVec;
template <> struct SkVec<bf16_t> { using type = skbf16x8; };
template <> struct SkVec<f16_t> { using type = skf16x8; };

template <typename T>
__device__ inline skfloatx4 sk_mfma(typename SkVec<T>::type a, typename SkVec<T>::type b,
                                    skfloatx4 c) {
  if constexpr (std::is_same<T, bf16_t>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

constexpr int kSkMaxWeights = 4;

struct SkArgs {
  const void* x;
  const void* w[kSkMaxWeights];
  const void* bias[kSkMaxWeights];  // or nullptr
  void* y[kSkMaxWeights];
  int64_t n[kSkMaxWeights];
  int64_t tile_end[kSkMaxWeights];   // 16-row tiles of the weights up to and with this one
  int64_t group_end[kSkMaxWeights];  // 8-row groups (wide mode)
  int64_t tiles, groups;             // of all of them
  int M, K;
  // What the decode step fuses around the product (MODE below).
  // SK_CONV: columns n < conv_ch are the inputs of the causal conv + SiLU step, continued from
  // (and shifting) tail [M, conv_k - 1, conv_ch]; the other columns go to y[0] [M, N - conv_ch].
  const float* conv_w;   // [conv_ch, conv_k]
  const float* conv_b;   // [conv_ch] or nullptr
  void* tail;
  void* act;             // [M, conv_ch]
  int conv_ch, conv_k;
  // SK_NORM_GATE: x [M, K / 4, 4] goes through the quaternion LayerNorm first, and
  // y[0] = res + sigmoid(z) * product, z with row stride zs.
  const float* gamma;    // [K / 4]
  const float* beta;     // [K / 4, 4]
  const void* res;
  const void* z;
  int64_t zs;
  float eps;
};

// Which weight holds 16-row tile (8-row group) i, and its first tile (group).
__device__ inline int sk_which(const int64_t (&end)[kSkMaxWeights], int64_t i, int64_t& first) {
  int which = 0;
  first = 0;
#pragma unroll
  for (int v = 1; v < kSkMaxWeights; ++v)
    if (i >= end[v - 1]) {
      which = v;
      first = end[v - 1];
    }
  return which;
}

constexpr int SK_PLAIN = 0;
constexpr int SK_CONV = 1;
constexpr int SK_NORM_GATE = 2;
constexpr int kSkMaxTaps = 4;  // conv taps under SK_CONV

// Elements per LDS row of X.
__host__ __device__ inline int64_t sk_lds_row(int64_t K) { return K + 8; }

// What the epilogue of column n and rows m0 .. m0 + 3 reads, requested ahead of the product
// (each is a miss of about a microsecond where it is first used).
template <int MODE>
struct SkEpi {};
template <>
struct SkEpi<SK_CONV> {
  float w[kSkMaxTaps], b;
  uint16_t tail[4][kSkMaxTaps - 1];
};
template <>
struct SkEpi<SK_NORM_GATE> {
  uint16_t z[4], res[4];
};

template <int MODE>
__device__ inline void sk_epi_load(const SkArgs& a, SkEpi<MODE>& e, int m0, int64_t n, int64_t N) {
  if constexpr (MODE == SK_CONV) {
    const int taps = a.conv_k - 1;
    const int64_t c = n < a.conv_ch ? n : 0;
    e.b = a.conv_b ? a.conv_b[c] : 0.f;
#pragma unroll
    for (int j = 0; j < kSkMaxTaps; ++j) e.w[j] = j <= taps ? a.conv_w[c * a.conv_k + j] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < kSkMaxTaps - 1; ++j)
        e.tail[i][j] = j < taps && m0 + i < a.M
                           ? ((const uint16_t*)a.tail)[((int64_t)(m0 + i) * taps + j) * a.conv_ch + c]
                           : 0;
  } else if constexpr (MODE == SK_NORM_GATE) {
    const int64_t c = n < N ? n : N - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + i < a.M ? m0 + i : a.M - 1;
      e.z[i] = ((const uint16_t*)a.z)[m * a.zs + c];
      e.res[i] = ((const uint16_t*)a.res)[m * N + c];
    }
  }
}

// Element (m = m0 + i, n) of the product, rounded to T.
//   SK_CONV: one step of the causal conv + SiLU for the conv's channels (conv.hip's
//   conv_silu_step_kernel: the same sum in the same order and the rounding of the forward's
//   16-byte path, which conv_ch takes, being a multiple of 8). Only this lane reads and
//   writes (m, n)'s column of the tail.
//   SK_NORM_GATE: the residual and the gate (elementwise.hip's out_gate_kernel).
template <typename T, int MODE>
__device__ inline void sk_store(const SkArgs& a, const SkEpi<MODE>& e, int i, T* y, int m,
                                int64_t n, int64_t N, T v) {
  if constexpr (MODE == SK_PLAIN) {
    y[(int64_t)m * N + n] = v;
  } else if constexpr (MODE == SK_CONV) {
    if (n >= a.conv_ch) {
      y[(int64_t)m * (N - a.conv_ch) + (n - a.conv_ch)] = v;
      return;
    }
    const int taps = a.conv_k - 1;
    uint16_t* tc = (uint16_t*)a.tail + (int64_t)m * taps * a.conv_ch + n;
    float p = e.b, wl = e.w[0];
#pragma unroll
    for (int j = 0; j < kSkMaxTaps - 1; ++j)
      if (j < taps) {
        p = fmaf(e.w[j], io<T>::bits_to_f32(e.tail[i][j]), p);
        wl = e.w[j + 1];
      }
    p = fmaf(wl, io<T>::to_f32(v), p);
    float o = p * front_sigmoid(p);
    asm volatile("" : "+v"(o));  // (rounded to fp32 before the conversion)
    ((uint16_t*)a.act)[(int64_t)m * a.conv_ch + n] = (uint16_t)(pack2<T>(o, o) & 0xffffu);
#pragma unroll
    for (int j = 0; j < kSkMaxTaps - 1; ++j)
      if (j < taps) {
        const int jn = j + 1 < kSkMaxTaps - 1 ? j + 1 : j;
        tc[(int64_t)j * a.conv_ch] = j + 1 < taps ? e.tail[i][jn] : v.bits;
      }
  } else {
    const float g = 1.f / (1.f + __expf(-io<T>::bits_to_f32(e.z[i])));
    y[(int64_t)m * N + n] =
        io<T>::from_f32(fmaf(g, io<T>::to_f32(v), io<T>::bits_to_f32(e.res[i])));
  }
}

// The quaternion LayerNorm (qln.hip) of the X rows on their way to LDS: the workgroup's W waves
// share the rows, several to a row where there are more waves than rows, each lane holding at
// most kNormHeld quaternions of its row. Every workgroup normalises all rows again, which costs less than
// a launch of its own.
constexpr int kNormHeld = 12;
template <int W>
struct NormLane {
  int per, at_once, slot, first;  // waves per row, rows at a time, this wave's row and lane's start
  __device__ NormLane(int M) {
    per = W;
    while (per > 1 && (W / per) * 2 <= M) per >>= 1;
    at_once = W / per;
    const int wave = threadIdx.x >> 6;
    slot = wave / per;
    first = (wave % per) * 64 + (threadIdx.x & 63);
  }
};

template <int W>
__device__ inline void sk_norm_load(const SkArgs& a, const NormLane<W>& l, int m0,
                                    uint2 (&q)[kNormHeld]) {
  const int D = a.K / 4;
  const int m = m0 + l.slot < a.M ? m0 + l.slot : a.M - 1;
  const uint2* row = (const uint2*)a.x + (int64_t)m * D;
#pragma unroll
  for (int i = 0; i < kNormHeld; ++i) {
    const int c = l.first + i * l.per * 64;
    if (i * l.per * 64 < D) q[i] = row[c < D ? c : D - 1];
  }
}

template <int W>
__device__ inline void sk_norm_params(const SkArgs& a, const NormLane<W>& l, float (&gm)[kNormHeld],
                                      float4 (&bt)[kNormHeld]) {
  const int D = a.K / 4;
#pragma unroll
  for (int i = 0; i < kNormHeld; ++i) {
    const int c = l.first + i * l.per * 64;
    if (i * l.per * 64 < D) {
      gm[i] = a.gamma[c < D ? c : D - 1];
      bt[i] = ((const float4*)a.beta)[c < D ? c : D - 1];
    }
  }
}

template <typename T, int W>
__device__ inline void sk_norm_rows(const SkArgs& a, const NormLane<W>& l, uint2 (&q)[kNormHeld],
                                    const float (&gm)[kNormHeld], const float4 (&bt)[kNormHeld],
                                    unsigned char* lds, int64_t ldsRow) {
  __shared__ float red[2][W];
  const int D = a.K / 4;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  auto quat_of = [](const uint2& w, float (&v)[4]) {
    if constexpr (std::is_same<T, bf16_t>::value) {
      v[0] = __uint_as_float(w.x << 16); v[1] = __uint_as_float(w.x & 0xffff0000u);
      v[2] = __uint_as_float(w.y << 16); v[3] = __uint_as_float(w.y & 0xffff0000u);
    } else {
      v[0] = io<T>::bits_to_f32(w.x & 0xffffu); v[1] = io<T>::bits_to_f32(w.x >> 16);
      v[2] = io<T>::bits_to_f32(w.y & 0xffffu); v[3] = io<T>::bits_to_f32(w.y >> 16);
    }
  };
  auto total = [&](float s, int which) {
    // Within rows of 16 lanes by DPP (quad permutes, half-row and row mirrors), then across.
    s += lane_xor1(s);
    s += lane_xor2(s);
    s += dpp_mov<0x141>(s);
    s += dpp_mov<0x140>(s);
    auto row = [&](int l) {
      return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), l));
    };
    s = (row(0) + row(16)) + (row(32) + row(48));
    if (lane == 0) red[which][wave] = s;
    __syncthreads();
    float t = 0.f;
    for (int p = 0; p < l.per; ++p) t += red[which][l.slot * l.per + p];
    return t;
  };
  for (int m0 = 0; m0 < a.M; m0 += l.at_once) {
    if (m0 > 0) sk_norm_load<W>(a, l, m0, q);
    float n[kNormHeld], v[4], s = 0.f;
#pragma unroll
    for (int i = 0; i < kNormHeld; ++i)
      if (i * l.per * 64 < D) {
        quat_of(q[i], v);
        n[i] = sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3] + a.eps);
        s += l.first + i * l.per * 64 < D ? n[i] : 0.f;
      }
    const float mu = total(s, 0) * (1.f / (float)D);
    s = 0.f;
#pragma unroll
    for (int i = 0; i < kNormHeld; ++i)
      if (i * l.per * 64 < D) {
        const float c = n[i] - mu;
        s = l.first + i * l.per * 64 < D ? fmaf(c, c, s) : s;
      }
    const float rstd = 1.f / sqrtf(total(s, 1) * (1.f / (float)D) + a.eps);
    T* x = (T*)(lds + (int64_t)(m0 + l.slot) * ldsRow * 2);
#pragma unroll
    for (int i = 0; i < kNormHeld; ++i) {
      const int c = l.first + i * l.per * 64;
      if (m0 + l.slot < a.M && c < D) {
        quat_of(q[i], v);
        const float f = gm[i] * ((n[i] - mu) * rstd) / (n[i] + a.eps);
        const float o[4] = {fmaf(f, v[0], bt[i].x), fmaf(f, v[1], bt[i].y),
                            fmaf(f, v[2], bt[i].z), fmaf(f, v[3], bt[i].w)};
        store_vec<T, 4>(x + 4 * c, o);
      }
    }
  }
}

// SPLIT = 1: each wave owns whole tiles (4 per workgroup). SPLIT = 4, 8 or 16:
// the workgroup's SPLIT waves share one tile, each summing a contiguous part
// of K, and the partial 16 x 16 tiles are added through LDS (for weights with
// few rows, which would otherwise leave most CUs idle).
//
// MODE: SK_CONV and SK_NORM_GATE run the decode step's neighbouring element-wise steps in the
// product's prologue or epilogue, rounding where the separate launches store (each launch less is about
// 4 us of a decode step; see sk_norm_rows and sk_store below).
// The split kernels are latency-bound (a few KB per wave): the first group of weights is requested
// right after X, before X is normalised or stored, later groups one ahead, and a last short group as one
// batch, and the epilogue's operands with the first weights (requested where they are used, in_proj + conv
// took 8.4 us). Small preset, 4 rows: in_proj + conv step 5.9 us (9.4 in two launches), LayerNorm +
// out_proj + gate 11.6 (16.2 in three); base preset 7.1 and 17.1 (13.0, 21.6).
constexpr int kXHeld = 4;  // 16-byte pieces of X per thread requested ahead of the weights
template <typename T, int SPLIT, int MODE>
__global__ __launch_bounds__(SPLIT == 1 ? kSkThreads : 64 * SPLIT) void skinny_nt_kernel(SkArgs a) {
  using V = typename SkVec<T>::type;
  constexpr int NT = SPLIT == 1 ? kSkThreads : 64 * SPLIT;
  constexpr int WPB = NT / 64;                      // waves per workgroup
  constexpr int TPB = SPLIT == 1 ? WPB : 1;         // tiles per workgroup
  extern __shared__ __align__(16) unsigned char sk_lds[];
  const int K = a.K;
  const int M = a.M;
  const int64_t ldsRow = sk_lds_row(K);
  float* red = (float*)(sk_lds + M * ldsRow * 2);   // SPLIT x 64 lanes x 4 partials
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;  // the A row (token) and the B column (weight row) of this lane
  const int grp = lane >> 4;  // which 8 of a step's 32 k this lane holds
  const bool arow = col < M;
  const unsigned char* xa = sk_lds + ((arow ? col : 0) * ldsRow + 8 * grp) * 2;
  const int steps = K / kSkStep;
  // This wave's K steps: all of them, or its share of the tile's.
  const int s_lo = SPLIT == 1 ? 0 : (int)((int64_t)steps * wave / SPLIT);
  const int s_hi = SPLIT == 1 ? steps : (int)((int64_t)steps * (wave + 1) / SPLIT);

  // The weight, row and first element of this lane in a tile.
  int which = 0;
  int64_t N = 0, n = 0;
  const T* wp = nullptr;
  auto locate = [&](int64_t tile) {
    int64_t first = 0;
    which = MODE == SK_PLAIN ? sk_which(a.tile_end, tile, first) : 0;
    N = a.n[which];
    n = (tile - first) * 16 + col;
    wp = (const T*)a.w[which] + (n < N ? n : N - 1) * K + 8 * grp;
  };
  auto load_group = [&](V (&b)[kSkGroup], int s) {
#pragma unroll
    for (int u = 0; u < kSkGroup; ++u)
      if (s + u < s_hi) b[u] = *(const V*)(wp + (int64_t)(s + u) * kSkStep);
  };
  skfloatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto use_group = [&](const V (&b)[kSkGroup], int s) {
#pragma unroll
    for (int u = 0; u < kSkGroup; ++u)
      if (s + u < s_hi) {
        V av{};
        if (arow) av = *(const V*)(xa + (s + u) * kSkStep * 2);
        acc = sk_mfma<T>(av, b[u], acc);
      }
  };

  // (One wave stores a split tile.)
  SkEpi<MODE> epi;
  auto load_epi = [&]() {
    if (MODE != SK_PLAIN && (SPLIT == 1 || wave == 0)) sk_epi_load<MODE>(a, epi, 4 * grp, n, N);
  };
  const int per_row = K / 8;
  const int64_t pieces = (int64_t)M * per_row;
  auto put_piece = [&](int64_t i, sku32x4 v) {
    const int64_t r = i / per_row;
    *(sku32x4*)(sk_lds + (r * ldsRow + (i - r * per_row) * 8) * 2) = v;
  };
  V b[kSkGroup];
  if constexpr (SPLIT > 1 && MODE == SK_NORM_GATE) {
    const NormLane<WPB> l(M);
    uint2 q[kNormHeld];
    sk_norm_load<WPB>(a, l, 0, q);
    __builtin_amdgcn_sched_barrier(0);
    float gm[kNormHeld];
    float4 bt[kNormHeld];
    sk_norm_params<WPB>(a, l, gm, bt);
    __builtin_amdgcn_sched_barrier(0);
    locate(blockIdx.x);
    load_group(b, s_lo);
    load_epi();
    __builtin_amdgcn_sched_barrier(0);
    sk_norm_rows<T, WPB>(a, l, q, gm, bt, sk_lds, ldsRow);
  } else if constexpr (SPLIT > 1) {
    sku32x4 x[kXHeld] = {};
#pragma unroll
    for (int i = 0; i < kXHeld; ++i) {
      const int64_t c = threadIdx.x + (int64_t)i * NT;
      if (c < pieces) x[i] = ((const sku32x4*)a.x)[c];
    }
    __builtin_amdgcn_sched_barrier(0);
    if ((int64_t)blockIdx.x < a.tiles) {
      locate(blockIdx.x);
      load_group(b, s_lo);
      load_epi();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kXHeld; ++i) {
      const int64_t c = threadIdx.x + (int64_t)i * NT;
      if (c < pieces) put_piece(c, x[i]);
    }
    for (int64_t c = threadIdx.x + (int64_t)kXHeld * NT; c < pieces; c += NT)
      put_piece(c, ((const sku32x4*)a.x)[c]);
  } else {
    for (int64_t c = threadIdx.x; c < pieces; c += NT) put_piece(c, ((const sku32x4*)a.x)[c]);
  }
  __syncthreads();
  bool ready = SPLIT > 1;  // b holds the tile's first group
  for (int64_t tile0 = (int64_t)blockIdx.x * TPB; tile0 < a.tiles;
       tile0 += (int64_t)gridDim.x * TPB) {
    const int64_t tile = tile0 + (SPLIT == 1 ? wave : 0);
    // (SPLIT == 1: a wave past the last tile has nothing to do; no barrier follows.)
    if (tile < a.tiles) {
      acc = skfloatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (SPLIT > 1) {
        if (!ready) {
          locate(tile);
          load_group(b, s_lo);
          load_epi();
        }
        ready = false;
        for (int s = s_lo; s < s_hi; s += kSkGroup) {
          V next[kSkGroup];
          if (s + kSkGroup < s_hi) load_group(next, s + kSkGroup);
          __builtin_amdgcn_sched_barrier(0);
          use_group(b, s);
#pragma unroll
          for (int u = 0; u < kSkGroup; ++u) b[u] = next[u];
        }
      } else {
        locate(tile);
        load_epi();
        for (int s = s_lo; s < s_hi; s += kSkGroup) {
          load_group(b, s);
          use_group(b, s);
        }
      }
      if constexpr (SPLIT > 1) {
        // Partial tiles through LDS; wave 0 adds them in wave order.
        *(skfloatx4*)(red + (wave * 64 + lane) * 4) = acc;
      }
      bool store = true;
      if constexpr (SPLIT > 1) {
        __syncthreads();
        store = wave == 0;
        if (store) {
          acc = *(const skfloatx4*)(red + lane * 4);
#pragma unroll
          for (int w = 1; w < SPLIT; ++w) acc += *(const skfloatx4*)(red + (w * 64 + lane) * 4);
        }
        __syncthreads();  // red is rewritten by the next tile
      }
      if (store && n < N) {
        const T* bp = (const T*)a.bias[which];
        const float bv = bp ? io<T>::to_f32(bp[n]) : 0.f;
        T* yp = (T*)a.y[which];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 4 * grp + i;
          if (m < M) sk_store<T, MODE>(a, epi, i, yp, m, n, N, io<T>::from_f32(acc[i] + bv));
        }
      }
    }
  }
}

// Wide mode. A wave takes 8 weight rows at a time; lane l reads row l / 8 and
// the 16 bytes at (l % 8) * 16 of each 128-byte line of it, so one load
// instruction covers 8 whole lines, and all K / 64 lines of the row group are
// issued before the first is used (LINES = K / 64 for the unrolled widths, 0
// for any other K, which runs in groups of 8 lines). Each 16-byte piece is
// dotted with the matching 8 k of every token, X read from LDS (the lanes of
// one row read consecutive 16 bytes, the lanes of one piece the same ones), as
// four dot2 instructions (two 16-bit products added to an fp32 sum). The 8
// lanes of a row are summed by two quad permutes and a half-row mirror, after
// which lane p holds the row's output for token p. MP: token rows padded to a
// power of two (X rows past M are zeros in LDS and never stored).
template <typename T> struct SkDot;
template <> struct SkDot<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ static inline float dot8(v8 w, v8 x, float acc) {
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(w, w, 0, 1), __builtin_shufflevector(x, x, 0, 1), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(w, w, 2, 3), __builtin_shufflevector(x, x, 2, 3), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(w, w, 4, 5), __builtin_shufflevector(x, x, 4, 5), acc, false);
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(w, w, 6, 7), __builtin_shufflevector(x, x, 6, 7), acc, false);
  }
};
template <> struct SkDot<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  __device__ static inline float dot8(v8 w, v8 x, float acc) {
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(w, w, 0, 1), __builtin_shufflevector(x, x, 0, 1), acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(w, w, 2, 3), __builtin_shufflevector(x, x, 2, 3), acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(w, w, 4, 5), __builtin_shufflevector(x, x, 4, 5), acc, false);
    return __builtin_amdgcn_fdot2(__builtin_shufflevector(w, w, 6, 7), __builtin_shufflevector(x, x, 6, 7), acc, false);
  }
};

constexpr int kWideThreads = 256;
constexpr int kWideMaxRows = 8;
constexpr int64_t kWideMinGroups = 4096;  // 8-row groups (both weights) for the wide mode
constexpr int kWideGenericLines = 8;

template <typename T, int MP, int LINES>
__global__ __launch_bounds__(kWideThreads) void skinny_wide_kernel(SkArgs a) {
  using D = SkDot<T>;
  using V8 = typename D::v8;
  constexpr int WPB = kWideThreads / 64;
  extern __shared__ __align__(16) unsigned char sk_lds[];
  const int K = a.K;
  const int M = a.M;
  {
    // X -> LDS as MP rows of K elements, rows past M zero.
    const int per_row = K / 8;
    for (int i = threadIdx.x; i < MP * per_row; i += kWideThreads) {
      sku32x4 v = {0u, 0u, 0u, 0u};
      if (i / per_row < M) v = ((const sku32x4*)a.x)[i];
      ((sku32x4*)sk_lds)[i] = v;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int r = lane >> 3;  // row of the wave's group
  const int p = lane & 7;   // 16-byte piece of each line
  const unsigned char* xp = sk_lds + p * 16;
  for (int64_t g = (int64_t)blockIdx.x * WPB + (threadIdx.x >> 6); g < a.groups;
       g += (int64_t)gridDim.x * WPB) {
    int64_t first;
    const int which = sk_which(a.group_end, g, first);
    const int64_t N = a.n[which];
    const int64_t n = (g - first) * 8 + r;
    const sku32x4* wp = (const sku32x4*)((const T*)a.w[which] + (n < N ? n : N - 1) * (int64_t)K) + p;
    float acc[MP];
#pragma unroll
    for (int m = 0; m < MP; ++m) acc[m] = 0.f;
    auto consume = [&](const sku32x4& w, int line) {
      const V8 wv = __builtin_bit_cast(V8, w);
#pragma unroll
      for (int m = 0; m < MP; ++m)
        acc[m] = D::dot8(wv, *(const V8*)(xp + ((int64_t)m * K + line * 64) * 2), acc[m]);
    };
    // Scheduling barriers keep every load ahead of the products and the products
    // line by line: left free, the compiler reads X for all lines before the
    // first product and runs out of registers.
    if constexpr (LINES > 0) {
      sku32x4 w[LINES];
#pragma unroll
      for (int i = 0; i < LINES; ++i) w[i] = __builtin_nontemporal_load(wp + i * 8);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < LINES; ++i) {
        consume(w[i], i);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      const int lines = K / 64;
      for (int c0 = 0; c0 < lines; c0 += kWideGenericLines) {
        sku32x4 w[kWideGenericLines];
#pragma unroll
        for (int i = 0; i < kWideGenericLines; ++i)
          if (c0 + i < lines) w[i] = __builtin_nontemporal_load(wp + (c0 + i) * 8);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kWideGenericLines; ++i) {
          if (c0 + i < lines) consume(w[i], c0 + i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    float mine = 0.f;
#pragma unroll
    for (int m = 0; m < MP; ++m) {
      float v = acc[m];
      v += lane_xor1(v);
      v += lane_xor2(v);
      v += dpp_mov<0x141>(v);  // row_half_mirror: the other quad of the row's 8 lanes
      if (p == m) mine = v;
    }
    if (p < M && n < N) {
      const T* bp = (const T*)a.bias[which];
      const float bv = bp ? io<T>::to_f32(bp[n]) : 0.f;
      ((T*)a.y[which])[(int64_t)p * N + n] = io<T>::from_f32(mine + bv);
    }
  }
}

// The grid is sized to the workgroups that are resident at once, since the
// grid-stride loop gives every workgroup an equal share: per CU, the smaller of
// what the kernel's registers allow (looked up once per instantiation) and what
// its LDS (X, MP x K 16-bit elements, of the CU's 160 KiB) allows.
constexpr int64_t kCULds = 160 << 10;

template <typename T, int MP, int LINES>
int skinny_wide_launch(const SkArgs& a, hipStream_t s) {
  static std::atomic<int> by_regs{0};
  const size_t lds = (size_t)MP * a.K * 2;
  int n = by_regs.load(std::memory_order_relaxed);
  if (n == 0) {
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, skinny_wide_kernel<T, MP, LINES>, kWideThreads, 0);
    if (e != hipSuccess) return (int)e;
    if (n < 1) n = 1;
    by_regs.store(n, std::memory_order_relaxed);
  }
  const int64_t by_lds = kCULds / (int64_t)lds;
  const int64_t per_cu = by_lds < n ? (by_lds < 1 ? 1 : by_lds) : n;
  const int64_t needed = (a.groups + kWideThreads / 64 - 1) / (kWideThreads / 64);
  const int64_t cap = (int64_t)kSkCUs * per_cu;
  const int64_t blocks = needed < cap ? needed : cap;
  skinny_wide_kernel<T, MP, LINES><<<dim3((unsigned)blocks), dim3(kWideThreads), lds, s>>>(a);
  return launch_status();
}

template <typename T, int MP>
int skinny_wide_lines(const SkArgs& a, hipStream_t s) {
  switch (a.K / 64) {
    case 16: return skinny_wide_launch<T, MP, 16>(a, s);
    case 24: return skinny_wide_launch<T, MP, 24>(a, s);
    case 32: return skinny_wide_launch<T, MP, 32>(a, s);
    default: return skinny_wide_launch<T, MP, 0>(a, s);
  }
}

template <typename T, int SPLIT, int MODE>
int skinny_launch_split(const SkArgs& a, hipStream_t s) {
  constexpr int NT = SPLIT == 1 ? kSkThreads : 64 * SPLIT;
  constexpr int TPB = SPLIT == 1 ? kSkWaves : 1;
  const int64_t lds = a.M * sk_lds_row(a.K) * 2 + (SPLIT > 1 ? SPLIT * 64 * 4 * 4 : 0);
  const int64_t blocks_needed = (a.tiles + TPB - 1) / TPB;
  const int64_t cap = (int64_t)kSkCUs * kSkBlocksPerCU;
  const int64_t blocks = blocks_needed < cap ? blocks_needed : cap;
  skinny_nt_kernel<T, SPLIT, MODE><<<dim3((unsigned)blocks), dim3(NT), (size_t)lds, s>>>(a);
  return launch_status();
}

// Waves per tile: one while the tiles alone give the chip enough waves
// (kSkFillWaves); otherwise 4, 8 or 16 waves share each tile's K, as long as
// each keeps at least kSkMinSteps K steps and X plus the partial tiles (1 KB
// per wave) fit the workgroup's 64 KB of LDS.
constexpr int64_t kSkFillWaves = 2048;
constexpr int kSkMinSteps = 4;

template <typename T, int MODE = SK_PLAIN>
int skinny_launch(const SkArgs& a, hipStream_t s) {
  const int mp = a.M <= 1 ? 1 : a.M <= 2 ? 2 : a.M <= 4 ? 4 : 8;
  if (MODE == SK_PLAIN && a.M <= kWideMaxRows && a.K % 64 == 0 && a.groups >= kWideMinGroups &&
      (int64_t)mp * a.K * 2 <= kSkMaxLds) {
    switch (mp) {
      case 1: return skinny_wide_lines<T, 1>(a, s);
      case 2: return skinny_wide_lines<T, 2>(a, s);
      case 4: return skinny_wide_lines<T, 4>(a, s);
      default: return skinny_wide_lines<T, 8>(a, s);
    }
  }
  if (a.tiles >= kSkFillWaves) return skinny_launch_split<T, 1, MODE>(a, s);
  const int steps = a.K / kSkStep;
  const int64_t xlds = a.M * sk_lds_row(a.K) * 2;
  // The smallest split that gives the chip kSkFillWaves waves, or the largest
  // the constraints allow.
  int split = 1;
  for (int cand : {4, 8, 16}) {
    // (Sixteen waves leave 128 registers, too few for the conv's operands.)
    if (MODE != SK_PLAIN && cand == 16) break;
    if (steps < cand * kSkMinSteps || xlds + cand * 64 * 4 * 4 > kSkMaxLds) break;
    split = cand;
    if (a.tiles * cand >= kSkFillWaves) break;
  }
  switch (split) {
    case 16:
      if constexpr (MODE == SK_PLAIN) return skinny_launch_split<T, 16, MODE>(a, s);
      break;
    case 8: return skinny_launch_split<T, 8, MODE>(a, s);
    case 4: return skinny_launch_split<T, 4, MODE>(a, s);
    default: break;
  }
  return skinny_launch_split<T, 1, MODE>(a, s);
}

// Waves sharing a tile's K under SK_NORM_GATE (at most eight: its operands take 200 registers), 0 where the rows do not fit a lane's registers
// (kNormHeld quaternions of a row) or the workgroup's LDS (half a CU's).
constexpr int64_t kNormLds = 80 << 10;
int sk_norm_split(int64_t M, int64_t d_inner) {
  const int64_t K = 4 * d_inner;
  if (M < 1 || M > kSkMaxRows || K % kSkStep != 0) return 0;
  const int64_t xlds = M * sk_lds_row(K) * 2 + 128;  // (and the sums)
  for (int split : {8, 4}) {
    if (split > 4 && K / kSkStep < split * kSkMinSteps) continue;
    if (xlds + split * 64 * 4 * 4 > kNormLds) continue;
    int per = split;
    while (per > 1 && (split / per) * 2 <= M) per >>= 1;
    if (d_inner <= (int64_t)kNormHeld * 64 * per) return split;
  }
  return 0;
}

template <typename T, int SPLIT>
int sk_norm_launch(const SkArgs& a, hipStream_t s) {
  static std::atomic<bool> attr_set[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64) return MQC_E_LIMIT;
  if (!attr_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute((const void*)skinny_nt_kernel<T, SPLIT, SK_NORM_GATE>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, kNormLds);
    if (e != hipSuccess) return (int)e;
    attr_set[dev].store(true, std::memory_order_release);
  }
  return skinny_launch_split<T, SPLIT, SK_NORM_GATE>(a, s);
}

template <typename T>
int sk_norm_dispatch(const SkArgs& a, int split, hipStream_t s) {
  if (split == 8) return sk_norm_launch<T, 8>(a, s);
  return sk_norm_launch<T, 4>(a, s);
}

// The weights of one launch (slots past `count` repeat the last and hold no tiles).
void sk_weights(SkArgs& a, const void* X, int64_t M, int64_t K, int count, const void* const* w,
                const void* const* bias, void* const* y, const int64_t* n) {
  a.x = X;
  a.M = (int)M;
  a.K = (int)K;
  a.tiles = a.groups = 0;
  for (int i = 0; i < kSkMaxWeights; ++i) {
    const int j = i < count ? i : count - 1;
    a.w[i] = w[j];
    a.bias[i] = bias[j];
    a.y[i] = y[j];
    a.n[i] = n[j];
    if (i < count) {
      a.tiles += (n[j] + 15) / 16;
      a.groups += (n[j] + 7) / 8;
    }
    a.tile_end[i] = a.tiles;
    a.group_end[i] = a.groups;
  }
}

// What every product here needs of X and K.
int sk_check(const void* X, int64_t M, int64_t K) {
  if (K == 0 || M > kSkMaxRows || K % kSkStep != 0) return MQC_E_LIMIT;
  if (M * sk_lds_row(K) * 2 > kSkMaxLds || K >= ((int64_t)1 << 30)) return MQC_E_LIMIT;
  if (M > 0 && !X) return MQC_E_NULL;
  return aligned(X, 16) ? MQC_OK : MQC_E_ALIGN;
}

// The SSM of one decode step from the projections' outputs, in place on the state: delta and s
// from dt_raw, g_raw and x (rounded to T as the front's launch stores them), then one step of
// ssm_scan.hpp's delta-lambda walk. One lane per (d, k) and up to BR batch rows, whose Cayley
// constants it shares; a group of G lanes owns a d. Latency-bound: loads of all BR rows are issued
// before the first is used.
constexpr int kStepThreads = 256;
struct StepArgs {
  const void *dt, *g, *x;  // [batch, Dm]
  const void *B, *C;       // [batch, Dm, S, 4]
  const float *lam_alpha, *lam_imag, *dvec;
  float* h;                // [batch, Dm, S, 4]
  void* y;                 // [batch, Dm, 4]
  int batch, Dm, S;
  float eps;
};

template <typename T, int G, int BR>
__global__ __launch_bounds__(kStepThreads) void ssm_step_kernel(StepArgs a) {
  const int lane = threadIdx.x & 63;
  const int j = threadIdx.x & (G - 1);
  const int d_raw = (int)blockIdx.x * (kStepThreads / G) + (int)threadIdx.x / G;
  const bool gvalid = d_raw < a.Dm, kvalid = j < a.S;
  const int d = gvalid ? d_raw : a.Dm - 1;
  const int k = kvalid ? j : a.S - 1;
  const int b0 = (int)blockIdx.y * BR;
  const int64_t dk = (int64_t)d * a.S + k;
  float4 h[BR];
  uint2 Bw[BR], Cw[BR];
  T dt[BR], gr[BR], xr[BR];
#pragma unroll
  for (int i = 0; i < BR; ++i) {
    // (Rows past the batch read the last one's, and store nothing.)
    const int64_t b = b0 + i < a.batch ? b0 + i : a.batch - 1;
    const int64_t e = b * a.Dm * a.S + dk;
    h[i] = ((const float4*)a.h)[e];
    Bw[i] = ((const uint2*)a.B)[e];
    Cw[i] = ((const uint2*)a.C)[e];
    dt[i] = ((const T*)a.dt)[b * a.Dm + d];
    gr[i] = ((const T*)a.g)[b * a.Dm + d];
    xr[i] = ((const T*)a.x)[b * a.Dm + d];
  }
  const LamConst L = lam_const(a.lam_alpha, a.lam_imag, dk);
  const float dskip = a.dvec[d];
  auto quat16 = [](const uint2& w) {
    float e[4];
    if constexpr (std::is_same<T, bf16_t>::value) {
      e[0] = __uint_as_float(w.x << 16); e[1] = __uint_as_float(w.x & 0xffff0000u);
      e[2] = __uint_as_float(w.y << 16); e[3] = __uint_as_float(w.y & 0xffff0000u);
    } else {
      e[0] = io<T>::bits_to_f32(w.x & 0xffffu); e[1] = io<T>::bits_to_f32(w.x >> 16);
      e[2] = io<T>::bits_to_f32(w.y & 0xffffu); e[3] = io<T>::bits_to_f32(w.y >> 16);
    }
    return quat{e[0], e[1], e[2], e[3]};
  };
#pragma unroll
  for (int i = 0; i < BR; ++i) {
    const int b = b0 + i;
    const float dl = io<T>::to_f32(io<T>::from_f32(front_softplus(io<T>::to_f32(dt[i]))));
    const float sv = io<T>::to_f32(
        io<T>::from_f32(front_sigmoid(io<T>::to_f32(gr[i])) * io<T>::to_f32(xr[i])));
    const quat q = cayley_step(dl, dl * dl, L, a.eps);
    const quat hn = state_step(q, quat{h[i].x, h[i].y, h[i].z, h[i].w}, sv, quat16(Bw[i]));
    quat acc{0.f, 0.f, 0.f, 0.f};
    qmul_acc(acc, quat16(Cw[i]), hn);
    if (!kvalid) acc = quat{0.f, 0.f, 0.f, 0.f};
    float v[4];
    int c0;
    const int nc = group_reduce<G>(acc, lane, v, c0);
    if (b < a.batch && gvalid) {
      if (kvalid)
        ((float4*)a.h)[(int64_t)b * a.Dm * a.S + dk] = float4{hn.w, hn.x, hn.y, hn.z};
      if (G < 4 || j < 4) {
        if (c0 == 0) v[0] = fmaf(dskip, sv, v[0]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < nc) ((T*)a.y)[((int64_t)b * a.Dm + d) * 4 + c0 + e] = io<T>::from_f32(v[e]);
      }
    }
  }
}

template <typename T, int G>
int ssm_step_launch_g(const StepArgs& a, hipStream_t s) {
  constexpr int GPB = kStepThreads / G;
  const dim3 one((unsigned)((a.Dm + GPB - 1) / GPB), 1);
  if (a.batch == 1) {
    ssm_step_kernel<T, G, 1><<<one, dim3(kStepThreads), 0, s>>>(a);
  } else if (a.batch == 2) {
    ssm_step_kernel<T, G, 2><<<one, dim3(kStepThreads), 0, s>>>(a);
  } else {
    ssm_step_kernel<T, G, 4><<<dim3(one.x, (unsigned)((a.batch + 3) / 4)), dim3(kStepThreads), 0, s>>>(a);
  }
  return launch_status();
}

template <typename T>
int ssm_step_launch(const StepArgs& a, hipStream_t s) {
  if (a.S <= 1) return ssm_step_launch_g<T, 1>(a, s);
  if (a.S <= 2) return ssm_step_launch_g<T, 2>(a, s);
  if (a.S <= 4) return ssm_step_launch_g<T, 4>(a, s);
  if (a.S <= 8) return ssm_step_launch_g<T, 8>(a, s);
  if (a.S <= 16) return ssm_step_launch_g<T, 16>(a, s);
  if (a.S <= 32) return ssm_step_launch_g<T, 32>(a, s);
  return ssm_step_launch_g<T, 64>(a, s);
}

}  // namespace
}  // namespace mqc

using namespace mqc;

extern "C" {

int mqc_gemm_skinny4_nt(const void* X, int64_t M, int64_t K, const void* W1, const void* bias1,
                        void* Y1, int64_t N1, const void* W2, const void* bias2, void* Y2,
                        int64_t N2, const void* W3, const void* bias3, void* Y3, int64_t N3,
                        const void* W4, const void* bias4, void* Y4, int64_t N4, int dtype,
                        void* stream) {
  if (M < 0 || K < 0) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  if (M == 0) return MQC_OK;
  const int st = sk_check(X, M, K);
  if (st != MQC_OK) return st;
  const void* w[4] = {W1, W2, W3, W4};
  const void* bias[4] = {bias1, bias2, bias3, bias4};
  void* y[4] = {Y1, Y2, Y3, Y4};
  const int64_t n[4] = {N1, N2, N3, N4};
  for (int i = 0; i < 4; ++i) {
    if (n[i] < 1) return MQC_E_SHAPE;
    if (!w[i] || !y[i]) return MQC_E_NULL;
    if (!aligned(w[i], 16) || !aligned(y[i], 2) || !aligned(bias[i], 2)) return MQC_E_ALIGN;
  }
  SkArgs a{};
  sk_weights(a, X, M, K, 4, w, bias, y, n);
  if (dtype == MQC_BF16) return skinny_launch<bf16_t>(a, (hipStream_t)stream);
  return skinny_launch<f16_t>(a, (hipStream_t)stream);
}

int mqc_step_in_proj_conv(const void* X, int64_t M, int64_t K, const void* W, const void* bias,
                          int64_t channels, int64_t z_cols, const float* conv_w,
                          const float* conv_b, int64_t conv_k, void* tail, void* act, void* z,
                          int dtype, void* stream) {
  if (M < 0 || K < 0 || channels < 1 || z_cols < 1 || conv_k < 1) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  if (M == 0) return MQC_OK;
  if (conv_k > kSkMaxTaps || channels % 8 != 0 || channels + z_cols > (1LL << 30)) return MQC_E_LIMIT;
  const int st = sk_check(X, M, K);
  if (st != MQC_OK) return st;
  if (!W || !conv_w || (conv_k > 1 && !tail) || !act || !z) return MQC_E_NULL;
  if (!aligned(W, 16) || !aligned(bias, 2) || !aligned(conv_w, 4) || !aligned(conv_b, 4) ||
      !aligned(tail, 2) || !aligned(act, 2) || !aligned(z, 2))
    return MQC_E_ALIGN;
  SkArgs a{};
  const int64_t n = channels + z_cols;
  sk_weights(a, X, M, K, 1, &W, &bias, &z, &n);
  a.conv_w = conv_w; a.conv_b = conv_b; a.tail = tail; a.act = act;
  a.conv_ch = (int)channels; a.conv_k = (int)conv_k;
  if (dtype == MQC_BF16) return skinny_launch<bf16_t, SK_CONV>(a, (hipStream_t)stream);
  return skinny_launch<f16_t, SK_CONV>(a, (hipStream_t)stream);
}

int mqc_step_norm_out_gate(const void* Y, int64_t M, int64_t d_inner, const float* gamma,
                           const float* beta, float eps, const void* W, const void* bias,
                           int64_t d_model, const void* x, const void* z, int64_t z_row_stride,
                           void* out, int dtype, void* stream) {
  if (M < 0 || d_inner < 1 || d_model < 1 || z_row_stride < d_model) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  if (M == 0) return MQC_OK;
  const int split = sk_norm_split(M, d_inner);
  if (split == 0) return MQC_E_LIMIT;
  if (!Y || !gamma || !beta || !W || !x || !z || !out) return MQC_E_NULL;
  if (!aligned(Y, 16)) return MQC_E_ALIGN;
  if (!aligned(W, 16) || !aligned(bias, 2) || !aligned(gamma, 4) || !aligned(beta, 16) ||
      !aligned(x, 2) || !aligned(z, 2) || !aligned(out, 2))
    return MQC_E_ALIGN;
  SkArgs a{};
  sk_weights(a, Y, M, 4 * d_inner, 1, &W, &bias, &out, &d_model);
  a.gamma = gamma; a.beta = beta; a.res = x; a.z = z; a.zs = z_row_stride; a.eps = eps;
  if (dtype == MQC_BF16) return sk_norm_dispatch<bf16_t>(a, split, (hipStream_t)stream);
  return sk_norm_dispatch<f16_t>(a, split, (hipStream_t)stream);
}

int mqc_step_norm_out_gate_fits(int64_t M, int64_t d_inner) {
  return M > 0 && d_inner > 0 && sk_norm_split(M, d_inner) > 0;
}

int mqc_step_ssm(const void* dt_raw, const void* g_raw, const void* x, const void* B,
                 const void* C, const float* lambda_alpha, const float* lambda_imag,
                 const float* D, float* h, void* y, int64_t batch, int64_t d_inner,
                 int64_t d_state, float eps, int dtype, void* stream) {
  if (batch < 0 || d_inner < 0 || d_state < 0) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  if (batch == 0 || d_inner == 0) return MQC_OK;
  if (d_state < 1 || d_state > 64 || d_inner > (1 << 24) || batch > 4 * 65535) return MQC_E_LIMIT;
  if (!dt_raw || !g_raw || !x || !B || !C || !lambda_alpha || !lambda_imag || !D || !h || !y)
    return MQC_E_NULL;
  if (!aligned(dt_raw, 2) || !aligned(g_raw, 2) || !aligned(x, 2) || !aligned(B, 8) ||
      !aligned(C, 8) || !aligned(h, 16) || !aligned(y, 2))
    return MQC_E_ALIGN;
  StepArgs a{dt_raw, g_raw, x, B, C, lambda_alpha, lambda_imag, D, h, y,
             (int)batch, (int)d_inner, (int)d_state, eps};
  if (dtype == MQC_BF16) return ssm_step_launch<bf16_t>(a, (hipStream_t)stream);
  return ssm_step_launch<f16_t>(a, (hipStream_t)stream);
}

}  // extern "C"

extern "C" int mqc_gemm_skinny_nt(const void* X, int64_t M, int64_t K, const void* W1,
                                  const void* bias1, void* Y1, int64_t N1, const void* W2,
                                  const void* bias2, void* Y2, int64_t N2, int dtype,
                                  void* stream) {
  if (M < 0 || K < 0 || N1 < 0 || N2 < 0) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  // K == 0 (an empty reduction) is left to the caller.
  if (M > kSkMaxRows || K == 0 || K % kSkStep != 0) return MQC_E_LIMIT;
  if (M * sk_lds_row(K) * 2 > kSkMaxLds || K >= ((int64_t)1 << 30)) return MQC_E_LIMIT;
  const bool pair = N2 > 0;
  if (M == 0 || (N1 == 0 && !pair)) return MQC_OK;
  if (!X || (N1 > 0 && (!W1 || !Y1)) || (pair && (!W2 || !Y2))) return MQC_E_NULL;
  if (!aligned(X, 16) || (N1 > 0 && (!aligned(W1, 16) || !aligned(Y1, 2))) ||
      (pair && (!aligned(W2, 16) || !aligned(Y2, 2))) || !aligned(bias1, 2) ||
      !aligned(bias2, 2))
    return MQC_E_ALIGN;
  SkArgs a{};
  const void* w[2] = {W1, W2};
  const void* bias[2] = {bias1, bias2};
  void* y[2] = {Y1, Y2};
  const int64_t n[2] = {N1, N2};
  sk_weights(a, X, M, K, pair ? 2 : 1, w, bias, y, n);
  if (dtype == MQC_BF16) return skinny_launch<bf16_t>(a, (hipStream_t)stream);
  return skinny_launch<f16_t>(a, (hipStream_t)stream);
}
