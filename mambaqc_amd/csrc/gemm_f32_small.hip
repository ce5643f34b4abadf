// Small fp32 products, several in one launch:
//   Y_i[m, n] = sum_k X_i(m, k) W_i(n, k) (+ bias_i[n]),  i < 4,
// on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32: fp32 products and sums, as hipBLASLt's
// fp32), for the projections of small fp32 blocks (F.linear,
// mambaqc/layers/quaternion_linear.py:145-172, and the block's nn.Linear layers,
// models/quaternion_mamba2_block.py:78-122).
//
// These products take less time on the GPU (3-10 us) than torch's dispatch of one hipBLASLt
// fp32 GEMM takes on the host (21 us), so a small block is bound by the host: one launch here
// carries up to four of them (dt, gate, B and C share their input).
//
//   - Workgroups of 4 waves own T x T tiles of one product (T 64, or 32 where the launch's 64-wide tiles
//     would leave most CUs idle); operands are strided views with k or the row index contiguous.
//   - K in steps of 32 through LDS as [k][row] (row pitch T + 20 words: neither the transposing
//     writes nor a fragment's 4 k x 16 rows take more than two words of a bank), the next step's
//     loads in registers while this one is multiplied.
//   - Latency-bound: at most a few tiles per CU and K steps in a chain. B1 T64 d_model 64, 16
//     states: the four projections of x_act in one launch 13 us, where the four hipBLASLt calls
//     took 27 us of GPU and 86 us of host time (whole block 264 -> 163 us).
#include "mfma_tile.hpp"

namespace mqc {
namespace {

using mfma::floatx4;

constexpr int kSmMax = 4;      // products per launch
constexpr int kSmBK = 32;
constexpr int kSmThreads = 256;

struct SmProduct {
  const float* X;
  const float* W;
  const float* bias;  // [N] or null
  float* Y;           // [M, N] dense
  int64_t xm, xk, wn, wk;
  int M, N, K;
  int tile0;          // first tile of this product in the launch
};
struct SmArgs {
  SmProduct p[kSmMax];
  int count;
};

// Four elements of an operand tile: rows r.. (or k..) in memory order, zero outside.
// KC: k contiguous (four k of one row), else four rows of one k.
template <bool KC>
__device__ inline floatx4 sm_load(const float* A, int64_t sr, int64_t sk, int r, int k, int R, int K,
                                  bool vec) {
  floatx4 v = {0.f, 0.f, 0.f, 0.f};
  const float* p = A + (int64_t)r * sr + (int64_t)k * sk;
  if (KC ? r < R : k < K) {
    const int left = KC ? K - k : R - r;
    if (vec && left >= 4) {
      v = *(const floatx4*)p;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < left) v[i] = p[i];
    }
  }
  return v;
}

template <int T>
__global__ __launch_bounds__(kSmThreads) void gemm_f32_small_kernel(SmArgs a) {
  constexpr int P = T + 20;               // LDS row pitch
  constexpr int L = T * kSmBK / 4 / kSmThreads;  // 16-byte loads per thread, operand and step
  constexpr int B = T / 32;               // 16-row blocks per wave and operand
  __shared__ float xs[kSmBK * P], ws[kSmBK * P];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int which = 0;
#pragma unroll
  for (int i = 1; i < kSmMax; ++i)
    if (i < a.count && (int)blockIdx.x >= a.p[i].tile0) which = i;
  const SmProduct p = a.p[__builtin_amdgcn_readfirstlane(which)];
  const int tile = (int)blockIdx.x - p.tile0;
  const int mt = (p.M + T - 1) / T;
  const int m0 = tile % mt * T, n0 = tile / mt * T;
  const bool xc = p.xk == 1, wc = p.wk == 1;
  const bool xv = ((xc ? p.xm : p.xk) & 3) == 0 && ((uintptr_t)p.X & 15) == 0;
  const bool wv = ((wc ? p.wn : p.wk) & 3) == 0 && ((uintptr_t)p.W & 15) == 0;
  floatx4 xr[L], wr[L];
  // Thread's piece i of a step: with k contiguous row q / 8, k 4 (q % 8); else k q / (T / 4),
  // rows 4 (q % (T / 4)).
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int q = i * kSmThreads + tid;
      const int rc = q >> 3, kc = (q & 7) * 4, rr = (q % (T / 4)) * 4, kr = q / (T / 4);
      xr[i] = xc ? sm_load<true>(p.X, p.xm, p.xk, m0 + rc, k0 + kc, p.M, p.K, xv)
                 : sm_load<false>(p.X, p.xm, p.xk, m0 + rr, k0 + kr, p.M, p.K, xv);
      wr[i] = wc ? sm_load<true>(p.W, p.wn, p.wk, n0 + rc, k0 + kc, p.N, p.K, wv)
                 : sm_load<false>(p.W, p.wn, p.wk, n0 + rr, k0 + kr, p.N, p.K, wv);
    }
  };
  auto put = [&](float* t, const floatx4& v, bool kc_, int q) {
    if (kc_) {
#pragma unroll
      for (int i = 0; i < 4; ++i) t[((q & 7) * 4 + i) * P + (q >> 3)] = v[i];
    } else {
      *(floatx4*)(t + (q / (T / 4)) * P + (q % (T / 4)) * 4) = v;
    }
  };
  const int rl = lane & 15, kq = lane >> 4;
  const int wb = (wave >> 1) * (T / 2) + rl, xb = (wave & 1) * (T / 2) + rl;
  floatx4 acc[B][B];
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  for (int k0 = 0; k0 < p.K; k0 += kSmBK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < L; ++i) {
      put(xs, xr[i], xc, i * kSmThreads + tid);
      put(ws, wr[i], wc, i * kSmThreads + tid);
    }
    __syncthreads();
    if (k0 + kSmBK < p.K) fetch(k0 + kSmBK);
#pragma unroll
    for (int s = 0; s < kSmBK / 4; ++s) {
      float wf[B], xf[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        wf[i] = ws[(4 * s + kq) * P + wb + 16 * i];
        xf[i] = xs[(4 * s + kq) * P + xb + 16 * i];
      }
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
  }
  // Lane: 4 consecutive n of one m per block.
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const int n = n0 + (wave >> 1) * (T / 2) + 16 * i + 4 * kq;
    float b[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = p.bias && n + e < p.N ? p.bias[n + e] : 0.f;
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int m = m0 + xb + 16 * j;
      if (m >= p.M) continue;
      float* y = p.Y + (int64_t)m * p.N + n;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < p.N) y[e] = acc[i][j][e] + b[e];
    }
  }
}

}  // namespace
}  // namespace mqc

using namespace mqc;

extern "C" int mqc_gemm_f32_small(const int64_t* products, int64_t count, void* stream) {
  if (count < 0 || count > kSmMax) return MQC_E_LIMIT;
  if (count == 0) return MQC_OK;
  if (!products) return MQC_E_NULL;
  SmArgs a{};
  a.count = (int)count;
  int64_t t64 = 0, t32 = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t* f = products + 11 * i;
    SmProduct& p = a.p[i];
    p.X = (const float*)f[0]; p.xm = f[1]; p.xk = f[2];
    p.W = (const float*)f[3]; p.wn = f[4]; p.wk = f[5];
    p.bias = (const float*)f[6];
    p.Y = (float*)f[7];
    const int64_t M = f[8], N = f[9], K = f[10];
    if (M < 1 || N < 1 || K < 1 || p.xm < 0 || p.xk < 0 || p.wn < 0 || p.wk < 0 ||
        (p.xm != 1 && p.xk != 1) || (p.wn != 1 && p.wk != 1))
      return MQC_E_SHAPE;
    if (M > (1 << 24) || N > (1 << 24) || K > (1 << 24)) return MQC_E_LIMIT;
    if (!p.X || !p.W || !p.Y) return MQC_E_NULL;
    if (!aligned(p.X, 4) || !aligned(p.W, 4) || !aligned(p.Y, 4) || !aligned(p.bias, 4))
      return MQC_E_ALIGN;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    t64 += (M + 63) / 64 * ((N + 63) / 64);
    t32 += (M + 31) / 32 * ((N + 31) / 32);
  }
  if (t32 > 0x7fffffffLL) return MQC_E_LIMIT;
  // 32-wide tiles below one 64-wide tile per CU.
  const bool big = t64 >= 256;
  int tile0 = 0;
  for (int i = 0; i < count; ++i) {
    a.p[i].tile0 = tile0;
    const int t = big ? 64 : 32;
    tile0 += (a.p[i].M + t - 1) / t * ((a.p[i].N + t - 1) / t);
  }
  if (big)
    gemm_f32_small_kernel<64><<<dim3((unsigned)tile0), dim3(kSmThreads), 0, (hipStream_t)stream>>>(a);
  else
    gemm_f32_small_kernel<32><<<dim3((unsigned)tile0), dim3(kSmThreads), 0, (hipStream_t)stream>>>(a);
  return launch_status();
}
