// Time-chunked forms of the two recurrences on a materialised q, for calls with too few lanes to
// fill the GPU: the cumulative Hamilton product (cumprod_scan.hip;
// mambaqc/kernels/parallel_scan.py:267-295) and the SSM's q form (ssm_scan.hpp, MODE_Q;
// mambaqc/kernels/ssm_fused.py:340-401).
//
// A lane's steps are one serial chain (0.2-0.4 us a step), so 4096 steps of 8192 states take over a
// millisecond while HBM could feed them in 0.3. The T axis is cut into chunks walked side by side:
//   1. every chunk but the last from the identity (and, for the SSM, from a zero state): the
//      product P of its q's and its end state H;
//   2. the carries, per lane over its chunks in order, the later factor on the left:
//      E_c = P_c (x) E_{c-1} (+ H_c);
//   3. the usual kernels on every chunk from its carry.
//
// P is held as a quaternion of magnitude about 1 times 2^X: a chunk of decaying (or growing) q's
// takes it far past fp32's range, where the carried value itself may be anywhere. What fp32 could
// not hold on the way, the walk itself would not have held either, or it is marked, and the prefix
// walks those lanes' chunks step by step from their carry: a q so small or large that P leaves the
// range within 8 steps, an inf or a NaN, and products that could overflow with the carry at hand.
// (The bookkeeping costs at most 7 us: cumulative product, T 4096, bf16 1024 lanes 36 without and
// 44 with it, fp32 4096 lanes 138 and 146, the SSM's q form within its noise.) Launch 1 reads q
// (and B) a second time, so it pays only where the chain, not HBM, is the bound: the rules are with
// the callers (kernels/parallel_scan.py, kernels/ssm_fused.py), both sides measured.
#include "ssm_scan.hpp"

namespace mqc {
namespace {

// A chunk's exponents: P is its stored value times 2^x, and no step's product was above 2^top.
// kWalk: the chunk has to be walked from its carry.
struct ChunkExp {
  int x, top;
};
constexpr int kWalk = 1 << 30;
constexpr int kTopExp = 120;             // exponents of carry and product together stay below this
constexpr float kLeast = 0x1p-100f;      // P keeps its precision from one renormalisation to the next
constexpr float kMost = 0x1p120f;

__device__ inline float top_of(const quat& p) {
  return fmaxf(fmaxf(fabsf(p.w), fabsf(p.x)), fmaxf(fabsf(p.y), fabsf(p.z)));
}
__device__ inline bool finite4(const quat& p) {
  return p.w * 0.f + p.x * 0.f + p.y * 0.f + p.z * 0.f == 0.f;
}

template <typename T>
struct QArgs {
  const T* q;   // [batch, T_len, lanes, 4]
  const T* Bm;  // the same (SSM)
  const T* Sq;  // [batch, T_len, lanes / S, 4] (SSM)
  int64_t batch, T_len, lanes, S, L, nc;
};

// The steps of chunk c of lane l, PF loads ahead: step(i, q) or step(i, q, b, s) in order, and
// group() after every PF of them.
template <typename T, bool SSM, typename Step, typename Group>
__device__ inline void q_chunk_steps(const QArgs<T>& a, int64_t b, int64_t c, int64_t l,
                                     const Step& step, const Group& group) {
  constexpr int PF = 8;
  const int64_t row = a.lanes * 4;
  const int64_t base = (b * a.T_len + c * a.L) * row + l * 4;  // (every chunk here is whole)
  const int64_t d = SSM ? l / a.S : 0, D = SSM ? a.lanes / a.S : 0;
  const T* sp = SSM ? a.Sq + ((b * a.T_len + c * a.L) * D + d) * 4 : nullptr;
  for (int64_t t0 = 0; t0 < a.L; t0 += PF) {
    float qv[PF][4], bv[SSM ? PF : 1][4], sv[SSM ? PF : 1][4];
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int64_t t = t0 + i < a.L ? t0 + i : a.L - 1;
      load_vec<T, 4>(a.q + base + t * row, qv[i]);
      if constexpr (SSM) {
        load_vec<T, 4>(a.Bm + base + t * row, bv[i]);
        load_vec<T, 4>(sp + t * D * 4, sv[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      if (t0 + i < a.L) {
        if constexpr (SSM)
          step(quat_from(qv[i]), quat_from(bv[i]), quat_from(sv[i]));
        else
          step(quat_from(qv[i]), quat{}, quat{});
      }
    }
    group();
  }
}

// 1. One thread per (chunk, b, lane); the next PF steps' loads are in flight.
template <typename T, bool SSM>
__global__ __launch_bounds__(256) void q_chunk_agg_kernel(QArgs<T> a, float* __restrict__ Hc,
                                                          float* __restrict__ Pc,
                                                          ChunkExp* __restrict__ Xc) {
  const int64_t l = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t b = blockIdx.y % a.batch, c = blockIdx.y / a.batch;
  if (l >= a.lanes) return;
  quat P{1.f, 0.f, 0.f, 0.f}, H{0.f, 0.f, 0.f, 0.f};
  int x = 0, top = 0;
  float m = 1.f, most = 0.f, mostH = 0.f;  // of P now, in this group; of H
  bool walk = false;
  q_chunk_steps<T, SSM>(
      a, b, c, l,
      [&](const quat& qq, const quat& Bq, const quat& Sv) {
        P = qmul(qq, P);
        // (A q of zero, and what follows it, makes an exact zero.)
        const float before = m;
        m = top_of(P);
        walk |= m < kLeast && before >= kLeast && top_of(qq) > 0.f;
        most = fmaxf(most, m);
        if constexpr (SSM) {
          quat hn = qmul(Bq, Sv);
          qmul_acc(hn, qq, H);
          H = hn;
          mostH = fmaxf(mostH, top_of(H));
        }
      },
      [&]() {
        // A power of two out of P; the largest on the way.
        walk |= !(most < kMost);
        const int g = most > 0.f && most < kMost ? __builtin_amdgcn_frexp_expf(most) : 0;
        top = x + g > top ? x + g : top;
        const int e = m > 0.f && m < kMost ? __builtin_amdgcn_frexp_expf(m) : 0;
        P.w = __builtin_amdgcn_ldexpf(P.w, -e);
        P.x = __builtin_amdgcn_ldexpf(P.x, -e);
        P.y = __builtin_amdgcn_ldexpf(P.y, -e);
        P.z = __builtin_amdgcn_ldexpf(P.z, -e);
        x += e;
        m = __builtin_amdgcn_ldexpf(m, -e);
        most = 0.f;
      });
  walk |= !finite4(P);
  if constexpr (SSM) walk |= !finite4(H) || !(mostH < kMost);
  const int64_t o = (b * a.nc + c) * a.lanes + l;
  const float e[4] = {P.w, P.x, P.y, P.z};
  store_vec<float, 4>(Pc + o * 4, e);
  Xc[o] = ChunkExp{x, walk ? kWalk : top};
  if constexpr (SSM) {
    const float h[4] = {H.w, H.x, H.y, H.z};
    store_vec<float, 4>(Hc + o * 4, h);
  }
}

// 2. One thread per (b, lane): the carries in place, in Pc (products) or Hc (states).
template <typename T, bool SSM>
__global__ __launch_bounds__(256) void q_chunk_prefix_kernel(QArgs<T> a, float* __restrict__ Hc,
                                                             float* __restrict__ Pc,
                                                             const ChunkExp* __restrict__ Xc) {
  constexpr int PF = 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.batch * a.lanes) return;
  const int64_t b = i / a.lanes, l = i - b * a.lanes;
  const int64_t o = b * a.nc * a.lanes + l;
  float* out = SSM ? Hc : Pc;
  quat E{SSM ? 0.f : 1.f, 0.f, 0.f, 0.f};
  for (int64_t c0 = 0; c0 < a.nc; c0 += PF) {
    float p[PF][4], h[SSM ? PF : 1][4];
    ChunkExp xs[PF];
#pragma unroll
    for (int k = 0; k < PF; ++k) {
      const int64_t at = o + (c0 + k < a.nc ? c0 + k : a.nc - 1) * a.lanes;
      load_vec<float, 4>(Pc + at * 4, p[k]);
      if constexpr (SSM) load_vec<float, 4>(Hc + at * 4, h[k]);
      xs[k] = Xc[at];
    }
    const quat E0 = E;
    bool walk = false;
#pragma unroll
    for (int k = 0; k < PF; ++k) {
      if (c0 + k < a.nc) {
        const float t = top_of(E);
        const bool nan = E.w != E.w && E.x != E.x && E.y != E.y && E.z != E.z;  // (and stays)
        walk |= !nan && (xs[k].top == kWalk || !finite4(E) ||
                         (t > 0.f && __builtin_amdgcn_frexp_expf(t) + xs[k].top > kTopExp));
        quat n = qmul(quat_from(p[k]), E);
        n.w = __builtin_amdgcn_ldexpf(n.w, xs[k].x);
        n.x = __builtin_amdgcn_ldexpf(n.x, xs[k].x);
        n.y = __builtin_amdgcn_ldexpf(n.y, xs[k].x);
        n.z = __builtin_amdgcn_ldexpf(n.z, xs[k].x);
        if constexpr (SSM) {
          n.w += h[k][0]; n.x += h[k][1]; n.y += h[k][2]; n.z += h[k][3];
        }
        E = n;
        const float e[4] = {E.w, E.x, E.y, E.z};
        store_vec<float, 4>(out + (o + (c0 + k) * a.lanes) * 4, e);
      }
    }
    if (walk) {
      // These chunks again, every step from the carry.
      E = E0;
      const int64_t end = c0 + PF < a.nc ? c0 + PF : a.nc;
#pragma unroll 1
      for (int64_t c = c0; c < end; ++c) {
        q_chunk_steps<T, SSM>(
            a, b, c, l,
            [&](const quat& qq, const quat& Bq, const quat& Sv) {
              if constexpr (SSM) {
                quat hn = qmul(Bq, Sv);
                qmul_acc(hn, qq, E);
                E = hn;
              } else {
                E = qmul(qq, E);
              }
            },
            [] {});
        const float e[4] = {E.w, E.x, E.y, E.z};
        store_vec<float, 4>(out + (o + c * a.lanes) * 4, e);
      }
    }
  }
}

// 3 (product). One thread per (chunk, b, lane) from its carry.
template <typename T>
__global__ __launch_bounds__(256) void cumprod_chunk_kernel(const T* __restrict__ q, T* __restrict__ out,
                                                            const float* __restrict__ Pc,
                                                            int64_t batch, int64_t T_len,
                                                            int64_t lanes, int64_t L, int64_t nc) {
  constexpr int PF = 8;
  const int64_t l = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t b = blockIdx.y % batch, c = blockIdx.y / batch;
  if (l >= lanes) return;
  const int64_t row = lanes * 4;
  const int64_t base = (b * T_len + c * L) * row + l * 4;
  const int64_t n = T_len - c * L < L ? T_len - c * L : L;
  quat E{1.f, 0.f, 0.f, 0.f};
  if (c > 0) {
    float e[4];
    load_vec<float, 4>(Pc + ((b * nc + c - 1) * lanes + l) * 4, e);
    E = quat_from(e);
  }
  for (int64_t t0 = 0; t0 < n; t0 += PF) {
    float qv[PF][4];
#pragma unroll
    for (int i = 0; i < PF; ++i) load_vec<T, 4>(q + base + (t0 + i < n ? t0 + i : n - 1) * row, qv[i]);
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      if (t0 + i < n) {
        E = qmul(quat_from(qv[i]), E);
        const float e[4] = {E.w, E.x, E.y, E.z};
        store_vec<T, 4, true>(out + base + (t0 + i) * row, e);
      }
    }
  }
}

template <typename T>
int launch_cumprod_chunked(const void* q, void* out, int64_t batch, int64_t T_len, int64_t lanes,
                           int64_t L, int64_t nc, float* ws, hipStream_t s) {
  if (!aligned(q, 4 * sizeof(T)) || !aligned(out, 4 * sizeof(T))) return MQC_E_ALIGN;
  const unsigned gx = (unsigned)((lanes + 255) / 256);
  const QArgs<T> a{(const T*)q, nullptr, nullptr, batch, T_len, lanes, 1, L, nc};
  ChunkExp* xs = (ChunkExp*)(ws + batch * nc * lanes * 4);
  q_chunk_agg_kernel<T, false>
      <<<dim3(gx, (unsigned)(batch * nc)), 256, 0, s>>>(a, nullptr, ws, xs);
  q_chunk_prefix_kernel<T, false>
      <<<dim3((unsigned)((batch * lanes + 255) / 256)), 256, 0, s>>>(a, nullptr, ws, xs);
  cumprod_chunk_kernel<T><<<dim3(gx, (unsigned)(batch * (nc + 1))), 256, 0, s>>>(
      (const T*)q, (T*)out, ws, batch, T_len, lanes, L, nc);
  return launch_status();
}

template <typename T>
int launch_ssm_q_chunked(SsmArgs a, int64_t nc, float* ws, hipStream_t s) {
  const int chk = ssm_check<T, MODE_Q>(a);
  if (chk != MQC_OK) return chk;
  const int64_t lanes = a.Dm * a.S;
  float* Hc = ws;
  float* Pc = ws + a.batch * nc * lanes * 4;
  ChunkExp* xs = (ChunkExp*)(Pc + a.batch * nc * lanes * 4);
  const QArgs<T> qa{(const T*)a.q, (const T*)a.Bm, (const T*)a.Sq, a.batch, a.T, lanes, a.S,
                    a.chunk_len, nc};
  q_chunk_agg_kernel<T, true>
      <<<dim3((unsigned)((lanes + 255) / 256), (unsigned)(a.batch * nc)), 256, 0, s>>>(qa, Hc, Pc, xs);
  q_chunk_prefix_kernel<T, true>
      <<<dim3((unsigned)((a.batch * lanes + 255) / 256)), 256, 0, s>>>(qa, Hc, Pc, xs);
  const int st = launch_status();
  if (st != MQC_OK) return st;
  a.h_chunk = Hc;
  return launch_ssm<T, MODE_Q>(a, s);
}

// Chunks with a carry (all but the last), 0 where one chunk holds the sequence.
int64_t carries(int64_t T_len, int64_t L) { return L < 1 || L >= T_len ? 0 : (T_len + L - 1) / L - 1; }

}  // namespace
}  // namespace mqc

using namespace mqc;

extern "C" {

int64_t mqc_q_chunked_workspace_bytes(int64_t batch, int64_t seq_len, int64_t lanes,
                                      int64_t chunk_len, int ssm) {
  if (batch < 0 || seq_len < 0 || lanes < 0 || chunk_len < 1) return MQC_E_SHAPE;
  return batch * carries(seq_len, chunk_len) * lanes *
         ((ssm ? 2 : 1) * 4 * (int64_t)sizeof(float) + (int64_t)sizeof(ChunkExp));
}

int mqc_cumprod_scan_chunked(const void* q, void* out, int64_t batch, int64_t seq_len,
                             int64_t lanes, int64_t chunk_len, int dtype, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  if (batch < 1 || seq_len < 1 || lanes < 1 || chunk_len < 1) return MQC_E_SHAPE;
  const int64_t nc = carries(seq_len, chunk_len);
  if (nc < 1) return MQC_E_SHAPE;
  if (!q || !out || !workspace) return MQC_E_NULL;
  if (!aligned(workspace, 16)) return MQC_E_ALIGN;
  if (batch * (nc + 1) > 65535 || lanes > ((int64_t)1 << 37)) return MQC_E_LIMIT;
  if (workspace_bytes < mqc_q_chunked_workspace_bytes(batch, seq_len, lanes, chunk_len, 0))
    return MQC_E_SPACE;
  float* ws = (float*)workspace;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case MQC_F32: return launch_cumprod_chunked<float>(q, out, batch, seq_len, lanes, chunk_len, nc, ws, s);
    case MQC_BF16: return launch_cumprod_chunked<bf16_t>(q, out, batch, seq_len, lanes, chunk_len, nc, ws, s);
    case MQC_F16: return launch_cumprod_chunked<f16_t>(q, out, batch, seq_len, lanes, chunk_len, nc, ws, s);
    default: return MQC_E_DTYPE;
  }
}

int mqc_ssm_q_fwd_chunked(const void* q, const void* B, const void* Sq, const void* C, const void* D,
                          int64_t d_stride_b, int64_t d_stride_t, int64_t d_stride_d, void* y,
                          int64_t batch, int64_t seq_len, int64_t d_model, int64_t d_state,
                          int64_t chunk_len, int dtype, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  if (batch < 1 || seq_len < 1 || d_model < 1 || d_state < 1 || chunk_len < 1) return MQC_E_SHAPE;
  const int64_t nc = carries(seq_len, chunk_len);
  if (nc < 1) return MQC_E_SHAPE;
  if (!q || !B || !Sq || !C || !D || !y || !workspace) return MQC_E_NULL;
  if (!aligned(workspace, 16)) return MQC_E_ALIGN;
  if (d_state > 256 || batch * (nc + 1) > 65535) return MQC_E_LIMIT;
  if (workspace_bytes < mqc_q_chunked_workspace_bytes(batch, seq_len, d_model * d_state, chunk_len, 1))
    return MQC_E_SPACE;
  SsmArgs a{};
  a.q = q; a.Bm = B; a.Sq = Sq; a.Cm = C; a.Dq = D;
  a.d_sb = d_stride_b; a.d_st = d_stride_t; a.d_sd = d_stride_d;
  a.y = y;
  a.batch = batch; a.T = seq_len; a.Dm = d_model; a.S = d_state;
  a.chunk_len = chunk_len; a.n_chunks = nc + 1;
  float* ws = (float*)workspace;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case MQC_F32: return launch_ssm_q_chunked<float>(a, nc, ws, s);
    case MQC_BF16: return launch_ssm_q_chunked<bf16_t>(a, nc, ws, s);
    case MQC_F16: return launch_ssm_q_chunked<f16_t>(a, nc, ws, s);
    default: return MQC_E_DTYPE;
  }
}

}  // extern "C"
