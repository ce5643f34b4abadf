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
// Launch 1 reads q (and B) a second time, so it pays only where the chain, not HBM, is the bound: the
// rules are with the callers (kernels/parallel_scan.py, kernels/ssm_fused.py), both sides measured.
#include "ssm_scan.hpp"

namespace mqc {
namespace {

// 1. One thread per (chunk, b, lane); the next PF steps' loads are in flight.
template <typename T, bool SSM>
__global__ __launch_bounds__(256) void q_chunk_agg_kernel(const T* __restrict__ q,
                                                          const T* __restrict__ Bm,
                                                          const T* __restrict__ Sq, float* __restrict__ Hc,
                                                          float* __restrict__ Pc, int64_t batch,
                                                          int64_t T_len, int64_t lanes, int64_t S,
                                                          int64_t L, int64_t nc) {
  constexpr int PF = 8;
  const int64_t l = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t b = blockIdx.y % batch, c = blockIdx.y / batch;
  if (l >= lanes) return;
  const int64_t row = lanes * 4;
  const int64_t base = (b * T_len + c * L) * row + l * 4;  // (every chunk here is whole)
  const int64_t d = SSM ? l / S : 0, D = SSM ? lanes / S : 0;
  const T* sp = SSM ? Sq + ((b * T_len + c * L) * D + d) * 4 : nullptr;
  quat P{1.f, 0.f, 0.f, 0.f}, H{0.f, 0.f, 0.f, 0.f};
  for (int64_t t0 = 0; t0 < L; t0 += PF) {
    float qv[PF][4], bv[SSM ? PF : 1][4], sv[SSM ? PF : 1][4];
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int64_t t = t0 + i < L ? t0 + i : L - 1;
      load_vec<T, 4>(q + base + t * row, qv[i]);
      if constexpr (SSM) {
        load_vec<T, 4>(Bm + base + t * row, bv[i]);
        load_vec<T, 4>(sp + t * D * 4, sv[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      if (t0 + i < L) {
        const quat qq = quat_from(qv[i]);
        P = qmul(qq, P);
        if constexpr (SSM) {
          quat hn = qmul(quat_from(bv[i]), quat_from(sv[i]));
          qmul_acc(hn, qq, H);
          H = hn;
        }
      }
    }
  }
  const int64_t o = ((b * nc + c) * lanes + l) * 4;
  const float e[4] = {P.w, P.x, P.y, P.z};
  store_vec<float, 4>(Pc + o, e);
  if constexpr (SSM) {
    const float h[4] = {H.w, H.x, H.y, H.z};
    store_vec<float, 4>(Hc + o, h);
  }
}

// 2. One thread per (b, lane): the carries in place, in Pc (products) or Hc (states).
template <bool SSM>
__global__ __launch_bounds__(256) void q_chunk_prefix_kernel(float* __restrict__ Hc,
                                                             float* __restrict__ Pc, int64_t batch,
                                                             int64_t lanes, int64_t nc) {
  constexpr int PF = 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= batch * lanes) return;
  const int64_t b = i / lanes, l = i - b * lanes;
  const int64_t o = (b * nc * lanes + l) * 4, step = lanes * 4;
  quat E{SSM ? 0.f : 1.f, 0.f, 0.f, 0.f};
  for (int64_t c0 = 0; c0 < nc; c0 += PF) {
    float p[PF][4], h[SSM ? PF : 1][4];
#pragma unroll
    for (int k = 0; k < PF; ++k) {
      const int64_t c = c0 + k < nc ? c0 + k : nc - 1;
      load_vec<float, 4>(Pc + o + c * step, p[k]);
      if constexpr (SSM) load_vec<float, 4>(Hc + o + c * step, h[k]);
    }
#pragma unroll
    for (int k = 0; k < PF; ++k) {
      if (c0 + k < nc) {
        quat n = qmul(quat_from(p[k]), E);
        if constexpr (SSM) {
          n.w += h[k][0]; n.x += h[k][1]; n.y += h[k][2]; n.z += h[k][3];
        }
        E = n;
        const float e[4] = {E.w, E.x, E.y, E.z};
        store_vec<float, 4>((SSM ? Hc : Pc) + o + (c0 + k) * step, e);
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
  q_chunk_agg_kernel<T, false><<<dim3(gx, (unsigned)(batch * nc)), 256, 0, s>>>(
      (const T*)q, nullptr, nullptr, nullptr, ws, batch, T_len, lanes, 1, L, nc);
  q_chunk_prefix_kernel<false><<<dim3((unsigned)((batch * lanes + 255) / 256)), 256, 0, s>>>(
      nullptr, ws, batch, lanes, nc);
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
  q_chunk_agg_kernel<T, true>
      <<<dim3((unsigned)((lanes + 255) / 256), (unsigned)(a.batch * nc)), 256, 0, s>>>(
          (const T*)a.q, (const T*)a.Bm, (const T*)a.Sq, Hc, Pc, a.batch, a.T, lanes, a.S,
          a.chunk_len, nc);
  q_chunk_prefix_kernel<true><<<dim3((unsigned)((a.batch * lanes + 255) / 256)), 256, 0, s>>>(
      Hc, Pc, a.batch, lanes, nc);
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
  return batch * carries(seq_len, chunk_len) * lanes * 4 * (int64_t)sizeof(float) * (ssm ? 2 : 1);
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
