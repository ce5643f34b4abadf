// The block's B/C projections fused with its SSM walk for short sequences (at most 128
// tokens; bf16 or fp16 storage, fp32 accumulation): the recurrence and the semantics of
// fused_bc.hip, in tiles that suit a prompt.
//
//   B = x . W_B^T, C = x . W_C^T     (F.linear, mambaqc/layers/quaternion_linear.py:145-161),
//   h_t = Cayley(delta_t Lambda) (x) h_{t-1} + s_t B_t,  y_t = sum_k C_{t,k} (x) h_{t,k} + D s_t
//                                    (models/quaternion_mamba2_block.py:206-228).
//
// At 100 tokens the projections read 2.4 GB of weights (d_inner 1536, 64 states) for 0.5
// TFLOP: the step is a stream of the weights from HBM (0.38 ms at 6.3 TB/s), and a 256-token
// tile spends 0.5 ms of MFMA time on mostly padding. So:
//   - One workgroup of 4 waves per (d, 16 states, pack of sequences): 64 rows of W_B and 64 of
//     W_C against TX = 64 or 128 tokens. Its LDS (72 or 80 KiB) lets two workgroups share a CU,
//     so one streams weights while the other walks. W has three LDS slots; at 128 tokens X, which
//     comes from the L2, has two, all that fits (both with two: 536 us at 100 tokens, as here 514).
//   - The tile holds whole sequences: TX / TP of them, TP the length rounded up to whole
//     chunks (TX / 16 tokens), so short sequences of a batch share one read of the weights.
//   - The walk is fused_bc.hip's: per (state, chunk) lane the chunk from zero, a DPP scan over
//     the 16 chunks of a state, restarted at each sequence's first chunk, where h0 enters, and
//     the chunk's outputs from its start state, summed over the 16 states of the row.
//   - y sums over the d's groups of 16 states: fp32 partial sums in the caller's workspace,
//     added in order by a last launch (with one group, written directly).
#include <atomic>

#include "fused_bc.hpp"

namespace mqc {
namespace {

constexpr int kQS = 16;          // states per workgroup
constexpr int kQRows = 4 * kQS;  // weight rows of each of W_B and W_C
constexpr int kQThreads = 256;
constexpr int kQChunks = 16;
constexpr int kTokB = kQS * 8;   // bytes of a token in the B or the C tile

// LDS: the K loop's slots, over which all of the walk's tables are laid: the B and C tiles, the
// chunks' (H, P), (delta, s) per token and the states' Cayley constants. 72 KiB for 64 tokens
// and exactly half a CU's 160 KiB for 128.
template <int TX, int NSW_, int NSX_>
struct Short {
  using Cfg = TileCfg<2 * kQRows, TX, 2, 2>;
  static constexpr int NSW = NSW_, NSX = NSX_;
  static constexpr int kCL = TX / kQChunks;  // tokens per chunk
  static constexpr int kOffC = TX * kTokB;
  static constexpr int kOffH = 2 * TX * kTokB;
  static constexpr int kOffP = kOffH + kQChunks * kQS * 16;
  static constexpr int kOffDS = kOffP + kQChunks * kQS * 8;
  static constexpr int kOffLT = kOffDS + TX * 8;
  static constexpr int kLds = NSW * Cfg::kWBytes + NSX * TX * kRowBytes;
  static_assert(kOffLT + kQS * 32 <= kLds, "the walk's tables fit the slots");
  static_assert(2 * kLds <= 160 * 1024, "two workgroups per CU");
};

// The same pointer in scalar registers, where the DMA takes it (it is wave-uniform; this
// kernel's 64-bit products of it otherwise end up on the VALU).
__device__ inline const void* uniform_ptr(const void* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const void*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

struct ShortArgs {
  const uint16_t* x;   // [batch, T, K] (K = d_inner)
  const uint16_t* wb;  // [d_inner * S * 4, K]
  const uint16_t* wc;
  const uint16_t* delta;  // [batch, T, d_inner]
  const uint16_t* s;
  const float* lam_alpha;  // [d_inner, S]
  const float* lam_imag;   // [d_inner, S, 3]
  const float* dvec;       // [d_inner]
  const float* h0;         // [batch, d_inner, S, 4] or null
  uint16_t* y;             // [batch, T, d_inner, 4] (one group of states)
  float* h_last;           // [batch, d_inner, S, 4] or null
  float* ypart;            // [groups, batch, T, d_inner, 4] (several)
  int batch, T, Dm, S;
  int TP;                  // T rounded up to whole chunks
  int per_pack;            // sequences per tile
  float eps;
};

// Sum of o[N] over the 16 lanes of a row, scattered: stages at lane distances 8 (row
// rotation), 4 (half-row mirror), 2 and 1 (quad permutes), at each of which a lane keeps the upper
// half of its values if its bit is set and adds its partner's. Afterwards lane u holds the sums
// of the N / 16 values from u * (N / 16) on.
template <int N>
__device__ inline void reduce_scatter16(float (&o)[N], int lane, float (&r)[N / 16]) {
  const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2, b0 = lane & 1;
  float w[N / 2], z[N / 4], v[N / 8];
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const float send = b3 ? o[i] : o[N / 2 + i];
    w[i] = (b3 ? o[N / 2 + i] : o[i]) + row_rot8(send);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const float send = b2 ? w[i] : w[N / 4 + i];
    z[i] = (b2 ? w[N / 4 + i] : w[i]) + row_half_mirror(send);
  }
#pragma unroll
  for (int i = 0; i < N / 8; ++i) {
    const float send = b1 ? z[i] : z[N / 8 + i];
    v[i] = (b1 ? z[N / 8 + i] : z[i]) + lane_xor2(send);
  }
#pragma unroll
  for (int i = 0; i < N / 16; ++i) {
    const float send = b0 ? v[i] : v[N / 16 + i];
    r[i] = (b0 ? v[N / 16 + i] : v[i]) + lane_xor1(send);
  }
}

// HBM-bound (the weights, read once by each pack): see the note above and the rule in
// kernels/ssm_fused.py for both sides of the choice, measured.
template <typename T, typename L>
__global__ __launch_bounds__(kQThreads) __attribute__((amdgpu_waves_per_eu(2))) void
fused_bc_short_kernel(ShortArgs a) {
  using E = typename std::conditional<std::is_same<T, bf16_t>::value, __bf16, _Float16>::type;
  using Cfg = typename L::Cfg;
  constexpr int TX = Cfg::TX, CL = L::kCL;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave / Cfg::NW_X, wm = wave % Cfg::NW_X;
  const int rl = lane & 15, q4 = lane >> 4;

  // Unit (d, group of states, pack), d-major with the packs adjacent (they share the weight rows),
  // each XCD a contiguous range.
  const int n = (int)gridDim.x, lin = (int)blockIdx.x;
  const int logical = n % kXCDs ? lin : (lin % kXCDs) * (n / kXCDs) + lin / kXCDs;
  const int K = a.Dm, S = a.S;
  const int groups = (S + kQS - 1) / kQS;
  const int packs = (a.batch + a.per_pack - 1) / a.per_pack;
  const int d = __builtin_amdgcn_readfirstlane(logical / (groups * packs));
  const int rem = logical - d * (groups * packs);
  const int g = __builtin_amdgcn_readfirstlane(rem / packs);
  const int b0 = __builtin_amdgcn_readfirstlane((rem - g * packs) * a.per_pack);
  const int hs = S - g * kQS < kQS ? S - g * kQS : kQS;

  // Row r of the tile is token r % TP of sequence b0 + r / TP; rows past a sequence's end, and
  // sequences past the batch, read its last token.
  auto token_row = [&](int r) {
    int bb = r / a.TP;
    int t = r - bb * a.TP;
    if (t >= a.T) t = a.T - 1;
    bb += b0;
    if (bb >= a.batch) bb = a.batch - 1;
    return bb * a.T + t;
  };
  const DmaLane dl(lane);
  uint32_t xoff[Cfg::kXLoads];
#pragma unroll
  for (int i = 0; i < Cfg::kXLoads; ++i)
    xoff[i] = (uint32_t)(token_row((wave * Cfg::kXLoads + i) * kRowsPerLoad + dl.lrow) - b0 * a.T) *
              (uint32_t)(K * 2);
  const WRowsOf<kQRows> wr{a.wb, a.wc, ((int64_t)d * S + g * kQS) * 4, 4 * hs, K};
  auto wrows = [&](int gr, int k0, int gi, uint32_t& voff, const DmaLane& l) -> const void* {
    return uniform_ptr(wr(gr, k0, gi, voff, l));
  };
  auto xrows = [&](int, int k0, int gi, uint32_t& voff, const DmaLane& l) -> const void* {
    uint32_t o = xoff[0];
#pragma unroll
    for (int i = 1; i < Cfg::kXLoads; ++i) o = gi == wave * Cfg::kXLoads + i ? xoff[i] : o;
    voff = o + l.cb(gi);
    return uniform_ptr(a.x + ((int64_t)b0 * a.T * K + k0));
  };

  // The tokens' delta and s and the states' parameters, loaded ahead of the first stages.
  float dl_t = 0.f, s_t = 0.f;
  bool real = false;
  if (tid < TX) {
    const int bb = tid / a.TP, t = tid - bb * a.TP;
    real = bb < a.per_pack && b0 + bb < a.batch && t < a.T;
    const int64_t e = (int64_t)token_row(tid) * a.Dm + d;
    dl_t = io<T>::bits_to_f32(a.delta[e]);
    s_t = io<T>::bits_to_f32(a.s[e]);
  }
  // (States past S are clamped and their results discarded.)
  float alpha = 0.f, imag0 = 0.f, imag1 = 0.f, imag2 = 0.f;
  if (tid < kQS) {
    const int64_t dk = (int64_t)d * S + g * kQS + (tid < hs ? tid : hs - 1);
    alpha = a.lam_alpha[dk];
    imag0 = a.lam_imag[dk * 3 + 0];
    imag1 = a.lam_imag[dk * 3 + 1];
    imag2 = a.lam_imag[dk * 3 + 2];
  }
  const uint32_t lds0 = lds_addr(lds);
  const int KT = K / kBK;
  // (With fewer stages of K than slots, a slot gets stage 0 again and is not read.)
#pragma unroll
  for (int kt = 0; kt < L::NSW - 1; ++kt) {
    if (L::NSX == 2 && kt == L::NSW - 2) tile_issue_x<Cfg, L::NSW>(0, 0, wave, lds0, dl, xrows);
    tile_issue_w<Cfg, L::NSW>(kt < KT ? kt : 0, kt, wave, lds0, dl, wrows);
    if (L::NSX > 2) tile_issue_x<Cfg, L::NSW>(kt < KT ? kt : 0, kt, wave, lds0, dl, xrows);
  }

  floatx4 acc[Cfg::WB][Cfg::XB];
#pragma unroll
  for (int i = 0; i < Cfg::WB; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::XB; ++j) acc[i][j] = (floatx4){};
  tile_kloop_deep<Cfg, L::NSW, L::NSX, E>(K, lds, acc, wrows, xrows);

  // The tile, rounded to T, over the stages: cell of (token t, state k) k ^ (t & 15) of the
  // token's 128-byte row in the B (wn 0) or C (wn 1) tile.
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int nb = 0; nb < Cfg::WB; ++nb)
#pragma unroll
    for (int mb = 0; mb < Cfg::XB; ++mb) {
      const int t = wm * (TX / Cfg::NW_X) + mb * 16 + rl;
      const floatx4& v = acc[nb][mb];
      const u32x2 pk = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
      *(u32x2*)(lds + wn * L::kOffC + t * kTokB + (((nb * 4 + q4) ^ rl) << 3)) = pk;
    }
  if (tid < kQS) {
    const LamConst lc = lam_from(alpha, imag0, imag1, imag2);
    *(float4*)(lds + L::kOffLT + tid * 32) =
        float4{lc.v0, lc.v1, lc.v2, lc.v0 * lc.v0 + lc.v1 * lc.v1 + lc.v2 * lc.v2};
    *(float4*)(lds + L::kOffLT + tid * 32 + 16) = float4{lc.a, lc.n2, 0.f, 0.f};
  }
  if (tid < TX)
    *(float2*)(lds + L::kOffDS + tid * 8) = float2{real ? dl_t : 0.f, real ? s_t : 0.f};
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();

  // Every chunk from zero (state kA, chunk cA): its states, the products of its q's and its transition.
  const int kA = tid & (kQS - 1), cA = tid / kQS;
  LamConst lam;
  float vv;
  {
    const float4 lv = *(const float4*)(lds + L::kOffLT + kA * 32);
    const float4 la = *(const float4*)(lds + L::kOffLT + kA * 32 + 16);
    lam.v0 = lv.x; lam.v1 = lv.y; lam.v2 = lv.z; vv = lv.w;
    lam.a = la.x; lam.n2 = la.y;
  }
  const int per_seq = a.TP / CL;  // chunks per sequence
  quat hl[CL];
  float pa[CL], pb[CL];
  {
    quat hh{0.f, 0.f, 0.f, 0.f};
    float ca = 1.f, cb = 0.f;
    // Steps of the chunk that are tokens.
    const int seq = cA / per_seq;
    const int live = a.T - (cA - seq * per_seq) * CL;
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      const int t = cA * CL + j;
      const float2 ds = *(const float2*)(lds + L::kOffDS + t * 8);
      const u32x2 br = *(const u32x2*)(lds + t * kTokB + ((kA ^ (t & 15)) << 3));
      const quat Bq{lo16<T>(br[0]), hi16<T>(br[0]), lo16<T>(br[1]), hi16<T>(br[1])};
      float c;
      quat qq = cayley_step_c(ds.x, ds.x * ds.x, lam, a.eps, c);
      float sv = ds.y;
      if (j >= live) {
        // Past the sequence: the identity, and no input (whatever the clamped row holds).
        qq = quat{1.f, 0.f, 0.f, 0.f};
        c = 0.f;
      } else {
        hh = state_step(qq, hh, sv, Bq);
      }
      const float na = fmaf(qq.w, ca, -c * cb * vv);
      cb = fmaf(qq.w, cb, c * ca);
      ca = na;
      hl[j] = hh;
      pa[j] = ca;
      pb[j] = cb;
    }
    *(float4*)(lds + L::kOffH + (cA * kQS + kA) * 16) = float4{hh.w, hh.x, hh.y, hh.z};
    *(float2*)(lds + L::kOffP + (cA * kQS + kA) * 8) = float2{ca, cb};
  }
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();

  // Start states: an inclusive scan over each state's chunks (one 16-lane row), within each
  // sequence, h0 folded into its first chunk and its last chunk's end the state.
  {
    const int kS = tid >> 4, cS = tid & 15;
    const int seq = cS / per_seq, cq = cS - seq * per_seq;
    const int bb = b0 + seq;
    const bool in = seq < a.per_pack && bb < a.batch && kS < hs;
    const int64_t sidx = (((int64_t)(in ? bb : b0) * a.Dm + d) * S + g * kQS + (kS < hs ? kS : 0)) * 4;
    const float4 e = *(const float4*)(lds + L::kOffH + (cS * kQS + kS) * 16);
    const float2 p = *(const float2*)(lds + L::kOffP + (cS * kQS + kS) * 8);
    const float4 lt = *(const float4*)(lds + L::kOffLT + kS * 32);
    float4 hc = {0.f, 0.f, 0.f, 0.f};
    if (a.h0 && in && cq == 0) hc = *(const float4*)(a.h0 + sidx);
    LamConst LS{};
    LS.v0 = lt.x; LS.v1 = lt.y; LS.v2 = lt.z;
    ChunkMap m;
    m.pa = p.x;
    m.pb = p.y;
    m.H = quat{e.x, e.y, e.z, e.w};
    if (cq == 0) {
      const quat ph = vplane_mul(m.pa, m.pb, LS, quat{hc.x, hc.y, hc.z, hc.w});
      m.H = quat{ph.w + m.H.w, ph.x + m.H.x, ph.y + m.H.y, ph.z + m.H.z};
    }
    const ChunkMap e1 = dpp_map<0x111, 0xF>(m);  // row_shr:1
    if (cq >= 1) m = compose(m, e1, lt.w, LS);
    const ChunkMap e2 = dpp_map<0x112, 0xF>(m);  // row_shr:2
    if (cq >= 2) m = compose(m, e2, lt.w, LS);
    const ChunkMap e4 = dpp_map<0x114, 0xF>(m);  // row_shr:4
    if (cq >= 4) m = compose(m, e4, lt.w, LS);
    const ChunkMap e8 = dpp_map<0x118, 0xF>(m);  // row_shr:8
    if (cq >= 8) m = compose(m, e8, lt.w, LS);
    // (A state's chunks are one row of one wave, whose reads above all precede these writes.)
    const float4 mh = {m.H.w, m.H.x, m.H.y, m.H.z};
    if (cq == per_seq - 1) {
      if (a.h_last && in) *(float4*)(a.h_last + sidx) = mh;
    } else if (cS < kQChunks - 1) {
      *(float4*)(lds + L::kOffH + ((cS + 1) * kQS + kS) * 16) = mh;
    }
    if (cq == 0) *(float4*)(lds + L::kOffH + (cS * kQS + kS) * 16) = hc;
  }
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();

  // Every chunk's states from its start state h_s, h_j = P_j (x) h_s + hl_j, and y's terms C_j (x) h_j.
  {
    const float4 e = *(const float4*)(lds + L::kOffH + (cA * kQS + kA) * 16);
    const quat hs0{e.x, e.y, e.z, e.w};
    const quat vh = qmul(quat{0.f, lam.v0, lam.v1, lam.v2}, hs0);
    float o[4 * CL];
    const bool live = kA < hs;
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      const int t = cA * CL + j;
      const u32x2 r = *(const u32x2*)(lds + L::kOffC + t * kTokB + ((kA ^ (t & 15)) << 3));
      const quat Cq{lo16<T>(r[0]), hi16<T>(r[0]), lo16<T>(r[1]), hi16<T>(r[1])};
      const quat hh{fmaf(pa[j], hs0.w, fmaf(pb[j], vh.w, hl[j].w)),
                    fmaf(pa[j], hs0.x, fmaf(pb[j], vh.x, hl[j].x)),
                    fmaf(pa[j], hs0.y, fmaf(pb[j], vh.y, hl[j].y)),
                    fmaf(pa[j], hs0.z, fmaf(pb[j], vh.z, hl[j].z))};
      const quat oc = qmul(Cq, hh);
      o[4 * j + 0] = live ? oc.w : 0.f;
      o[4 * j + 1] = live ? oc.x : 0.f;
      o[4 * j + 2] = live ? oc.y : 0.f;
      o[4 * j + 3] = live ? oc.z : 0.f;
    }
    constexpr int NR = CL / 4;  // sums per lane: 1 or 2 components of one token
    float r[NR];
    reduce_scatter16<4 * CL>(o, lane, r);
    const int i0 = (lane & 15) * NR;
    const int row = cA * CL + (i0 >> 2);
    const int bb = row / a.TP, t = row - bb * a.TP;
    if (bb < a.per_pack && b0 + bb < a.batch && t < a.T) {
      const int64_t tok = (int64_t)(b0 + bb) * a.T + t;
      const int64_t idx = (tok * a.Dm + d) * 4 + (i0 & 3);
      if (a.ypart) {
        float* yp = a.ypart + (int64_t)g * a.batch * a.T * a.Dm * 4 + idx;
#pragma unroll
        for (int i = 0; i < NR; ++i) yp[i] = r[i];
      } else {
        if ((i0 & 3) == 0)
          r[0] = fmaf(a.dvec[d], (*(const float2*)(lds + L::kOffDS + row * 8)).y, r[0]);
#pragma unroll
        for (int i = 0; i < NR; ++i) a.y[idx + i] = io<T>::from_f32(r[i]).bits;
      }
    }
  }
}

// y = T(the groups' partial sums in order + (D s, 0, 0, 0)).
template <typename T>
__global__ __launch_bounds__(256) void fused_bc_short_sum_kernel(const float* __restrict__ ypart,
                                                                 const uint16_t* __restrict__ s,
                                                                 const float* __restrict__ dvec,
                                                                 uint16_t* __restrict__ y,
                                                                 int64_t n, int groups, int Dm) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  float4 v = *(const float4*)(ypart + e * 4);
  for (int g = 1; g < groups; ++g) {
    const float4 p = *(const float4*)(ypart + ((int64_t)g * n + e) * 4);
    v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
  }
  const float sv = io<T>::bits_to_f32(s[e]);
  const u32x2 pk = {pack2<T>(fmaf(dvec[e % Dm], sv, v.x), v.y), pack2<T>(v.z, v.w)};
  *(u32x2*)(y + e * 4) = pk;
}

using Short64 = Short<64, 3, 3>;
using Short128 = Short<128, 3, 2>;
constexpr int kShortMax = 128;

int64_t short_groups(int64_t d_state) { return (d_state + kQS - 1) / kQS; }

int64_t short_workspace(int64_t batch, int64_t T, int64_t d_inner, int64_t d_state) {
  const int64_t g = short_groups(d_state);
  return g > 1 ? g * batch * T * d_inner * 4 * (int64_t)sizeof(float) : 0;
}

template <typename T, typename L>
int launch_short(const ShortArgs& a0, hipStream_t st) {
  static std::atomic<bool> attr_set[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64) return MQC_E_LIMIT;
  if (!attr_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute((const void*)fused_bc_short_kernel<T, L>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, L::kLds);
    if (e != hipSuccess) return (int)e;
    attr_set[dev].store(true, std::memory_order_release);
  }
  ShortArgs a = a0;
  a.TP = (a.T + L::kCL - 1) / L::kCL * L::kCL;
  a.per_pack = L::Cfg::TX / a.TP;
  const int64_t packs = (a.batch + a.per_pack - 1) / a.per_pack;
  const int64_t units = (int64_t)a.Dm * short_groups(a.S) * packs;
  if (units > 0x7fffffffLL) return MQC_E_LIMIT;
  fused_bc_short_kernel<T, L><<<dim3((unsigned)units), dim3(kQThreads), L::kLds, st>>>(a);
  int status = launch_status();
  if (status != MQC_OK || !a.ypart) return status;
  const int64_t n = (int64_t)a.batch * a.T * a.Dm;
  fused_bc_short_sum_kernel<T><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(
      a.ypart, a.s, a.dvec, a.y, n, (int)short_groups(a.S), a.Dm);
  return launch_status();
}

}  // namespace
}  // namespace mqc

using namespace mqc;

extern "C" {

int64_t mqc_ssm_fused_bc_short_workspace_bytes(int64_t batch, int64_t seq_len, int64_t d_inner,
                                               int64_t d_state) {
  if (batch < 0 || seq_len < 0 || d_inner < 0 || d_state < 0) return MQC_E_SHAPE;
  return short_workspace(batch, seq_len, d_inner, d_state);
}

int mqc_ssm_fused_bc_short_fwd(const void* x, const void* B_weight, const void* C_weight,
                               const void* delta, const void* s, const float* lambda_alpha,
                               const float* lambda_imag, const float* D, const void* h0, void* y,
                               void* h_last, int64_t batch, int64_t seq_len, int64_t d_inner,
                               int64_t d_state, float eps, int dtype, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  if (batch < 0 || seq_len < 0 || d_inner < 0 || d_state < 0) return MQC_E_SHAPE;
  if (dtype != MQC_BF16 && dtype != MQC_F16) return MQC_E_DTYPE;
  if (batch == 0 || d_inner == 0) return MQC_OK;
  if (d_state < 1 || d_state > 64 || seq_len > kShortMax) return MQC_E_LIMIT;
  if (seq_len < 1 || d_state % 2 != 0 || d_inner % kBK != 0) return MQC_E_SHAPE;
  if (!x || !B_weight || !C_weight || !delta || !s || !y || !lambda_alpha || !lambda_imag || !D)
    return MQC_E_NULL;
  if (!aligned(x, 16) || !aligned(B_weight, 16) || !aligned(C_weight, 16) || !aligned(y, 8) ||
      !aligned(delta, 2) || !aligned(s, 2) || (h0 && !aligned(h0, 16)) ||
      (h_last && !aligned(h_last, 16)))
    return MQC_E_ALIGN;
  // 32-bit token and unit indices, and byte offsets inside a tile's rows of x.
  if (batch * d_inner * 64 > 0x7fffffffLL || batch * seq_len > (1LL << 30) ||
      kShortMax * d_inner * 2 >= (1LL << 31))
    return MQC_E_LIMIT;
  const int64_t need = short_workspace(batch, seq_len, d_inner, d_state);
  if (need > 0) {
    if (!workspace) return MQC_E_NULL;
    if (!aligned(workspace, 16)) return MQC_E_ALIGN;
    if (workspace_bytes < need) return MQC_E_SPACE;
  }
  // A unit reads its states of h0 before it writes them to h_last.
  if (partial_overlap(h0, h_last, batch * d_inner * d_state * 4 * (int64_t)sizeof(float)))
    return MQC_E_OVERLAP;
  ShortArgs a{};
  a.x = (const uint16_t*)x; a.wb = (const uint16_t*)B_weight; a.wc = (const uint16_t*)C_weight;
  a.delta = (const uint16_t*)delta; a.s = (const uint16_t*)s;
  a.lam_alpha = lambda_alpha; a.lam_imag = lambda_imag; a.dvec = D;
  a.h0 = (const float*)h0; a.y = (uint16_t*)y; a.h_last = (float*)h_last;
  a.ypart = need > 0 ? (float*)workspace : nullptr;
  a.batch = (int)batch; a.T = (int)seq_len; a.Dm = (int)d_inner; a.S = (int)d_state; a.eps = eps;
  hipStream_t st = (hipStream_t)stream;
  // The 64-token tile where the sequences of the batch fit it.
  const bool small = batch * ((seq_len + 3) / 4 * 4) <= 64;
  if (dtype == MQC_BF16)
    return small ? launch_short<bf16_t, Short64>(a, st) : launch_short<bf16_t, Short128>(a, st);
  return small ? launch_short<f16_t, Short64>(a, st) : launch_short<f16_t, Short128>(a, st);
}

}  // extern "C"
