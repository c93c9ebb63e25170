// Recurrent gated delta rule (state on chip in fp32, any number of tokens) and the fused decode step.
//
// Per token (sore/model/gdn_ref.py:17-21):
//   a = exp(g), S_dec = a S, delta = beta (v - S_dec^T k), S' = S_dec + k delta^T, o = scale S'^T q.
// The state [K, V] fp32 of a (sequence, value head) is read from HBM once, kept in registers and written once.
// Three kernels: gated_delta_recurrent_kernel takes 16 tokens at a time on fp32 MFMAs,
// gated_delta_recurrent_short_kernel a few tokens one by one, gated_delta_decode_w4_kernel one token together
// with the conv cache's step (gated_delta_decode_kernel for other conv widths and types, with the state in 256
// threads: thread t owns the columns 4*(t % (V/4)) .. +3 and the rows rg + RG*i, rg = t / (V/4)).

#include <type_traits>

#include "gdn_common.h"
#include "gdn_mfma.h"

namespace gdn {

struct RecParams {
  const void *q, *k, *v, *g, *beta;
  const float* h0;
  void* o;
  float* ht;
  const void* cu;
  int cu_i32;
  int64_t T, H, HV;
  int dq, dg, db;
  float scale;
  unsigned flags;
  const float *A_log, *dt_bias;
};

template <int KD, int VD>
struct RecLayout {
  static constexpr int NT = 256;
  static constexpr int CG = VD / 4;  // column groups of 4 columns
  static constexpr int RG = NT / CG;  // row groups
  static constexpr int RPT = KD / RG;  // rows per thread
  static constexpr int NW = NT / kWave;
  static constexpr int NRED = 11;  // S^T k (4), S^T q (4), k.q, k.k, q.q
  static_assert(CG <= kWave && RG * RPT == KD, "unsupported head dims");
};

// The thread's slice of the state: RPT rows x 4 columns, in registers.
template <int KD, int VD>
struct StateRegs {
  float4 r[RecLayout<KD, VD>::RPT];
};

// Decay and write strength of one (token, value head).
__device__ __forceinline__ void gate_values(const RecParams& p, int64_t idx, int hv, float& a, float& b) {
  float gv = load_as_f32(p.g, p.dg, idx);
  if (p.flags & GDN_FLAG_GATE_IN_KERNEL) gv = -expf(p.A_log[hv]) * softplus_f32(gv + p.dt_bias[hv]);
  a = expf(gv);
  float bv = load_as_f32(p.beta, p.db, idx);
  b = (p.flags & GDN_FLAG_BETA_SIGMOID) ? sigmoid_f32(bv) : bv;
}

// One token on the register-resident state. q_l/k_l/v_l are the token's vectors in LDS (fp32),
// red is an LDS exchange buffer of NW*CG*12 floats. Writes the 4 output columns into o4.
template <int KD, int VD>
__device__ __forceinline__ void rec_token(StateRegs<KD, VD>& sr, const float* q_l, const float* k_l,
                                          const float* v_l, float a, float b, bool l2, float scale, float* red,
                                          float (&o4)[4]) {
  using L = RecLayout<KD, VD>;
  auto& s = sr.r;
  const int t = threadIdx.x, cg = t % L::CG, rg = t / L::CG, lane = t % kWave, w = t / kWave;
  float p[L::NRED];
#pragma unroll
  for (int j = 0; j < L::NRED; ++j) p[j] = 0.f;
#pragma unroll
  for (int i = 0; i < L::RPT; ++i) {
    const int r = rg + L::RG * i;
    const float kr = k_l[r], qr = q_l[r];
    p[0] += s[i].x * kr; p[1] += s[i].y * kr; p[2] += s[i].z * kr; p[3] += s[i].w * kr;
    p[4] += s[i].x * qr; p[5] += s[i].y * qr; p[6] += s[i].z * qr; p[7] += s[i].w * qr;
    p[8] += kr * qr; p[9] += kr * kr; p[10] += qr * qr;
  }
#pragma unroll
  for (int j = 0; j < L::NRED; ++j) p[j] = wave_xor_sum(p[j], L::CG);
  if (lane < L::CG) {
#pragma unroll
    for (int j = 0; j < L::NRED; ++j) red[(w * L::CG + cg) * 12 + j] = p[j];
  }
  __syncthreads();
  float tot[L::NRED];
#pragma unroll
  for (int j = 0; j < L::NRED; ++j) {
    float x = 0.f;
#pragma unroll
    for (int ww = 0; ww < L::NW; ++ww) x += red[(ww * L::CG + cg) * 12 + j];
    tot[j] = x;
  }
  // F.normalize semantics: x / max(||x||, 1e-12)
  const float ik = l2 ? 1.f / fmaxf(sqrtf(tot[9]), 1e-12f) : 1.f;
  const float iq = l2 ? 1.f / fmaxf(sqrtf(tot[10]), 1e-12f) : 1.f;
  float d[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    d[c] = b * (v_l[4 * cg + c] - a * tot[c] * ik);
    o4[c] = scale * (a * tot[4 + c] * iq + d[c] * tot[8] * ik * iq);
  }
#pragma unroll
  for (int i = 0; i < L::RPT; ++i) {
    const float kr = k_l[rg + L::RG * i] * ik;
    s[i].x = a * s[i].x + kr * d[0];
    s[i].y = a * s[i].y + kr * d[1];
    s[i].z = a * s[i].z + kr * d[2];
    s[i].w = a * s[i].w + kr * d[3];
  }
}

template <int KD, int VD>
__device__ __forceinline__ void load_state(StateRegs<KD, VD>& sr, const float* base) {
  using L = RecLayout<KD, VD>;
  auto& s = sr.r;
  const int t = threadIdx.x, cg = t % L::CG, rg = t / L::CG;
#pragma unroll
  for (int i = 0; i < L::RPT; ++i) {
    if (base) s[i] = *reinterpret_cast<const float4*>(base + (int64_t)(rg + L::RG * i) * VD + 4 * cg);
    else s[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

template <int KD, int VD>
__device__ __forceinline__ void store_state(const StateRegs<KD, VD>& sr, float* base) {
  using L = RecLayout<KD, VD>;
  const auto& s = sr.r;
  const int t = threadIdx.x, cg = t % L::CG, rg = t / L::CG;
#pragma unroll
  for (int i = 0; i < L::RPT; ++i) *reinterpret_cast<float4*>(base + (int64_t)(rg + L::RG * i) * VD + 4 * cg) = s[i];
}

template <typename E, int N>
struct RowVec {
  typedef E T __attribute__((ext_vector_type(N), aligned(sizeof(E))));  // rows may start at any element
};

constexpr int kShortTokens = 4;
constexpr float kGrowth = 13.8f;  // log of 2^20

// The recurrence of a few tokens (a decode call, a draft of two or three): one pass over at most G = 4 tokens at a
// time, all their loads issued at once. Columns of the state are independent (column j needs only S[:, j]), so
// a wave owns 16 columns and nothing crosses waves: no LDS, no barrier. Lane (c4, rg) holds rows rg R ..
// rg R + R - 1 (R = K / 16) of columns 4 c4 .. 4 c4 + 3; sums over rows stay inside a 16-lane DPP row. Gates and
// q/k norms are computed with one token per lane and broadcast by readlane; lane rg stores token rg's outputs.
// The state's bytes bound it from 16 sequences of 16 heads up: 64 sequences, T = 1, bf16, d = 128: 25.1 us (134 MB
// of state, 5.3 TB/s); the kernel before it (one workgroup per state, two barriers a token) took 25.5, and 42.4
// at T = 4 against 28.7 here.
template <typename E, int KD, int VD>
__global__ __launch_bounds__(256) void gated_delta_recurrent_short_kernel(RecParams p) {
  constexpr int G = kShortTokens, R = KD / 16, NC = 4;
  using VK = typename RowVec<E, R>::T;
  using VV = typename RowVec<E, NC>::T;
  using VS = typename RowVec<float, NC>::T;
  const int lane = threadIdx.x % kWave, rg = lane % 16;
  constexpr int kSlices = VD / 64;
  const int hv = blockIdx.x / kSlices, col = (blockIdx.x % kSlices) * 64 + (threadIdx.x / 16) * NC;
  const int64_t n = blockIdx.y;
  const int h = hv / (int)(p.HV / p.H);
  int64_t bos, eos;
  if (p.cu) {
    bos = load_index(p.cu, p.cu_i32, n);
    eos = load_index(p.cu, p.cu_i32, n + 1);
  } else {
    bos = n * p.T;
    eos = bos + p.T;
  }
  const int64_t sbase = (n * p.HV + hv) * (int64_t)KD * VD + (int64_t)rg * R * VD + col;
  VS s[R];
#pragma unroll
  for (int i = 0; i < R; ++i) s[i] = p.h0 ? *reinterpret_cast<const VS*>(p.h0 + sbase + i * VD) : VS{};
  const E* __restrict__ kp = static_cast<const E*>(p.k) + (int64_t)h * KD + rg * R;
  const E* __restrict__ qp = static_cast<const E*>(p.q) + (int64_t)h * KD + rg * R;
  const E* __restrict__ vp = static_cast<const E*>(p.v) + (int64_t)hv * VD + col;
  E* __restrict__ op = static_cast<E*>(p.o) + (int64_t)hv * VD + col;
  auto bcast = [](float x, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); };
  for (int64_t t = bos; t < eos; t += G) {
    VK k[G], q[G];
    VV v[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {  // tokens past the end re-read the last one (never used)
      const int64_t tok = t + g < eos ? t + g : eos - 1;
      k[g] = *reinterpret_cast<const VK*>(kp + tok * p.H * KD);
      q[g] = *reinterpret_cast<const VK*>(qp + tok * p.H * KD);
      v[g] = *reinterpret_cast<const VV*>(vp + tok * p.HV * VD);
    }
    const int64_t gt = t + rg % G < eos ? t + rg % G : eos - 1;  // one token's gates per lane
    float av, bv;
    gate_values(p, gt * p.HV + hv, hv, av, bv);
    float ikv = 1.f, iqv = p.scale;  // lane g: 1 / max(|k|, 1e-12) and scale / max(|q|, 1e-12) of token g
    if (p.flags & GDN_FLAG_QK_L2NORM) {
      float kkv = 0.f, qqv = 0.f;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (t + g >= eos) break;
        float kk = 0.f, qq = 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          kk += (float)k[g][i] * (float)k[g][i];
          qq += (float)q[g][i] * (float)q[g][i];
        }
        kk = group_sum<16>(kk);
        qq = group_sum<16>(qq);
        kkv = rg == g ? kk : kkv;
        qqv = rg == g ? qq : qqv;
      }
      ikv = 1.f / fmaxf(sqrtf(kkv), 1e-12f);
      iqv = p.scale / fmaxf(sqrtf(qqv), 1e-12f);
    }
    VV keep{};
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (t + g >= eos) break;
      const float a = bcast(av, g), b = bcast(bv, g), ik = bcast(ikv, g), iq = bcast(iqv, g);
      float kr[R];
#pragma unroll
      for (int i = 0; i < R; ++i) kr[i] = (float)k[g][i] * ik;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float x = 0.f, o = 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          s[i][c] *= a;
          x += s[i][c] * kr[i];
        }
        const float d = b * ((float)v[g][c] - group_sum<16>(x));
#pragma unroll
        for (int i = 0; i < R; ++i) {
          s[i][c] += kr[i] * d;
          o += s[i][c] * (float)q[g][i];
        }
        o = group_sum<16>(o) * iq;
        keep[c] = rg == g ? (E)o : keep[c];
      }
    }
    if (rg < G && t + rg < eos) *reinterpret_cast<VV*>(op + (t + rg) * p.HV * VD) = keep;
  }
  if (p.ht) {
#pragma unroll
    for (int i = 0; i < R; ++i) *reinterpret_cast<VS*>(p.ht + sbase + i * VD) = s[i];
  }
}

// T tokens of the recurrence in fp32, 16 at a time. With S the state before the 16 tokens, a_t the decays,
// E_tj = a_{j+1} .. a_t and e_t = a_0 .. a_t (products, not exponentials of differences: exact for any decay):
//   x_t = beta_t (v_t - e_t k_t^T S),  delta_t = x_t - sum_{j<t} beta_t E_tj (k_t . k_j) delta_j,
//   o_t = e_t q_t^T S + sum_{j<=t} E_tj (q_t . k_j) delta_j,  S' = e_15 S + sum_j k_j E_15,j delta_j:
// the token-by-token recurrence with its sums in another order, every product in fp32. The contractions over K
// and over the tokens are v_mfma_f32_16x16x4_f32 (fp32 operands and accumulation, twice the rate of
// v_fma_f32); the triangular parts are summed in VALU code, where no token reads a later one (a NaN in a token
// does not reach those before it).
//   A workgroup owns 64 columns of one (sequence, value head); state waves 0-3 own 16 of them each: S [K x 16]
// stays in the accumulators (tile a: keys 16a + 4g + r, lane (g, i) column i), which are the B operands of K S
// and Q S as they stand. Helper waves prepare what does not depend on S, ahead of them: waves 4 and 5 the k and
// q rows of the tokens two steps ahead (normalised, fp32, in LDS; their loads a step earlier still), wave 6 the
// decays and the k.k coefficients of the next step, wave 7 its q.k coefficients. One barrier per 16 tokens.
//   The model's decays are at most 1, but the call takes any g. A product of decays past fp32's range would meet a zero
// (a zero state, a zero product of rows) as 0 * inf, and past a small state it overflows where the state itself does
// not. A sequence with 16 tokens whose positive log decays add up to more than kGrowth takes a token a step.
//   Rounding: the decays' products are formed in 64 bits (by the helpers) and rounded once, a step's update and
// what earlier tokens take from x are summed apart and added once, and the sums over K run in partial sums, so
// that the error against 64 bits is that of the token-by-token kernel before it (fp32, 500 tokens of K = 128: o
// 1.32e-7 against 1.34e-7, state 8.5e-8 against 9.3e-8). 16-bit outputs take two partial sums instead of four, which lets
// two workgroups run on a CU: 109 registers at K = 64, 128 with 4 spilled at K = 128 (16 sequences of 7 tokens 15.3 us
// against 18.4).
//   What bounds it: the 3 K / 4 fp32 MFMAs of a step (K = 128: 96 x 32 cycles a wave) and, for few sequences, the
// chain of a step (K S, x through LDS, the triangular solve, the update). bf16, 16 heads of 128: 16 sequences of 64
// tokens 37 us against 194 for the kernel before it (a token at a time, two barriers each); fp32, 2 sequences of
// 512 tokens 122 against 1390; 4 heads of 64, 256 tokens 46 against 384.
template <typename E, int KD, int VD>
__global__ __launch_bounds__(512, sizeof(E) == 4 ? 2 : 4) void gated_delta_recurrent_kernel(RecParams p) {
  constexpr int C = 16, A = KD / 16, KP = KD + 4, P = C + 4;  // 16-byte rows, spread over the banks
  constexpr int NP = sizeof(E) == 4 ? 4 : 2;
  __shared__ __align__(16) float kt[3][C * KP], qt[3][C * KP];
  __shared__ __align__(16) float cm[2][C * P], pm[2][C * P];  // cm[j][t] = beta_t E_tj k_t.k_j, pm[t][j] = E_tj q_t.k_j
  __shared__ __align__(16) float bs[2][C], es[2][C], ed[2][C];  // beta_t, e_t, E_15,j
  __shared__ __align__(16) float xs[4][C * P];                  // per state wave: x by column
  __shared__ int tokens;                                        // a step's tokens
  const int t = threadIdx.x, lane = t % kWave, w = __builtin_amdgcn_readfirstlane(t / kWave);
  const int li = lane % 16, g = lane / 16;
  constexpr int kSlices = VD / 64;
  const int hv = blockIdx.x / kSlices;
  const int64_t n = blockIdx.y;
  const int h = hv / (int)(p.HV / p.H);
  int64_t bos, eos;
  if (p.cu) {
    bos = load_index(p.cu, p.cu_i32, n);
    eos = load_index(p.cu, p.cu_i32, n + 1);
  } else {
    bos = n * p.T;
    eos = bos + p.T;
  }
  // Tokens a step: 16, or 1 where the decays of 16 tokens grow too far (a gate formed in the kernel is never positive).
  // Each helper wave looks at all of the sequence's log decays by itself, under its first loads: no exchange, no barrier.
  auto step_tokens = [&]() {
    bool up = false;
    auto raw_g = [&](int64_t at) { return at < eos ? load_raw32(p.g, p.dg, at * p.HV + hv) : 0u; };
    auto look = [&](uint32_t raw) {  // at 64 tokens, a step's in 16 lanes
      const float x = fmaxf(raw32_to_f32(raw, p.dg), 0.f);
      if (__any(x > 0.f)) up |= group_sum<C>(x) > kGrowth;
    };
    if (!(p.flags & GDN_FLAG_GATE_IN_KERNEL)) {
      look(raw_g(bos + lane));
      for (int64_t at = bos + kWave; at < eos; at += 4 * kWave) {
        uint32_t raw[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) raw[u] = raw_g(at + u * kWave + lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) look(raw[u]);
      }
    }
    return __any(up) ? 1 : C;
  };
  auto mm = [](float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); };
  auto ld4 = [](const float* x) { return *reinterpret_cast<const f32x4*>(x); };
  auto tok = [&](int64_t first, int c) {  // token c from `first` on; past the end the last token (its values are cleared)
    return first + c < eos ? first + c : eos - 1;
  };

  if (w < 4) {
    const int col = (blockIdx.x % kSlices) * 64 + w * 16 + li;
    const int64_t sbase = (n * p.HV + hv) * (int64_t)KD * VD + col;
    f32x4 s[A];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[a][r] = p.h0 ? p.h0[sbase + (16 * a + 4 * g + r) * VD] : 0.f;
    const E* __restrict__ vp = static_cast<const E*>(p.v) + (int64_t)hv * VD + col;
    E* __restrict__ op = static_cast<E*>(p.o) + (int64_t)hv * VD + col;
    E vr[4];
    if (bos < eos) {
#pragma unroll
      for (int r = 0; r < 4; ++r) vr[r] = vp[tok(bos, 4 * g + r) * p.HV * VD];
    }
    __syncthreads();
    const int L = __builtin_amdgcn_readfirstlane(tokens), steps = (int)((eos - bos + L - 1) / L);
    __syncthreads();
    for (int i = 0; i < steps; ++i) {
      const float* kl = kt[i % 3];
      const float* ql = qt[i % 3];
      const int li = opaque_int(lane % 16), g = opaque_int(lane / 16);  // addresses made here, not kept across steps
      const int64_t first = bos + (int64_t)i * L;
      const int b = i & 1, left = (int)(eos - first < L ? eos - first : L);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = 4 * g + r < left ? (float)vr[r] : 0.f;
      if (i + 1 < steps) {
#pragma unroll
        for (int r = 0; r < 4; ++r) vr[r] = vp[tok(first + L, 4 * g + r) * p.HV * VD];
      }
      f32x4 yp[NP]{}, zp[NP]{};  // K S and Q S in partial sums: lane (g, i) column i, tokens 4g + r
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const f32x4 kf = ld4(kl + li * KP + 16 * a + 4 * g), qf = ld4(ql + li * KP + 16 * a + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          yp[r % NP] = mm(kf[r], s[a][r], yp[r % NP]);
          zp[r % NP] = mm(qf[r], s[a][r], zp[r % NP]);
        }
        if (a % 2) __builtin_amdgcn_sched_barrier(0);  // the rows of two tiles in flight, not of all
      }
      f32x4 y = yp[0] + yp[1], z = zp[0] + zp[1];
      if constexpr (NP == 4) {
        y += yp[2] + yp[3];
        z += zp[2] + zp[3];
      }
      __builtin_amdgcn_sched_barrier(0);
      const f32x4 eg = ld4(es[b] + 4 * g), bg = ld4(bs[b] + 4 * g);
      f32x4 x[4];  // x, then delta, of this lane's column: all 16 tokens
      {
        f32x4 xg;
#pragma unroll
        for (int r = 0; r < 4; ++r) xg[r] = 4 * g + r < left ? bg[r] * (v[r] - eg[r] * y[r]) : 0.f;  // y may be 0 * inf
        *reinterpret_cast<f32x4*>(xs[w] + li * P + 4 * g) = xg;
        __builtin_amdgcn_wave_barrier();  // the wave reads its own writes (LDS operations of a wave are in order)
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = ld4(xs[w] + li * P + 4 * u);
      }
      f32x4 sub[4]{};  // what the earlier tokens take from x: summed apart, so that x is rounded once
#pragma unroll
      for (int j = 0; j < C; ++j) {
        x[j / 4][j % 4] -= sub[j / 4][j % 4];  // now delta of token j
#pragma unroll
        for (int u = (j + 1) / 4; u < 4; ++u) {
          const f32x4 c = ld4(cm[b] + j * P + 4 * u);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * u + r > j) sub[u][r] += c[r] * x[j / 4][j % 4];
        }
        if (j % 4 == 4 - 1) __builtin_amdgcn_sched_barrier(0);
      }
      f32x4 dg;  // delta of the tokens 4g + r
#pragma unroll
      for (int r = 0; r < 4; ++r) dg[r] = g < 2 ? (g == 0 ? x[0][r] : x[1][r]) : (g == 2 ? x[2][r] : x[3][r]);
      const f32x4 edg = ld4(ed[b] + 4 * g);
      f32x4 db;
      const float last = es[b][C - 1];
#pragma unroll
      for (int r = 0; r < 4; ++r) db[r] = dg[r] * edg[r];
#pragma unroll
      for (int a = 0; a < A; ++a) {
        f32x4 u{};  // summed apart and added once: one rounding of the state per step
#pragma unroll
        for (int r = 0; r < 4; ++r) u = mm(kl[(4 * g + r) * KP + 16 * a + li], db[r], u);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[a][r] = s[a][r] * last + u[r];
        if (a % 2) __builtin_amdgcn_sched_barrier(0);
      }
      f32x4 o{};
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (u < g) {  // tokens of earlier quads
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const f32x4 pr = ld4(pm[b] + (4 * g + r) * P + 4 * u);
            o[r] += (pr[0] * x[u][0] + pr[1] * x[u][1]) + (pr[2] * x[u][2] + pr[3] * x[u][3]);
          }
        }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const f32x4 pr = ld4(pm[b] + (4 * g + r) * P + 4 * g);
#pragma unroll
        for (int j = 0; j <= r; ++j) o[r] += pr[j] * dg[j];
        o[r] += eg[r] * z[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * g + r < left) op[(first + 4 * g + r) * p.HV * VD] = (E)o[r];
      __syncthreads();
    }
    if (p.ht) {
#pragma unroll
      for (int a = 0; a < A; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) p.ht[sbase + (16 * a + 4 * g + r) * VD] = s[a][r];
    }
  } else if (w < 6) {  // k and q rows: 8 threads per token, KD / 8 elements each
    constexpr int R = KD / 8;
    using VK = typename RowVec<E, R>::T;
    const int row = (t - 256) / 8, pos = (t % 8) * R;
    const E* __restrict__ kp = static_cast<const E*>(p.k) + (int64_t)h * KD + pos;
    const E* __restrict__ qp = static_cast<const E*>(p.q) + (int64_t)h * KD + pos;
    const bool l2 = p.flags & GDN_FLAG_QK_L2NORM;
    VK kr{}, qr{};
    auto load = [&](int64_t first) {
      kr = *reinterpret_cast<const VK*>(kp + tok(first, row) * p.H * KD);
      qr = *reinterpret_cast<const VK*>(qp + tok(first, row) * p.H * KD);
    };
    if (bos < eos) load(bos);
    const int L = step_tokens(), steps = (int)((eos - bos + L - 1) / L);
    for (int i = -2; i < steps; ++i) {
      if (i + 2 < steps) {  // F.normalize: x / max(|x|, 1e-12); q times the scale; zeros past the end
        const bool live = row < L && bos + (int64_t)(i + 2) * L + row < eos;
        float kf[R], qf[R], kk = 0.f, qq = 0.f;
#pragma unroll
        for (int e = 0; e < R; ++e) {
          kf[e] = live ? (float)kr[e] : 0.f;
          qf[e] = live ? (float)qr[e] : 0.f;
          kk += kf[e] * kf[e];
          qq += qf[e] * qf[e];
        }
        float ks = 1.f, qs = p.scale;
        if (l2) {
          ks = 1.f / fmaxf(sqrtf(group_sum<8>(kk)), 1e-12f);
          qs = p.scale / fmaxf(sqrtf(group_sum<8>(qq)), 1e-12f);
        }
        float* kl = kt[(i + 2) % 3] + row * KP + pos;
        float* ql = qt[(i + 2) % 3] + row * KP + pos;
#pragma unroll
        for (int e = 0; e < R; e += 4) {
          *reinterpret_cast<f32x4*>(kl + e) = f32x4{kf[e] * ks, kf[e + 1] * ks, kf[e + 2] * ks, kf[e + 3] * ks};
          *reinterpret_cast<f32x4*>(ql + e) = f32x4{qf[e] * qs, qf[e + 1] * qs, qf[e + 2] * qs, qf[e + 3] * qs};
        }
        if (i + 3 < steps) load(bos + (int64_t)(i + 3) * L);
      }
      __syncthreads();
    }
  } else {  // coefficients of the next step: wave 6 k.k (with beta), wave 7 q.k
    uint32_t graw = 0, braw = 0;
    auto load = [&](int64_t first) {
      graw = load_raw32(p.g, p.dg, tok(first, li) * p.HV + hv);
      if (w == 6) braw = load_raw32(p.beta, p.db, tok(first, li) * p.HV + hv);
    };
    const float neg_a = p.flags & GDN_FLAG_GATE_IN_KERNEL ? -expf(p.A_log[hv]) : 0.f;
    const float dtb = p.flags & GDN_FLAG_GATE_IN_KERNEL ? p.dt_bias[hv] : 0.f;
    if (bos < eos) load(bos);
    const int L = step_tokens(), steps = (int)((eos - bos + L - 1) / L);
    if (t == 6 * kWave) tokens = L;
    __syncthreads();
    for (int i = 0; i <= steps; ++i) {  // step i, while the state waves work on step i - 1
      if (i < steps) {
        const int b = i & 1;
        const bool live = li < L && bos + (int64_t)i * L + li < eos;
        float gv = raw32_to_f32(graw, p.dg), bv = raw32_to_f32(braw, p.db);
        if (p.flags & GDN_FLAG_GATE_IN_KERNEL) gv = neg_a * softplus_f32(gv + dtb);
        if (p.flags & GDN_FLAG_BETA_SIGMOID) bv = sigmoid_f32(bv);
        const double av = live ? exp((double)gv) : 1.0;  // decays in 64 bits up to the products that leave here
        bv = live ? bv : 0.f;
        if (i + 1 < steps) load(bos + (int64_t)(i + 1) * L);
        const float* kl = kt[i % 3] + li * KP + 4 * g;
        const float* rl = w == 6 ? kl : qt[i % 3] + li * KP + 4 * g;
        f32x4 dp[8]{};  // lane (g, j): rows (tokens) 4g + r, column (earlier token) j
#pragma unroll
        for (int a = 0; a < A; a += 2) {
          const f32x4 k0 = ld4(kl + 16 * a), r0 = ld4(rl + 16 * a), k1 = ld4(kl + 16 * a + 16), r1 = ld4(rl + 16 * a + 16);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            dp[r] = mm(r0[r], k0[r], dp[r]);
            dp[4 + r] = mm(r1[r], k1[r], dp[4 + r]);
          }
          __builtin_amdgcn_sched_barrier(0);  // the rows of two tiles in flight: 128 registers have to do
        }
        const int lo = opaque_int(li), go = opaque_int(g);  // compared 32 times: no masks kept across the loop
        double e = 1.0, ei = 1.0;  // E_mj while m runs; e_t of token li: rounded to fp32 once
        f32x4 eg{};
#pragma unroll
        for (int m = 0; m < C; ++m) {
          const uint64_t bits = __builtin_bit_cast(uint64_t, av);
          const double am = __builtin_bit_cast(double, (uint64_t)__builtin_amdgcn_readlane((uint32_t)(bits >> 32), m) << 32 |
                                                           (uint32_t)__builtin_amdgcn_readlane((uint32_t)bits, m));
          e *= m > lo ? am : 1.0;
          if (w == 6) ei *= m <= lo ? am : 1.0;
          eg[m % 4] = m / 4 == go ? (float)e : eg[m % 4];
        }
        const f32x4 d = ((dp[0] + dp[1]) + (dp[2] + dp[3])) + ((dp[4] + dp[5]) + (dp[6] + dp[7]));
        if (w == 6) {
          f32x4 c;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float bt = __shfl(bv, 4 * g + r, kWave);
            c[r] = 4 * g + r > li ? bt * eg[r] * d[r] : 0.f;
          }
          *reinterpret_cast<f32x4*>(cm[b] + li * P + 4 * g) = c;
          if (g == 0) {
            bs[b][li] = bv;
            es[b][li] = (float)ei;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) pm[b][(4 * g + r) * P + li] = 4 * g + r >= li ? eg[r] * d[r] : 0.f;
          if (g == 0) ed[b][li] = (float)e;
        }
      }
      __syncthreads();
    }
  }
}

struct DecodeParams {
  const void* x;
  void* conv_state;
  const float* conv_w;
  const void *g, *beta;
  float* state;
  void* o;
  int64_t H, HV, W;
  int dx, dcs, dg, db;
  float scale;
  unsigned flags;
  const float *A_log, *dt_bias;
};

// Conv-cache update + conv + SiLU of channel ch of batch row b; returns the activation rounded to
// the activation dtype (as a separate conv kernel would store it).
__device__ __forceinline__ float decode_conv_channel(const DecodeParams& p, int64_t b, int64_t C, int64_t ch) {
  // window = (state[1..W-1], x); y = sum_i w[ch, i] window[i]; the new state is the window.
  const int64_t cbase = (b * C + ch) * p.W;
  float acc = 0.f;
  for (int i = 1; i < p.W; ++i) {
    const float xi = load_as_f32(p.conv_state, p.dcs, cbase + i);
    acc += p.conv_w[ch * p.W + i - 1] * xi;
    store_from_f32(p.conv_state, p.dcs, cbase + i - 1, xi);  // index i-1 was read one step earlier
  }
  const float xc = load_as_f32(p.x, p.dx, b * C + ch);
  acc += p.conv_w[ch * p.W + p.W - 1] * xc;
  store_from_f32(p.conv_state, p.dcs, cbase + p.W - 1, xc);
  return round_to(p.dx, silu_f32(acc));
}

// grid (H, B): one workgroup per (q/k head, batch row). It computes the q/k conv of its head once
// (so the shared conv cache of q/k is written by exactly one workgroup) and then updates the
// HV/H value heads that read this q/k head, one after the other.
template <int D>
__global__ __launch_bounds__(256) void gated_delta_decode_kernel(DecodeParams p) {
  using L = RecLayout<D, D>;
  __shared__ float qk[2 * D];
  __shared__ float vs[2][D];
  __shared__ float red[2][L::NW * L::CG * 12];
  const int h = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int rep = (int)(p.HV / p.H);
  const int64_t C = (2 * p.H + p.HV) * D;
  const int t = threadIdx.x;
  for (int e = t; e < 2 * D; e += L::NT) {
    const int64_t ch = (e < D) ? (int64_t)h * D + e : p.H * D + (int64_t)h * D + (e - D);
    qk[e] = decode_conv_channel(p, b, C, ch);
  }
  const bool l2 = p.flags & GDN_FLAG_QK_L2NORM;
  for (int r = 0; r < rep; ++r) {
    const int hv = h * rep + r;
    const int par = r & 1;
    const int64_t sbase = (b * p.HV + hv) * (int64_t)D * D;
    StateRegs<D, D> s;
    load_state<D, D>(s, p.state + sbase);
    for (int e = t; e < D; e += L::NT) vs[par][e] = decode_conv_channel(p, b, C, 2 * p.H * D + (int64_t)hv * D + e);
    RecParams gp{};
    gp.g = p.g; gp.beta = p.beta; gp.dg = p.dg; gp.db = p.db; gp.flags = p.flags;
    gp.A_log = p.A_log; gp.dt_bias = p.dt_bias;
    float a, bb;
    gate_values(gp, b * p.HV + hv, hv, a, bb);
    __syncthreads();
    float o4[4];
    rec_token<D, D>(s, qk, qk + D, vs[par], a, bb, l2, p.scale, red[par], o4);
    if (t < L::CG) {
      const int64_t ob = (b * p.HV + hv) * D + 4 * t;
#pragma unroll
      for (int c = 0; c < 4; ++c) store_from_f32(p.o, p.dx, ob + c, o4[c]);
    }
    store_state<D, D>(s, p.state + sbase);
  }
}


template <class T>
__device__ __forceinline__ float elem_to_f32(T x) { return static_cast<float>(x); }
template <class T>
__device__ __forceinline__ T f32_to_elem(float x) { return static_cast<T>(x); }

// Width-W conv cache of one channel as one vector access (W * sizeof(T) bytes).
template <int W, class T>
struct alignas(W * sizeof(T) >= 16 ? 16 : W * sizeof(T)) ConvWindow {
  T v[W];
};

// Sum over the 8 row groups of a column group (lanes l ^ 8, l ^ 16, l ^ 32) in three VALU steps:
// DPP row_ror:8 inside each 16-lane row, then the 16- and 32-lane swaps of gfx950
__device__ __forceinline__ float rg_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));
  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// Fast decode step for width-4 conv caches whose dtype equals the activation dtype T: one
// workgroup per (sequence, q/k head), looping over that head's value heads. Wave w owns the 32-column
// block w of the state (columns of the recurrence are independent: column j needs only S[:, j]), 16
// rows x 4 columns per lane, so the reductions over the state's rows (S^T k, S^T q) stay inside the
// wave and no reduction crosses waves: one barrier per value head publishes the conv outputs q, k, v
// in LDS. The four waves read their blocks at once, i.e. the whole 64 KB state, with non-temporal
// loads and write it back with non-temporal stores: the state is touched once per step, and with
// the state served from DRAM (B = 64, H = 16, D = 128) the step took 25.0 us this way against
// 29.0 us for cached accesses in column blocks.
template <int D, class T>
__global__ __launch_bounds__(256) void gated_delta_decode_w4_kernel(DecodeParams p) {
  constexpr int W = 4, VB = 32, NWB = D / VB;                // column blocks, one per wave (waves 0..NWB-1)
  constexpr int CG = VB / 4, RG = kWave / CG, RPT = D / RG;  // lane (rg, cg): rows rg + RG i, columns 4cg..+3
  using Win = ConvWindow<W, T>;
  __shared__ float qk[2 * D];
  __shared__ float vs[2][D];
  const int h = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int rep = (int)(p.HV / p.H);
  const int64_t C = (2 * p.H + p.HV) * D;
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave, cg = lane % CG, rg = lane / CG;
  const T* __restrict__ xg = static_cast<const T*>(p.x);
  Win* __restrict__ cs = static_cast<Win*>(p.conv_state);
  const float4* __restrict__ wg = reinterpret_cast<const float4*>(p.conv_w);
  const bool l2 = p.flags & GDN_FLAG_QK_L2NORM;
  const bool has_qk = t < 2 * D, has_v = t < D;
  const int64_t ch_qk = (t < D) ? (int64_t)h * D + t : p.H * D + (int64_t)h * D + (t - D);

  for (int r = 0; r < rep; ++r) {
    const int hv = h * rep + r;
    const int par = r & 1;
    const int64_t sbase = (b * p.HV + hv) * (int64_t)D * D;
    const int64_t ch_v = 2 * p.H * D + (int64_t)hv * D + t;
    // The state first, so that the step's 64 KB per head is in flight before the conv window and
    // gate loads: through a buffer resource (one lane offset plus a scalar offset per row step, so
    // the 16 row addresses take no registers), non-temporal (the state is touched once a step).
    float4 s[RPT];
    const auto rs = make_rsrc(p.state + sbase, (uint32_t)(D * D * 4));
    const int voff = ((rg * D) + w * VB + 4 * cg) * 4;
    if (w < NWB) {
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, i * RG * D * 4, 2);
        s[i] = __builtin_bit_cast(float4, x);
      }
    }
    Win wq{}, wv{};
    T xq{}, xv{};
    float4 kq{}, kv{};
    const bool do_qk = has_qk && r == 0;
    if (do_qk) {
      wq = cs[b * C + ch_qk];
      xq = xg[b * C + ch_qk];
      kq = wg[ch_qk];
    }
    if (has_v) {
      wv = cs[b * C + ch_v];
      xv = xg[b * C + ch_v];
      kv = wg[ch_v];
    }
    const uint32_t graw = load_raw32(p.g, p.dg, b * p.HV + hv);
    const uint32_t braw = load_raw32(p.beta, p.db, b * p.HV + hv);
    if (do_qk) {
      const float y = kq.x * elem_to_f32(wq.v[1]) + kq.y * elem_to_f32(wq.v[2]) + kq.z * elem_to_f32(wq.v[3]) +
                      kq.w * elem_to_f32(xq);
      Win nw;
      nw.v[0] = wq.v[1]; nw.v[1] = wq.v[2]; nw.v[2] = wq.v[3]; nw.v[3] = xq;
      cs[b * C + ch_qk] = nw;
      qk[t] = elem_to_f32(f32_to_elem<T>(silu_f32(y)));
    }
    if (has_v) {
      const float y = kv.x * elem_to_f32(wv.v[1]) + kv.y * elem_to_f32(wv.v[2]) + kv.z * elem_to_f32(wv.v[3]) +
                      kv.w * elem_to_f32(xv);
      Win nw;
      nw.v[0] = wv.v[1]; nw.v[1] = wv.v[2]; nw.v[2] = wv.v[3]; nw.v[3] = xv;
      cs[b * C + ch_v] = nw;
      vs[par][t] = elem_to_f32(f32_to_elem<T>(silu_f32(y)));
    }
    float gv = raw32_to_f32(graw, p.dg), bv = raw32_to_f32(braw, p.db);
    if (p.flags & GDN_FLAG_GATE_IN_KERNEL) gv = -expf(p.A_log[hv]) * softplus_f32(gv + p.dt_bias[hv]);
    if (p.flags & GDN_FLAG_BETA_SIGMOID) bv = sigmoid_f32(bv);
    const float a = expf(gv);
    __syncthreads();
    if (w < NWB) {
      const float* q_l = qk;
      const float* k_l = qk + D;
      float pr[11];
#pragma unroll
      for (int j2 = 0; j2 < 11; ++j2) pr[j2] = 0.f;
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const int row = rg + RG * i;
        const float kr = k_l[row], qr = q_l[row];
        pr[0] += s[i].x * kr; pr[1] += s[i].y * kr; pr[2] += s[i].z * kr; pr[3] += s[i].w * kr;
        pr[4] += s[i].x * qr; pr[5] += s[i].y * qr; pr[6] += s[i].z * qr; pr[7] += s[i].w * qr;
        pr[8] += kr * qr; pr[9] += kr * kr; pr[10] += qr * qr;
      }
#pragma unroll
      for (int j2 = 0; j2 < 11; ++j2) pr[j2] = rg_sum(pr[j2]);
      const float ik = l2 ? 1.f / fmaxf(sqrtf(pr[9]), 1e-12f) : 1.f;
      const float iq = l2 ? 1.f / fmaxf(sqrtf(pr[10]), 1e-12f) : 1.f;
      const float* v_l = vs[par] + w * VB + 4 * cg;
      float d[4], o4[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        d[c] = bv * (v_l[c] - a * pr[c] * ik);
        o4[c] = p.scale * (a * pr[4 + c] * iq + d[c] * pr[8] * ik * iq);
      }
      if (rg == 0) {
        T* og = static_cast<T*>(p.o) + (b * p.HV + hv) * D + w * VB + 4 * cg;
#pragma unroll
        for (int c = 0; c < 4; ++c) og[c] = f32_to_elem<T>(o4[c]);
      }
      // the row step goes into the lane offset, not the scalar offset: for a wide buffer store whose
      // scalar offset is a register the compiler inserts no wait states before the store's data
      // registers are rewritten, and the last lanes of a row then stored the rewritten values
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const float kr = k_l[rg + RG * i] * ik;
        const float4 n{a * s[i].x + kr * d[0], a * s[i].y + kr * d[1], a * s[i].z + kr * d[2], a * s[i].w + kr * d[3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, n), rs, voff + i * RG * D * 4, 0, 2);
      }
    }
  }
}

}  // namespace gdn

using namespace gdn;

static int check_dims(int64_t K, int64_t V) {
  if ((K != 64 && K != 128) || (V != 64 && V != 128)) {
    gdn_internal_set_error("head dims K=%lld V=%lld unsupported (each must be 64 or 128)", (long long)K, (long long)V);
    return GDN_ERR_UNSUPPORTED;
  }
  return GDN_OK;
}

extern "C" int gdn_recurrent_fwd(const void* q, const void* k, const void* v, const void* g, const void* beta,
                                 const float* initial_state, void* o, float* final_state, const void* cu_seqlens,
                                 int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V, int64_t N,
                                 int qkv_dtype, int g_dtype, int beta_dtype, float scale, unsigned flags,
                                 const float* A_log, const float* dt_bias, void* stream) {
  if (!q || !k || !v || !g || !beta || !o) {
    gdn_internal_set_error("gdn_recurrent_fwd: null tensor pointer");
    return GDN_ERR_INVALID;
  }
  if (B <= 0 || T < 0 || H <= 0 || HV <= 0 || HV % H || N <= 0) {
    gdn_internal_set_error("gdn_recurrent_fwd: bad sizes B=%lld T=%lld H=%lld HV=%lld N=%lld", (long long)B,
                           (long long)T, (long long)H, (long long)HV, (long long)N);
    return GDN_ERR_INVALID;
  }
  if (cu_seqlens ? B != 1 : N != B) {
    gdn_internal_set_error("gdn_recurrent_fwd: cu_seqlens requires B == 1 (and N == B without it)");
    return GDN_ERR_INVALID;
  }
  if ((flags & GDN_FLAG_GATE_IN_KERNEL) && (!A_log || !dt_bias)) {
    gdn_internal_set_error("gdn_recurrent_fwd: gate in kernel needs A_log and dt_bias");
    return GDN_ERR_INVALID;
  }
  if (int rc = check_dims(K, V)) return rc;
  if (N > 65535) {
    gdn_internal_set_error("gdn_recurrent_fwd: N=%lld exceeds the grid limit 65535", (long long)N);
    return GDN_ERR_UNSUPPORTED;
  }
  RecParams p{q, k, v, g, beta, initial_state, o, final_state, cu_seqlens, (flags & GDN_FLAG_CU_INT32) ? 1 : 0,
              T, H, HV, qkv_dtype, g_dtype, beta_dtype, scale, flags, A_log, dt_bias};
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Few tokens a sequence: the 16-token steps would be mostly padding. bf16, 16 heads of 128, us at 3 / 5 / 8 / 12
  // tokens in the short kernel and in the 16-token one: 1 sequence 5.9 / 7.5 / 9.3 / 12.0 and 8.5; 16 sequences
  // 11.1 / 13.8 / 16.6 / 21.7 and 15.3; 64 sequences 27.4 / 32.3 / 40.5 / 55.2 and 42 (heads of 64: 11.3 / 14.8 / 17.8
  // / 22.8 and 17.5). The line is at 4 tokens, at 6 from 512 waves of 64 columns up and at 8 from 1,024 up, where
  // the state's bytes set the time of either. The mean length decides, as the host does not read cu_seqlens: one long
  // sequence among many of one token may take the short kernel, at 0.7 us a token.
  const int64_t tokens = cu_seqlens ? T : B * T, cols = N * HV * V;
  const bool few = tokens <= (cols >= 65536 ? 8 : cols >= 32768 ? 6 : kShortTokens) * N;
  auto go = [&](auto e_tag, auto k_c, auto v_c) {
    constexpr int KD = decltype(k_c)::value, VD = decltype(v_c)::value;
    const dim3 grid((unsigned)(HV * (VD / 64)), (unsigned)N);
    if (few) hipLaunchKernelGGL((gated_delta_recurrent_short_kernel<decltype(e_tag), KD, VD>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((gated_delta_recurrent_kernel<decltype(e_tag), KD, VD>), grid, dim3(512), 0, s, p);
  };
  auto by_dims = [&](auto e_tag) {
    using C64 = std::integral_constant<int, 64>;
    using C128 = std::integral_constant<int, 128>;
    if (K == 128 && V == 128) go(e_tag, C128{}, C128{});
    else if (K == 64 && V == 64) go(e_tag, C64{}, C64{});
    else if (K == 128) go(e_tag, C128{}, C64{});
    else go(e_tag, C64{}, C128{});
  };
  if (qkv_dtype == GDN_DTYPE_BF16) by_dims(bf16{});
  else if (qkv_dtype == GDN_DTYPE_F16) by_dims(f16{});
  else by_dims(float{});
  return gdn_internal_check_launch("gated_delta_recurrent_kernel");
}

extern "C" int gdn_decode_step(const void* x_qkv, void* conv_state, const float* conv_weight, const void* g,
                               const void* beta, float* state, void* o, int64_t B, int64_t H, int64_t HV, int64_t D,
                               int64_t W, int x_dtype, int conv_state_dtype, int g_dtype, int beta_dtype, float scale,
                               unsigned flags, const float* A_log, const float* dt_bias, void* stream) {
  if (!x_qkv || !conv_state || !conv_weight || !g || !beta || !state || !o) {
    gdn_internal_set_error("gdn_decode_step: null tensor pointer");
    return GDN_ERR_INVALID;
  }
  if (B <= 0 || H <= 0 || HV <= 0 || HV % H || W < 1 || W > 16) {
    gdn_internal_set_error("gdn_decode_step: bad sizes B=%lld H=%lld HV=%lld W=%lld", (long long)B, (long long)H,
                           (long long)HV, (long long)W);
    return GDN_ERR_INVALID;
  }
  if (D != 64 && D != 128) {
    gdn_internal_set_error("gdn_decode_step: head dim %lld unsupported (64 or 128)", (long long)D);
    return GDN_ERR_UNSUPPORTED;
  }
  if ((flags & GDN_FLAG_GATE_IN_KERNEL) && (!A_log || !dt_bias)) {
    gdn_internal_set_error("gdn_decode_step: gate in kernel needs A_log and dt_bias");
    return GDN_ERR_INVALID;
  }
  if (B > 65535) {
    gdn_internal_set_error("gdn_decode_step: B=%lld exceeds the grid limit 65535", (long long)B);
    return GDN_ERR_UNSUPPORTED;
  }
  DecodeParams p{x_qkv, conv_state, conv_weight, g, beta, state, o, H, HV, W, x_dtype, conv_state_dtype,
                 g_dtype, beta_dtype, scale, flags, A_log, dt_bias};
  dim3 grid((unsigned)H, (unsigned)B), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (W == 4 && conv_state_dtype == x_dtype) {  // vectorised width-4 path
#define GDN_DECODE_W4(D_, T_) hipLaunchKernelGGL((gated_delta_decode_w4_kernel<D_, T_>), grid, block, 0, s, p)
    if (x_dtype == GDN_DTYPE_BF16) { if (D == 128) GDN_DECODE_W4(128, bf16); else GDN_DECODE_W4(64, bf16); }
    else if (x_dtype == GDN_DTYPE_F16) { if (D == 128) GDN_DECODE_W4(128, f16); else GDN_DECODE_W4(64, f16); }
    else { if (D == 128) GDN_DECODE_W4(128, float); else GDN_DECODE_W4(64, float); }
#undef GDN_DECODE_W4
    return gdn_internal_check_launch("gated_delta_decode_w4_kernel");
  }
  if (D == 128) hipLaunchKernelGGL((gated_delta_decode_kernel<128>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gated_delta_decode_kernel<64>), grid, block, 0, s, p);
  return gdn_internal_check_launch("gated_delta_decode_kernel");
}
