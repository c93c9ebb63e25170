// Row-wise epilogue/prologue norms: L2 normalisation (q/k) and gated RMSNorm (GDN output).
//
// One wave per row (rows of D = 64 or 128 elements in the GDN path, any D here): each lane reads
// D/64 elements, the sum of squares is reduced across the wave, and the row is written once with
// fp32 math and a single rounding. Both kernels are HBM-bound elementwise passes.

#include <type_traits>

#include "gdn_chunk.h"

namespace gdn {

struct NormParams {
  const void* x;
  const void* gate;
  const float* w;
  const float* bias;
  void* y;
  int64_t rows, D;
  int dt, act;
  float eps;
  int mode;   // 0 = L2 norm, 1 = (gated) RMSNorm, 2 = L2 norm as the chunk kernels form it (vector path only)
  int split;  // RMSNorm with a gate: the norm (w, bias) and act(gate) each rounded before their product
  const void* x2;  // a second tensor of the same rows, normalised by the blocks with blockIdx.y = 1
  void* y2;
};

constexpr int kNormMaxPerLane = 16;  // D <= 1024

__global__ __launch_bounds__(256) void gated_delta_norm_kernel(NormParams p) {
  if (blockIdx.y) {
    p.x = p.x2;
    p.y = p.y2;
  }
  const int lane = threadIdx.x % kWave;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
  for (int64_t r = wave; r < p.rows; r += nwaves) {
    const int64_t base = r * p.D;
    float xv[kNormMaxPerLane];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kNormMaxPerLane; ++j) {
      const int64_t e = lane + (int64_t)j * kWave;
      xv[j] = e < p.D ? load_as_f32(p.x, p.dt, base + e) : 0.f;
      ss += xv[j] * xv[j];
    }
    ss = wave_xor_sum(ss, 1);
    float scale;
    if (p.mode == 0) scale = 1.f / fmaxf(sqrtf(ss), p.eps);  // F.normalize: x / max(||x||, eps)
    else scale = 1.f / sqrtf(ss / (float)p.D + p.eps);  // RMSNorm: rsqrt(mean(x^2) + eps)
#pragma unroll
    for (int j = 0; j < kNormMaxPerLane; ++j) {
      const int64_t e = lane + (int64_t)j * kWave;
      if (e >= p.D) break;
      float out = xv[j] * scale;
      if (p.mode == 1) {
        if (p.w) out *= p.w[e];
        if (p.bias) out += p.bias[e];
        if (p.gate) {
          const float gv = load_as_f32(p.gate, p.dt, base + e);
          const float a = (p.act == GDN_ACT_SILU) ? silu_f32(gv) : gv;
          out = p.split ? round_to(p.dt, out) * round_to(p.dt, a) : out * a;
        }
      }
      store_from_f32(p.y, p.dt, base + e, out);
    }
  }
}

// Vector path of the same two norms for 16-bit rows of D = 64 or 128: LPR = D / 8 lanes per row,
// each lane one 16-byte chunk of x (and of the gate), so a wave covers 64 / LPR rows with
// 16-byte loads and stores; the sum of squares is reduced inside the row's lane group by DPP.
// Each wave takes kNormV8Groups row groups per pass and issues all their loads before the first
// use (memory-level parallelism for an HBM-bound pass). fp32 math, one rounding; the RMS factor is
// v_rsq_f32 (the reference computes it with torch.rsqrt).
constexpr int kNormV8Groups = 4;

template <typename E, int LPR>
__global__ __launch_bounds__(256) void gated_delta_norm_v8_kernel(NormParams p) {
  if (blockIdx.y) {
    p.x = p.x2;
    p.y = p.y2;
  }
  typedef E V8 __attribute__((ext_vector_type(8)));
  constexpr int RPW = kWave / LPR, U = kNormV8Groups;
  const int lane = threadIdx.x % kWave, sub = lane / LPR, li = lane % LPR;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
  const bool gated = p.mode == 1 && p.gate;
  float wv[8], bv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    wv[e] = (p.mode == 1 && p.w) ? p.w[li * 8 + e] : 1.f;
    bv[e] = (p.mode == 1 && p.bias) ? p.bias[li * 8 + e] : 0.f;
  }
  for (int64_t r0 = wave * RPW * U; r0 < p.rows; r0 += nwaves * RPW * U) {
    V8 xv[U], gv[U];
    int64_t base[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // every lane loads (clamped rows): the reductions need all lanes
      const int64_t r = r0 + u * RPW + sub;
      base[u] = (r < p.rows ? r : p.rows - 1) * p.D + li * 8;
      xv[u] = *reinterpret_cast<const V8*>(static_cast<const E*>(p.x) + base[u]);
      if (gated) gv[u] = *reinterpret_cast<const V8*>(static_cast<const E*>(p.gate) + base[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float xf[8], ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xf[e] = (float)xv[u][e];
        ss += xf[e] * xf[e];
      }
      ss = group_sum<LPR>(ss);
      const float scale = p.mode == 0   ? 1.f / fmaxf(sqrtf(ss), p.eps)
                          : p.mode == 2 ? __builtin_amdgcn_rsqf(fmaxf(ss, 1e-24f))  // as l2norm_row_chunks, its sums too
                                        : __builtin_amdgcn_rsqf(ss / (float)p.D + p.eps);
      V8 yv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float out = xf[e] * scale;
        if (p.mode == 1) {
          out = out * wv[e] + bv[e];
          if (gated) {
            const float g = (float)gv[u][e];
            const float a = (p.act == GDN_ACT_SILU) ? silu_fast(g) : g;
            out = p.split ? (float)(E)out * (float)(E)a : out * a;
          }
        }
        yv[e] = (E)out;
      }
      if (r0 + u * RPW + sub < p.rows) *reinterpret_cast<V8*>(static_cast<E*>(p.y) + base[u]) = yv;
    }
  }
}

// Backward of both norms, one wave per row (the reference trains through F.normalize and through
// RMSNorm * silu(gate) by autograd, sore/model/gdn.py:177,180-188; FLA's fused l2norm and
// rms_norm_gated kernels have their own backward):
//   L2:  y = x / max(|x|, eps):          dx = (dy - y (y . dy)) / |x|   (dy / eps where |x| <= eps)
//   RMS: n = x r, r = rsqrt(mean(x^2) + eps), u = n w + b, y = u act(g):
//        du = dy act(g), dg = dy u act'(g), dx = r (du w) - x r^3 mean((du w) x),
//        dw = sum_rows du n, db = sum_rows du  (per-wave partial sums, reduced by a second kernel).
struct NormBwdParams {
  const void* x;
  const void* gate;
  const float* w;
  const float* bias;
  const void* dy;
  void* dx;
  void* dgate;
  float* part;  // [waves][2][D] partial dw, db (RMS mode)
  int64_t rows, D;
  int dt, act;
  float eps;
  int mode;
};

__global__ __launch_bounds__(256) void gated_delta_norm_bwd_kernel(NormBwdParams p) {
  const int lane = threadIdx.x % kWave;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
  float pw[kNormMaxPerLane], pb[kNormMaxPerLane];
#pragma unroll
  for (int j = 0; j < kNormMaxPerLane; ++j) pw[j] = pb[j] = 0.f;
  for (int64_t r = wave; r < p.rows; r += nwaves) {
    const int64_t base = r * p.D;
    float xv[kNormMaxPerLane], dv[kNormMaxPerLane];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kNormMaxPerLane; ++j) {
      const int64_t e = lane + (int64_t)j * kWave;
      xv[j] = e < p.D ? load_as_f32(p.x, p.dt, base + e) : 0.f;
      dv[j] = e < p.D ? load_as_f32(p.dy, p.dt, base + e) : 0.f;
      ss += xv[j] * xv[j];
    }
    ss = wave_xor_sum(ss, 1);
    if (p.mode == 0) {
      const float nrm = sqrtf(ss), inv = 1.f / fmaxf(nrm, p.eps);
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < kNormMaxPerLane; ++j) dot += xv[j] * inv * dv[j];
      dot = nrm > p.eps ? wave_xor_sum(dot, 1) : 0.f;
#pragma unroll
      for (int j = 0; j < kNormMaxPerLane; ++j) {
        const int64_t e = lane + (int64_t)j * kWave;
        if (e >= p.D) continue;
        store_from_f32(p.dx, p.dt, base + e, (dv[j] - xv[j] * inv * dot) * inv);
      }
    } else {
      const float rr = 1.f / sqrtf(ss / (float)p.D + p.eps);
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < kNormMaxPerLane; ++j) {
        const int64_t e = lane + (int64_t)j * kWave;
        if (e >= p.D) continue;
        const float n = xv[j] * rr, wv = p.w ? p.w[e] : 1.f;
        float du = dv[j];
        if (p.gate) {
          const float gv = load_as_f32(p.gate, p.dt, base + e);
          const float u = n * wv + (p.bias ? p.bias[e] : 0.f);
          float act = gv, dact = 1.f;
          if (p.act == GDN_ACT_SILU) {
            const float sg = sigmoid_f32(gv);
            act = gv * sg;
            dact = sg * (1.f + gv * (1.f - sg));
          }
          store_from_f32(p.dgate, p.dt, base + e, du * u * dact);
          du *= act;
        }
        pw[j] += du * n;
        pb[j] += du;
        dv[j] = du * wv;  // dn
        dot += dv[j] * xv[j];
      }
      dot = wave_xor_sum(dot, 1) / (float)p.D;
#pragma unroll
      for (int j = 0; j < kNormMaxPerLane; ++j) {
        const int64_t e = lane + (int64_t)j * kWave;
        if (e >= p.D) continue;
        store_from_f32(p.dx, p.dt, base + e, rr * dv[j] - xv[j] * rr * rr * rr * dot);
      }
    }
  }
  if (p.mode == 1) {
#pragma unroll
    for (int j = 0; j < kNormMaxPerLane; ++j) {
      const int64_t e = lane + (int64_t)j * kWave;
      if (e >= p.D) continue;
      p.part[(wave * 2) * p.D + e] = pw[j];
      p.part[(wave * 2 + 1) * p.D + e] = pb[j];
    }
  }
}

// Vector path of the same two backwards for rows of D = 64 or 128 (16-byte aligned tensors): LPR = D / V
// lanes per row, V elements (16 bytes) of each tensor per lane, so a wave covers 64 / LPR rows and its
// loads of U row groups are in flight together; the row sums stay in the row's lane group (DPP). MODE 0 is
// the L2 norm, 1 the RMS norm without a gate, 2 with a gate and SiLU, 3 with a gate used as is. HBM-bound:
// every tensor is read or written once. dw and db are summed in the lanes over all of a block's rows, then
// over the block in LDS: one [2][D] row of partial sums per block. On one MI355X, 262,144 rows of 128 in
// bf16 (config 1's 16,384 tokens x 16 heads): L2 37 us (5.4 TB/s) against 353 for the one-wave-per-row kernel
// above (kept for other D and for unaligned tensors), RMS with the gate 65 us (5.2 TB/s) against 687.
template <typename E, int V, int LPR, int MODE>
__global__ __launch_bounds__(256) void gated_delta_norm_bwd_vec_kernel(NormBwdParams p) {
  typedef E VE __attribute__((ext_vector_type(V)));
  constexpr int D = V * LPR, RPW = kWave / LPR, U = MODE == 0 ? 4 : 2;
  constexpr bool kGate = MODE >= 2;
  const int lane = threadIdx.x % kWave, sub = lane / LPR, li = lane % LPR;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
  const E* __restrict__ xp = static_cast<const E*>(p.x);
  const E* __restrict__ dyp = static_cast<const E*>(p.dy);
  const E* __restrict__ gp = static_cast<const E*>(p.gate);
  float wv[V], bv[V], pw[V], pb[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    wv[e] = (MODE != 0 && p.w) ? p.w[li * V + e] : 1.f;
    bv[e] = (MODE != 0 && p.bias) ? p.bias[li * V + e] : 0.f;
    pw[e] = pb[e] = 0.f;
  }
  for (int64_t r0 = wave * RPW * U; r0 < p.rows; r0 += nwaves * RPW * U) {
    VE xv[U], dv[U], gv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // rows past the end: zeros, so that they add nothing to db
      const int64_t r = r0 + u * RPW + sub;
      xv[u] = dv[u] = gv[u] = VE{};
      if (r < p.rows) {
        const int64_t at = r * D + li * V;
        xv[u] = *reinterpret_cast<const VE*>(xp + at);
        dv[u] = *reinterpret_cast<const VE*>(dyp + at);
        if (kGate) gv[u] = *reinterpret_cast<const VE*>(gp + at);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = r0 + u * RPW + sub;
      float x[V], d[V], ss = 0.f, dot = 0.f;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        x[e] = (float)xv[u][e];
        d[e] = (float)dv[u][e];
        ss += x[e] * x[e];
      }
      ss = group_sum<LPR>(ss);
      VE ox, og;
      if (MODE == 0) {
        const float nrm = sqrtf(ss), inv = 1.f / fmaxf(nrm, p.eps);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          x[e] *= inv;
          dot += x[e] * d[e];
        }
        dot = group_sum<LPR>(dot);
        dot = nrm > p.eps ? dot : 0.f;
#pragma unroll
        for (int e = 0; e < V; ++e) ox[e] = (E)((d[e] - x[e] * dot) * inv);
      } else {
        // 0 past the end: with eps = 0 a row of zeros has r = inf, and its 0 * inf would reach dw
        const float rr = r < p.rows ? 1.f / sqrtf(ss / (float)D + p.eps) : 0.f;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const float n = x[e] * rr;
          float du = d[e];
          if (kGate) {
            const float g = (float)gv[u][e], un = n * wv[e] + bv[e];
            float act = g, dact = 1.f;
            if (MODE == 2) {
              const float sg = sizeof(E) == 2 ? sigmoid_comp(g) : sigmoid_f32(g);
              act = g * sg;
              dact = sg * (1.f + g * (1.f - sg));
            }
            og[e] = (E)(du * un * dact);
            du *= act;
          }
          pw[e] += du * n;
          pb[e] += du;
          d[e] = du * wv[e];  // dn
          dot += d[e] * x[e];
        }
        dot = group_sum<LPR>(dot) / (float)D;
        const float c = rr * (rr * dot);  // of the order of d: r^3 alone is subnormal from an rms of 4e12 up
#pragma unroll
        for (int e = 0; e < V; ++e) ox[e] = (E)(rr * d[e] - x[e] * rr * c);
      }
      if (r < p.rows) {
        const int64_t at = r * D + li * V;
        *reinterpret_cast<VE*>(static_cast<E*>(p.dx) + at) = ox;
        if (kGate) *reinterpret_cast<VE*>(static_cast<E*>(p.dgate) + at) = og;
      }
    }
  }
  if (MODE != 0) {
    __shared__ float red[4][2 * D];
    const int w = threadIdx.x / kWave;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float sw = wave_xor_sum(pw[e], LPR), sb = wave_xor_sum(pb[e], LPR);
      if (sub == 0) {
        red[w][li * V + e] = sw;
        red[w][D + li * V + e] = sb;
      }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < 2 * D; c += 256)
      p.part[(int64_t)blockIdx.x * 2 * D + c] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  }
}

// dweight, dbias [D] from the partial sums [parts][2][D]: one workgroup per 16 columns, 64 rows of partial
// sums at a time, then the 64 row lanes in LDS. Latency-bound (1 MB from the vector kernel at D = 128), so the columns are spread
// over workgroups and the rows over lanes: 4 us for 1024 rows of D = 128, against 970 us for
// 4096 rows with one thread per column.
constexpr int kParamCols = 16, kParamLanes = 64;

__global__ __launch_bounds__(kParamCols* kParamLanes) void gated_delta_norm_param_grad_kernel(
    const float* __restrict__ part, int64_t parts, int64_t D, float* dw, float* db) {
  __shared__ float red[kParamLanes][kParamCols + 1];
  const int ci = threadIdx.x % kParamCols, rl = threadIdx.x / kParamCols;
  const int64_t col = (int64_t)blockIdx.x * kParamCols + ci;  // = k * D + column, k = 0 (dw), 1 (db)
  float acc = 0.f;
  if (col < 2 * D) {
#pragma unroll 8
    for (int64_t r = rl; r < parts; r += kParamLanes) acc += part[r * 2 * D + col];
  }
  red[rl][ci] = acc;
  __syncthreads();
  for (int s = kParamLanes / 2; s > 0; s >>= 1) {
    if (rl < s) red[rl][ci] += red[rl + s][ci];
    __syncthreads();
  }
  if (rl == 0 && col < 2 * D) {
    float* out = col < D ? dw : db;
    if (out) out[col % D] = red[0][ci];
  }
}

// Most blocks of the RMS backward: 4 per CU, up to 4096 rows of partial sums. The 132 registers of the gated 16-bit
// kernels let 3 run on a CU at once, the fourth follows.
constexpr int64_t kNormBwdBlocks = 1024;

// Launches the vector backward when the rows allow it. `blocks` returns the rows of partial sums (RMS).
static bool launch_norm_bwd_vec(const NormBwdParams& p, hipStream_t s, int64_t* blocks) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.gate) |
                         reinterpret_cast<uintptr_t>(p.dy) | reinterpret_cast<uintptr_t>(p.dx) |
                         reinterpret_cast<uintptr_t>(p.dgate)) & 15) == 0;
  if (!aligned || (p.D != 64 && p.D != 128)) return false;
  auto go = [&](auto e_tag, auto lpr_c, auto mode_c) {
    using E = decltype(e_tag);
    constexpr int V = 16 / sizeof(E), LPR = decltype(lpr_c)::value, MODE = decltype(mode_c)::value;
    const int64_t rpb = 4 * (kWave / LPR) * (MODE == 0 ? 4 : 2);  // rows per block and pass
    const int64_t most = MODE == 0 ? 65536 : kNormBwdBlocks, passes = (p.rows + rpb - 1) / rpb;
    *blocks = passes < 1 ? 1 : (passes < most ? passes : most);
    hipLaunchKernelGGL((gated_delta_norm_bwd_vec_kernel<E, V, LPR, MODE>), dim3((unsigned)*blocks), dim3(256), 0, s, p);
  };
  auto by_mode = [&](auto e_tag, auto lpr_c) {
    if (p.mode == 0) go(e_tag, lpr_c, std::integral_constant<int, 0>{});
    else if (!p.gate) go(e_tag, lpr_c, std::integral_constant<int, 1>{});
    else if (p.act == GDN_ACT_SILU) go(e_tag, lpr_c, std::integral_constant<int, 2>{});
    else go(e_tag, lpr_c, std::integral_constant<int, 3>{});
  };
  auto by_d = [&](auto e_tag) {
    constexpr int V = 16 / sizeof(e_tag);
    if (p.D == 128) by_mode(e_tag, std::integral_constant<int, 128 / V>{});
    else by_mode(e_tag, std::integral_constant<int, 64 / V>{});
  };
  if (p.dt == GDN_DTYPE_BF16) by_d(bf16{});
  else if (p.dt == GDN_DTYPE_F16) by_d(f16{});
  else by_d(float{});
  return true;
}

static int launch_norm(const NormParams& p, void* stream, const char* what) {
  if (p.rows == 0) return GDN_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool aligned = ((reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.y) |
                         reinterpret_cast<uintptr_t>(p.x2) | reinterpret_cast<uintptr_t>(p.y2) |
                         reinterpret_cast<uintptr_t>(p.gate)) & 15) == 0;
  const unsigned two = p.x2 ? 2 : 1;
  if (aligned && (p.D == 64 || p.D == 128) && (p.dt == GDN_DTYPE_BF16 || p.dt == GDN_DTYPE_F16)) {
    const int64_t rpb = 4 * (kWave / (p.D / 8)) * kNormV8Groups;  // rows per 256-thread block and pass
    int64_t vb = (p.rows + rpb - 1) / rpb;
    if (vb > 65536) vb = 65536;
    const dim3 g((unsigned)vb, two), b(256);
    if (p.dt == GDN_DTYPE_BF16) {
      if (p.D == 128) hipLaunchKernelGGL((gated_delta_norm_v8_kernel<bf16, 16>), g, b, 0, s, p);
      else hipLaunchKernelGGL((gated_delta_norm_v8_kernel<bf16, 8>), g, b, 0, s, p);
    } else {
      if (p.D == 128) hipLaunchKernelGGL((gated_delta_norm_v8_kernel<f16, 16>), g, b, 0, s, p);
      else hipLaunchKernelGGL((gated_delta_norm_v8_kernel<f16, 8>), g, b, 0, s, p);
    }
    return gdn_internal_check_launch(what);
  }
  int64_t blocks = (p.rows + 3) / 4;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(gated_delta_norm_kernel, dim3((unsigned)blocks, two), dim3(256), 0, s, p);
  return gdn_internal_check_launch(what);
}

}  // namespace gdn

using namespace gdn;

int gdn::gdn_internal_rms_norm_gated(const void* x, const void* gate, const float* w, void* y, int64_t rows, int64_t D,
                                     float eps, int split, hipStream_t s) {
  NormParams p{x, gate, w, nullptr, y, rows, D, GDN_DTYPE_BF16, GDN_ACT_SILU, eps, 1, split, nullptr, nullptr};
  return launch_norm(p, s, "gated_delta_norm_kernel(rms)");
}

extern "C" int gdn_l2norm_fwd(const void* x, void* y, int64_t rows, int64_t D, int dtype, float eps, void* stream) {
  if (!x || !y || rows < 0 || D <= 0) {
    gdn_internal_set_error("gdn_l2norm_fwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  if (D > kNormMaxPerLane * kWave) {
    gdn_internal_set_error("gdn_l2norm_fwd: D=%lld exceeds %d", (long long)D, kNormMaxPerLane * kWave);
    return GDN_ERR_UNSUPPORTED;
  }
  NormParams p{x, nullptr, nullptr, nullptr, y, rows, D, dtype, GDN_ACT_NONE, eps, 0, 0, nullptr, nullptr};
  return launch_norm(p, stream, "gated_delta_norm_kernel(l2)");
}

extern "C" int gdn_qk_l2norm_fwd(const void* q, const void* k, void* q_out, void* k_out, int64_t rows, int64_t D, int dtype,
                                 float eps, void* stream) {
  if (!q || !k || !q_out || !k_out || rows < 0 || D <= 0) {
    gdn_internal_set_error("gdn_qk_l2norm_fwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  if (D > kNormMaxPerLane * kWave) {
    gdn_internal_set_error("gdn_qk_l2norm_fwd: D=%lld exceeds %d", (long long)D, kNormMaxPerLane * kWave);
    return GDN_ERR_UNSUPPORTED;
  }
  NormParams p{q, nullptr, nullptr, nullptr, q_out, rows, D, dtype, GDN_ACT_NONE, eps, 0, 0, k, k_out};
  return launch_norm(p, stream, "gated_delta_norm_kernel(qk l2)");
}

extern "C" int gdn_qk_l2norm_chunk_fwd(const void* q, const void* k, void* q_out, void* k_out, int64_t rows, int64_t D,
                                       void* stream) {
  const uintptr_t al = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                       reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_out);
  if (!q || !k || !q_out || !k_out || rows < 0 || (D != 64 && D != 128) || (al & 15)) {
    gdn_internal_set_error("gdn_qk_l2norm_chunk_fwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  NormParams p{q, nullptr, nullptr, nullptr, q_out, rows, D, GDN_DTYPE_BF16, GDN_ACT_NONE, 0.f, 2, 0, k, k_out};
  return launch_norm(p, stream, "gated_delta_norm_kernel(chunk qk l2)");
}

extern "C" int gdn_rms_norm_gated_fwd(const void* x, const void* gate, const float* weight, const float* bias, void* y,
                                      int64_t rows, int64_t D, int dtype, float eps, int activation, void* stream) {
  if (!x || !y || rows < 0 || D <= 0) {
    gdn_internal_set_error("gdn_rms_norm_gated_fwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  if (D > kNormMaxPerLane * kWave) {
    gdn_internal_set_error("gdn_rms_norm_gated_fwd: D=%lld exceeds %d", (long long)D, kNormMaxPerLane * kWave);
    return GDN_ERR_UNSUPPORTED;
  }
  if (activation != GDN_ACT_NONE && activation != GDN_ACT_SILU) {
    gdn_internal_set_error("gdn_rms_norm_gated_fwd: unknown activation %d", activation);
    return GDN_ERR_INVALID;
  }
  NormParams p{x, gate, weight, bias, y, rows, D, dtype, activation, eps, 1, 0, nullptr, nullptr};
  return launch_norm(p, stream, "gated_delta_norm_kernel(rms)");
}

extern "C" int gdn_l2norm_bwd(const void* x, const void* dy, void* dx, int64_t rows, int64_t D, int dtype, float eps,
                              void* stream) {
  if (!x || !dy || !dx || rows < 0 || D <= 0) {
    gdn_internal_set_error("gdn_l2norm_bwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  if (D > kNormMaxPerLane * kWave) {
    gdn_internal_set_error("gdn_l2norm_bwd: D=%lld exceeds %d", (long long)D, kNormMaxPerLane * kWave);
    return GDN_ERR_UNSUPPORTED;
  }
  if (rows == 0) return GDN_OK;
  NormBwdParams p{x, nullptr, nullptr, nullptr, dy, dx, nullptr, nullptr, rows, D, dtype, GDN_ACT_NONE, eps, 0};
  int64_t blocks = 0;
  if (!launch_norm_bwd_vec(p, static_cast<hipStream_t>(stream), &blocks)) {
    blocks = (rows + 3) / 4;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(gated_delta_norm_bwd_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  }
  return gdn_internal_check_launch("gated_delta_norm_bwd_kernel(l2)");
}

extern "C" size_t gdn_rms_norm_gated_bwd_workspace_size(int64_t rows, int64_t D) {
  if (rows < 0 || D <= 0) return 0;
  return (size_t)(kNormBwdBlocks * 4 * 2 * D * 4);
}

extern "C" int gdn_rms_norm_gated_bwd(const void* x, const void* gate, const float* weight, const float* bias,
                                      const void* dy, void* dx, void* dgate, float* dweight, float* dbias, int64_t rows,
                                      int64_t D, int dtype, float eps, int activation, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  if (!x || !dy || !dx || rows < 0 || D <= 0 || (gate && !dgate)) {
    gdn_internal_set_error("gdn_rms_norm_gated_bwd: bad arguments (rows=%lld D=%lld)", (long long)rows, (long long)D);
    return GDN_ERR_INVALID;
  }
  if (D > kNormMaxPerLane * kWave) {
    gdn_internal_set_error("gdn_rms_norm_gated_bwd: D=%lld exceeds %d", (long long)D, kNormMaxPerLane * kWave);
    return GDN_ERR_UNSUPPORTED;
  }
  if (activation != GDN_ACT_NONE && activation != GDN_ACT_SILU) {
    gdn_internal_set_error("gdn_rms_norm_gated_bwd: unknown activation %d", activation);
    return GDN_ERR_INVALID;
  }
  const size_t need = gdn_rms_norm_gated_bwd_workspace_size(rows, D);
  if (!workspace || workspace_bytes < need) {
    gdn_internal_set_error("gdn_rms_norm_gated_bwd: workspace of %zu bytes needed", need);
    return GDN_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  NormBwdParams p{x, gate, weight, bias, dy, dx, dgate, static_cast<float*>(workspace), rows, D, dtype, activation, eps, 1};
  int64_t parts = 0;
  if (!launch_norm_bwd_vec(p, s, &parts)) {
    parts = kNormBwdBlocks * 4;  // one row of partial sums per wave
    hipLaunchKernelGGL(gated_delta_norm_bwd_kernel, dim3((unsigned)kNormBwdBlocks), dim3(256), 0, s, p);
  }
  int rc = gdn_internal_check_launch("gated_delta_norm_bwd_kernel(rms)");
  if (rc != GDN_OK) return rc;
  hipLaunchKernelGGL(gated_delta_norm_param_grad_kernel, dim3((unsigned)((2 * D + kParamCols - 1) / kParamCols)),
                     dim3(kParamCols * kParamLanes), 0, s, static_cast<const float*>(workspace), parts, D, dweight, dbias);
  return gdn_internal_check_launch("gated_delta_norm_param_grad_kernel");
}
