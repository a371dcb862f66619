// The model's LayerNorms (the local blocks' ln1 / ln2 and the final ln_f; reference asrn/nucleo.py:969-1014, 1047-1125),
// as torch.nn.LayerNorm computes them in fp32 (biased variance, rstd = 1 / sqrt(var + eps)), with two things fused:
//   forward   y = (x - mean) rstd gamma + beta written in fp32 or straight in bf16 (rounded to nearest even, as the cast
//             that autocast puts before the next bf16 product rounds), and (mean, rstd) kept per row;
//   backward  from dy (fp32 or bf16): g = dy gamma, dx = rstd (g - mean(g) - xhat mean(g xhat)) [+ dres, the gradient
//             of the same x through the residual path, so that autograd adds nothing], and d gamma = sum dy xhat,
//             d beta = sum dy as per-workgroup partial rows summed in a fixed order by asrn_column_sums.
// The local block's middle is fused into its second LayerNorm (GC: c, the convolution's output, in fp32 or bf16): forward
// x = h + gelu(c), kept for the residual path, then the norm of x; backward also dc = gelu'(c) dx, each rounded where
// autocast's separate ops round (gelu's output, dx and dc to c's dtype). HBM-bound; at 16,384 rows of 768 in bf16 the
// forward's three kernels took 59 us and the backward's three 90 us, the fused ones 32 and 66.
// Forward: a workgroup takes 8 rows, each wave 2 with both rows (float4 per lane) loaded at once. Backward: a workgroup
// takes 32 rows, each wave 8 of them, 2 rows' loads at a time.
#include "common.h"

namespace asrn {

constexpr int kLnThreads = 256;
constexpr int kLnWaves = kLnThreads / kWave;
constexpr int kLnFwdRows = 8;
constexpr int kLnFwdPerWave = kLnFwdRows / kLnWaves;
constexpr int kLnBwdRows = 32;
constexpr int kLnBwdPerWave = kLnBwdRows / kLnWaves;
constexpr int kLnBatch = 2;
constexpr int kLnMaxD4 = 4;      // d <= 1024

struct LnArgs {
  const float* x; int64_t ldx; const float* gamma; const float* beta;
  int64_t rows; int d; float eps;
  void* y; int64_t ldy; float2* stats;                                   // forward
  const void* dy; int64_t lddy; const float* dres; float* dx; float* partial;   // backward (dx and dres: ldx)
  const void* c; float* xout; void* dc;     // GC: c (rows, d) dense; forward x + gelu(c) out (ldx); backward dc out
};

// exact GELU and its derivative, as torch forms them in fp32
__device__ __forceinline__ float ln_gelu(float x) { return x * 0.5f * (1.f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float ln_dgelu(float x) {
  return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * (expf(-0.5f * x * x) * 0.39894228040143268f);
}

__device__ __forceinline__ uint32_t ln_bf16(float v) {
  const uint32_t u = __float_as_uint(v);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;        // NaN stays a (quiet) NaN
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float4 ld_row4(const void* p, bool b16, int64_t off4) {
  if (b16) {
    const uint2 u = reinterpret_cast<const uint2*>(p)[off4];
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u));
  }
  return reinterpret_cast<const float4*>(p)[off4];
}
// v rounded to bf16 and back
__device__ __forceinline__ float ln_round(float v) { return __uint_as_float(ln_bf16(v) << 16); }
template <bool B16, class F>
__device__ __forceinline__ float4 ln_map(float4 v, F f) {
  const float4 r = make_float4(f(v.x), f(v.y), f(v.z), f(v.w));
  return B16 ? make_float4(ln_round(r.x), ln_round(r.y), ln_round(r.z), ln_round(r.w)) : r;
}
__device__ __forceinline__ float ln_dot4(float4 a, float4 b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

template <int D4, bool OB16, int GC>
__global__ __launch_bounds__(kLnThreads) void k_ln_fwd(LnArgs a) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int d4 = a.d >> 2;
  const float inv_d = 1.f / (float)a.d;
  const int64_t r0 = (int64_t)blockIdx.x * kLnFwdRows + wave * kLnFwdPerWave;
  float4 xv[kLnFwdPerWave][D4];
  float s[kLnFwdPerWave];
#pragma unroll
  for (int u = 0; u < kLnFwdPerWave; ++u) {
    const int64_t r = r0 + u;
    s[u] = 0.f;
#pragma unroll
    for (int k = 0; k < D4; ++k) {
      const int q = lane + kWave * k;
      xv[u][k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r < a.rows && q < d4) {
        xv[u][k] = reinterpret_cast<const float4*>(a.x + r * a.ldx)[q];
        if constexpr (GC > 0) {
          const float4 g = ln_map<GC == 2>(ld_row4(a.c, GC == 2, r * d4 + q), ln_gelu);
          xv[u][k].x += g.x; xv[u][k].y += g.y; xv[u][k].z += g.z; xv[u][k].w += g.w;
          reinterpret_cast<float4*>(a.xout + r * a.ldx)[q] = xv[u][k];
        }
        s[u] += (xv[u][k].x + xv[u][k].y) + (xv[u][k].z + xv[u][k].w);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kLnFwdPerWave; ++u) {
    const int64_t r = r0 + u;
    if (r >= a.rows) break;
    const float mean = wave_sum_u(s[u]) * inv_d;
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < D4; ++k) {
      const int q = lane + kWave * k;
      if (q < d4) {
        const float4 c = make_float4(xv[u][k].x - mean, xv[u][k].y - mean, xv[u][k].z - mean, xv[u][k].w - mean);
        v += ln_dot4(c, c);
      }
    }
    const float rstd = rsqrtf(wave_sum_u(v) * inv_d + a.eps);
#pragma unroll
    for (int k = 0; k < D4; ++k) {
      const int q = lane + kWave * k;
      if (q < d4) {
        const float4 w = reinterpret_cast<const float4*>(a.gamma)[q], b = reinterpret_cast<const float4*>(a.beta)[q];
        const float4 y = make_float4((xv[u][k].x - mean) * rstd * w.x + b.x, (xv[u][k].y - mean) * rstd * w.y + b.y,
                                     (xv[u][k].z - mean) * rstd * w.z + b.z, (xv[u][k].w - mean) * rstd * w.w + b.w);
        if constexpr (OB16) {
          reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.y) + r * a.ldy)[q] =
              make_uint2(ln_bf16(y.x) | (ln_bf16(y.y) << 16), ln_bf16(y.z) | (ln_bf16(y.w) << 16));
        } else {
          reinterpret_cast<float4*>(reinterpret_cast<float*>(a.y) + r * a.ldy)[q] = y;
        }
      }
    }
    if (lane == 0) a.stats[r] = make_float2(mean, rstd);
  }
}

template <int D4, bool DB16, int GC>
__global__ __launch_bounds__(kLnThreads) void k_ln_bwd(LnArgs a) {
  __shared__ float red[kLnWaves][2 * 4 * D4 * kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int d4 = a.d >> 2;
  const float inv_d = 1.f / (float)a.d;
  const int64_t r0 = (int64_t)blockIdx.x * kLnBwdRows + wave * kLnBwdPerWave;
  float4 gw[D4], gb[D4];
#pragma unroll
  for (int k = 0; k < D4; ++k) gw[k] = gb[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int b = 0; b < kLnBwdPerWave; b += kLnBatch) {
    float4 xv[kLnBatch][D4], dv[kLnBatch][D4], rv[kLnBatch][D4], cv[kLnBatch][GC > 0 ? D4 : 1];
    float2 st[kLnBatch];
#pragma unroll
    for (int u = 0; u < kLnBatch; ++u) {
      const int64_t r = r0 + b + u;
      const bool ok = r < a.rows;
      st[u] = ok ? a.stats[r] : make_float2(0.f, 1.f);
#pragma unroll
      for (int k = 0; k < D4; ++k) {
        const int q = lane + kWave * k;
        xv[u][k] = dv[u][k] = rv[u][k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (ok && q < d4) {
          xv[u][k] = reinterpret_cast<const float4*>(a.x + r * a.ldx)[q];
          dv[u][k] = DB16 ? ld_row4(reinterpret_cast<const uint16_t*>(a.dy) + r * a.lddy, true, q)
                          : ld_row4(reinterpret_cast<const float*>(a.dy) + r * a.lddy, false, q);
          if (a.dres) rv[u][k] = reinterpret_cast<const float4*>(a.dres + r * a.ldx)[q];
          if constexpr (GC > 0) cv[u][k] = ld_row4(a.c, GC == 2, r * d4 + q);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kLnBatch; ++u) {
      const int64_t r = r0 + b + u;
      if (r >= a.rows) break;
      const float mean = st[u].x, rstd = st[u].y;
      float4 xh[D4], g[D4];
      float m1 = 0.f, m2 = 0.f;
#pragma unroll
      for (int k = 0; k < D4; ++k) {
        const int q = lane + kWave * k;
        if (q < d4) {
          const float4 w = reinterpret_cast<const float4*>(a.gamma)[q];
          xh[k] = make_float4((xv[u][k].x - mean) * rstd, (xv[u][k].y - mean) * rstd, (xv[u][k].z - mean) * rstd,
                              (xv[u][k].w - mean) * rstd);
          g[k] = make_float4(dv[u][k].x * w.x, dv[u][k].y * w.y, dv[u][k].z * w.z, dv[u][k].w * w.w);
          m1 += (g[k].x + g[k].y) + (g[k].z + g[k].w);
          m2 += ln_dot4(g[k], xh[k]);
          gw[k].x += dv[u][k].x * xh[k].x; gw[k].y += dv[u][k].y * xh[k].y;
          gw[k].z += dv[u][k].z * xh[k].z; gw[k].w += dv[u][k].w * xh[k].w;
          gb[k].x += dv[u][k].x; gb[k].y += dv[u][k].y; gb[k].z += dv[u][k].z; gb[k].w += dv[u][k].w;
        }
      }
      m1 = wave_sum_u(m1) * inv_d;
      m2 = wave_sum_u(m2) * inv_d;
#pragma unroll
      for (int k = 0; k < D4; ++k) {
        const int q = lane + kWave * k;
        if (q < d4) {
          const float4 dx =
              make_float4(rstd * (g[k].x - m1 - xh[k].x * m2) + rv[u][k].x, rstd * (g[k].y - m1 - xh[k].y * m2) + rv[u][k].y,
                          rstd * (g[k].z - m1 - xh[k].z * m2) + rv[u][k].z, rstd * (g[k].w - m1 - xh[k].w * m2) + rv[u][k].w);
          reinterpret_cast<float4*>(a.dx + r * a.ldx)[q] = dx;
          if constexpr (GC > 0) {
            const float4 e = ln_map<GC == 2>(dx, [](float v) { return v; }), w = ln_map<false>(cv[u][k], ln_dgelu);
            const float4 dc = make_float4(e.x * w.x, e.y * w.y, e.z * w.z, e.w * w.w);
            if constexpr (GC == 2)
              reinterpret_cast<uint2*>(a.dc)[r * d4 + q] =
                  make_uint2(ln_bf16(dc.x) | (ln_bf16(dc.y) << 16), ln_bf16(dc.z) | (ln_bf16(dc.w) << 16));
            else
              reinterpret_cast<float4*>(a.dc)[r * d4 + q] = dc;
          }
        }
      }
    }
  }
  // workgroup partial row [d gamma | d beta], the waves in order
  float* mine = red[wave];
#pragma unroll
  for (int k = 0; k < D4; ++k) {
    const int q = lane + kWave * k;
    float* o = mine + 4 * q;
    o[0] = gw[k].x; o[1] = gw[k].y; o[2] = gw[k].z; o[3] = gw[k].w;
    float* ob = mine + 4 * D4 * kWave + 4 * q;
    ob[0] = gb[k].x; ob[1] = gb[k].y; ob[2] = gb[k].z; ob[3] = gb[k].w;
  }
  __syncthreads();
  float* prow = a.partial + (int64_t)blockIdx.x * 2 * a.d;
  for (int c = threadIdx.x; c < 2 * a.d; c += kLnThreads) {
    const int src = c < a.d ? c : 4 * D4 * kWave + (c - a.d);
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kLnWaves; ++w) v += red[w][src];
    prow[c] = v;
  }
}

static int64_t ln_bwd_groups(int64_t rows) { return rows > 0 ? (rows + kLnBwdRows - 1) / kLnBwdRows : 1; }
static int ln_d4(int d) { return (d + 4 * kWave - 1) / (4 * kWave); }

}  // namespace asrn

using namespace asrn;

// GC of c: 0 none, 1 fp32, 2 bf16
#define LN_GC(KERNEL, D4, B16)                                                                        \
  if (gc == 0) hipLaunchKernelGGL((KERNEL<D4, B16, 0>), grid, block, 0, st, a);                       \
  else if (gc == 1) hipLaunchKernelGGL((KERNEL<D4, B16, 1>), grid, block, 0, st, a);                  \
  else hipLaunchKernelGGL((KERNEL<D4, B16, 2>), grid, block, 0, st, a);
#define LN_B16(KERNEL, D4) \
  if (b16) { LN_GC(KERNEL, D4, true) } else { LN_GC(KERNEL, D4, false) }
#define LN_LAUNCH(KERNEL)                  \
  switch (ln_d4(a.d)) {                    \
    case 1: LN_B16(KERNEL, 1) break;       \
    case 2: LN_B16(KERNEL, 2) break;       \
    case 3: LN_B16(KERNEL, 3) break;       \
    default: LN_B16(KERNEL, 4) break;      \
  }

static int ln_fwd(LnArgs a, bool b16, int gc, hipStream_t st, const char* what) {
  ASRN_REQUIRE(a.rows >= 0 && a.d > 0 && a.d % 4 == 0 && a.d <= 4 * kLnMaxD4 * kWave && a.ldx >= a.d &&
                   a.ldx % 4 == 0 && a.ldy >= a.d && a.ldy % 4 == 0 && a.eps > 0.f,
               "%s: bad sizes rows=%lld d=%d (a multiple of 4, <= %d) ldx=%lld ldy=%lld", what, (long long)a.rows, a.d,
               4 * kLnMaxD4 * kWave, (long long)a.ldx, (long long)a.ldy);
  if (a.rows == 0) return 0;
  ASRN_REQUIRE(((uintptr_t)a.x & 15) == 0 && ((uintptr_t)a.y & (b16 ? 7 : 15)) == 0 && ((uintptr_t)a.gamma & 15) == 0 &&
                   ((uintptr_t)a.beta & 15) == 0 && ((uintptr_t)a.c & (gc == 2 ? 7 : 15)) == 0 &&
                   ((uintptr_t)a.xout & 15) == 0,
               "%s: rows and parameters must be 16-byte aligned (8 for bf16)", what);
  const dim3 grid((unsigned)((a.rows + kLnFwdRows - 1) / kLnFwdRows)), block(kLnThreads);
  LN_LAUNCH(k_ln_fwd)
  return check_launch(what);
}

static int ln_bwd(LnArgs a, bool b16, int gc, float* dparams, void* workspace, int64_t workspace_bytes, void* stream,
                  const char* what) {
  ASRN_REQUIRE(a.rows >= 0 && a.d > 0 && a.d % 4 == 0 && a.d <= 4 * kLnMaxD4 * kWave && a.ldx >= a.d &&
                   a.ldx % 4 == 0 && a.lddy >= a.d && a.lddy % 4 == 0,
               "%s: bad sizes rows=%lld d=%d (a multiple of 4, <= %d) ldx=%lld lddy=%lld", what, (long long)a.rows,
               a.d, 4 * kLnMaxD4 * kWave, (long long)a.ldx, (long long)a.lddy);
  const int64_t need = asrn_layer_norm_bwd_workspace(a.rows, a.d);
  ASRN_REQUIRE(need >= 0 && workspace_bytes >= need && workspace != nullptr && ((uintptr_t)workspace % 256) == 0,
               "%s: needs a 256-byte aligned workspace of %lld bytes", what, (long long)need);
  if (a.rows == 0)
    return asrn_column_sums(nullptr, 0, 0, 2 * (int64_t)a.d, 2 * (int64_t)a.d, dparams, nullptr, 0, stream);
  ASRN_REQUIRE(((uintptr_t)a.x & 15) == 0 && ((uintptr_t)a.dx & 15) == 0 && ((uintptr_t)a.dy & (b16 ? 7 : 15)) == 0 &&
                   ((uintptr_t)a.dres & 15) == 0 && ((uintptr_t)a.gamma & 15) == 0 &&
                   (((uintptr_t)a.c | (uintptr_t)a.dc) & (gc == 2 ? 7 : 15)) == 0,
               "%s: rows and parameters must be 16-byte aligned (8 for bf16)", what);
  a.partial = (float*)workspace;
  const int64_t groups = ln_bwd_groups(a.rows);
  ASRN_REQUIRE(groups < (int64_t(1) << 31), "%s: too many rows", what);
  const dim3 grid((unsigned)groups), block(kLnThreads);
  hipStream_t st = (hipStream_t)stream;
  LN_LAUNCH(k_ln_bwd)
  if (check_launch(what)) return 1;
  // one launch for up to 1,024 partial rows (two rounds of its loads); more are summed in two levels
  if (groups <= 1024) return group_sums(a.partial, (int)groups, 2 * a.d, dparams, st);
  const int64_t part_bytes = (groups * 2 * a.d * 4 + 255) / 256 * 256;
  return asrn_column_sums(a.partial, 0, groups, 2 * (int64_t)a.d, 2 * (int64_t)a.d, dparams,
                          (char*)workspace + part_bytes, need - part_bytes, stream);
}

extern "C" int asrn_layer_norm_fwd(const float* x, int64_t ldx, const float* gamma, const float* beta, int64_t rows,
                                   int32_t d, float eps, int32_t out_bf16, void* y, int64_t ldy, float* stats,
                                   void* stream) {
  LnArgs a{};
  a.x = x; a.ldx = ldx; a.gamma = gamma; a.beta = beta; a.rows = rows; a.d = d; a.eps = eps; a.y = y; a.ldy = ldy;
  a.stats = reinterpret_cast<float2*>(stats);
  ASRN_REQUIRE(out_bf16 == 0 || out_bf16 == 1, "asrn_layer_norm_fwd: out_bf16 must be 0 or 1");
  return ln_fwd(a, out_bf16, 0, (hipStream_t)stream, "asrn_layer_norm_fwd");
}

extern "C" int asrn_gelu_norm_fwd(const float* h, const void* c, int32_t c_bf16, const float* gamma, const float* beta,
                                  int64_t rows, int32_t d, float eps, int32_t out_bf16, float* x, void* y,
                                  float* stats, void* stream) {
  LnArgs a{};
  a.x = h; a.ldx = d; a.gamma = gamma; a.beta = beta; a.rows = rows; a.d = d; a.eps = eps; a.y = y; a.ldy = d;
  a.stats = reinterpret_cast<float2*>(stats); a.c = c; a.xout = x;
  ASRN_REQUIRE(rows == 0 || (c && x), "asrn_gelu_norm_fwd: null c or x");
  return ln_fwd(a, out_bf16 != 0, c_bf16 ? 2 : 1, (hipStream_t)stream, "asrn_gelu_norm_fwd");
}

extern "C" int64_t asrn_layer_norm_bwd_workspace(int64_t rows, int32_t d) {
  if (rows < 0 || d <= 0) return -1;
  const int64_t groups = ln_bwd_groups(rows);
  const int64_t part = (groups * 2 * d * 4 + 255) / 256 * 256;
  const int64_t sums = asrn_column_sums_workspace(groups, 2 * (int64_t)d);
  return sums < 0 ? -1 : part + sums;
}

extern "C" int asrn_layer_norm_bwd(const float* x, int64_t ldx, const float* gamma, const float* stats, int64_t rows,
                                   int32_t d, const void* dy, int32_t dy_bf16, int64_t lddy, const float* dres,
                                   float* dx, float* dparams, void* workspace, int64_t workspace_bytes,
                                   void* stream) {
  LnArgs a{};
  a.x = x; a.ldx = ldx; a.gamma = gamma; a.rows = rows; a.d = d; a.stats = reinterpret_cast<float2*>(const_cast<float*>(stats));
  a.dy = dy; a.lddy = lddy; a.dres = dres; a.dx = dx;
  ASRN_REQUIRE(dy_bf16 == 0 || dy_bf16 == 1, "asrn_layer_norm_bwd: dy_bf16 must be 0 or 1");
  return ln_bwd(a, dy_bf16, 0, dparams, workspace, workspace_bytes, stream, "asrn_layer_norm_bwd");
}

extern "C" int asrn_gelu_norm_bwd(const float* x, const void* c, int32_t c_bf16, const float* gamma, const float* stats,
                                  int64_t rows, int32_t d, const void* dy, int32_t dy_bf16, const float* dres,
                                  float* dx, void* dc, float* dparams, void* workspace, int64_t workspace_bytes,
                                  void* stream) {
  LnArgs a{};
  a.x = x; a.ldx = d; a.gamma = gamma; a.rows = rows; a.d = d; a.stats = reinterpret_cast<float2*>(const_cast<float*>(stats));
  a.dy = dy; a.lddy = d; a.dres = dres; a.dx = dx; a.c = c; a.dc = dc;
  ASRN_REQUIRE(rows == 0 || (c && dc), "asrn_gelu_norm_bwd: null c or dc");
  return ln_bwd(a, dy_bf16 != 0, c_bf16 ? 2 : 1, dparams, workspace, workspace_bytes, stream, "asrn_gelu_norm_bwd");
}
