// The training step's gradient clipping and its check, as clip_grad_norm_ and the non-finite test after it compute them
// (reference asrn/nucleo.py:2253-2343), in three launches for all gradients instead of about twenty small ones: the
// sums of squares of every gradient in blocks, the norm with the factor and the skip flag from them, the scaling.
// Small models are bound by launches (a few microseconds each), large ones by HBM: the gradients are read twice and
// written once, as before. Sums in fp32 within a block of 8,192 values, in double over the blocks, in a fixed order.
#include <type_traits>

#include "common.h"

namespace asrn {

constexpr int kClipThr = 256;
constexpr int kClipBlock = 8192;      // values a workgroup takes
constexpr int kClipTensors = 110;     // gradients a launch takes (its arguments hold their addresses)

struct ClipList {
  float* g[kClipTensors];
  int64_t n[kClipTensors];
  int32_t first[kClipTensors];        // the tensor's first block in this launch
  int count;
};

__device__ __forceinline__ int clip_tensor(const ClipList& l, int blk) {
  int lo = 0, hi = l.count - 1;       // the last tensor whose blocks start at or before blk
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (l.first[mid] <= blk) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// the block's values as float4 (f4: U of them a thread, kClipThr apart from p) when the tensor is 16-byte aligned, the
// rest one by one (f1)
template <class F4, class F1>
__device__ __forceinline__ void clip_block(const ClipList& l, F4 f4, F1 f1) {
  const int t = clip_tensor(l, blockIdx.x);
  const int64_t i0 = (int64_t)(blockIdx.x - l.first[t]) * kClipBlock;
  const int64_t left = l.n[t] - i0;
  const int n = left < kClipBlock ? (int)left : kClipBlock;
  float* p = l.g[t] + i0;
  const int n4 = ((uintptr_t)p & 15) == 0 ? n / 4 : 0;
  if (n4 == kClipBlock / 4) {
    f4(p, std::integral_constant<int, kClipBlock / 4 / kClipThr>{});
  } else {
    for (int i = threadIdx.x; i < n4; i += kClipThr)
      f4(p + 4 * (i - (int)threadIdx.x), std::integral_constant<int, 1>{});
    for (int i = 4 * n4 + threadIdx.x; i < n; i += kClipThr) f1(p + i);
  }
}

__global__ __launch_bounds__(kClipThr) void k_clip_sums(ClipList l, double* __restrict__ part) {
  __shared__ float red[kClipThr / kWave];
  float s = 0.f;
  clip_block(
      l,
      [&](const float* p, auto u) {
        float4 v[decltype(u)::value];
#pragma unroll
        for (int i = 0; i < decltype(u)::value; ++i)
          v[i] = reinterpret_cast<const float4*>(p)[threadIdx.x + i * kClipThr];
#pragma unroll
        for (int i = 0; i < decltype(u)::value; ++i)
          s += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
      },
      [&](const float* p) { s += *p * *p; });
  s = wave_sum(s);
  if (lane_id() == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((double)red[0] + red[1]) + ((double)red[2] + red[3]);
}

// norm = sqrt(sum); factor = min(1, max_norm / (norm + 1e-6)) (NaN stays); skip = 1 when the loss or the norm is not finite
__global__ __launch_bounds__(kClipThr) void k_clip_norm(const double* __restrict__ part, int blocks, float max_norm,
                                                        const float* __restrict__ loss, float* norm, float* factor,
                                                        float* skip) {
  __shared__ double red[kClipThr];
  double s = 0.0;
  for (int i0 = threadIdx.x; i0 < blocks; i0 += 8 * kClipThr) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = part[i0 + u * kClipThr < blocks ? i0 + u * kClipThr : i0];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += i0 + u * kClipThr < blocks ? v[u] : 0.0;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = kClipThr / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float n = (float)sqrt(red[0]);
    const float c = max_norm / (n + 1e-6f);
    *norm = n;
    *factor = c > 1.f ? 1.f : c;
    *skip = fabsf(*loss) < INFINITY && fabsf(n) < INFINITY ? 0.f : 1.f;
  }
}

__global__ __launch_bounds__(kClipThr) void k_clip_scale(ClipList l, const float* __restrict__ factor) {
  const float c = *factor;
  clip_block(
      l,
      [&](float* p, auto u) {
        float4 v[decltype(u)::value];
#pragma unroll
        for (int i = 0; i < decltype(u)::value; ++i) v[i] = reinterpret_cast<float4*>(p)[threadIdx.x + i * kClipThr];
#pragma unroll
        for (int i = 0; i < decltype(u)::value; ++i)
          reinterpret_cast<float4*>(p)[threadIdx.x + i * kClipThr] =
              make_float4(v[i].x * c, v[i].y * c, v[i].z * c, v[i].w * c);
      },
      [&](float* p) { *p *= c; });
}

static int64_t clip_blocks(int64_t n) { return (n + kClipBlock - 1) / kClipBlock; }

}  // namespace asrn

using namespace asrn;

extern "C" int64_t asrn_clip_gradients_workspace(int32_t n, const int64_t* sizes) {
  int64_t b = 0;
  for (int i = 0; i < n; ++i) b += clip_blocks(sizes[i]);
  return 8 * (b + 2);
}

extern "C" int asrn_clip_gradients(int32_t n, float* const* grads, const int64_t* sizes, float max_norm,
                                   const float* loss, float* norm, float* skip, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  ASRN_REQUIRE(n >= 0 && loss && norm && skip && max_norm >= 0.f, "asrn_clip_gradients: bad arguments");
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    ASRN_REQUIRE(sizes[i] >= 0 && (sizes[i] == 0 || grads[i]) && ((uintptr_t)grads[i] & 3) == 0,
                 "asrn_clip_gradients: bad gradient %d", i);
    total += clip_blocks(sizes[i]);
  }
  ASRN_REQUIRE(total < (int64_t(1) << 31), "asrn_clip_gradients: too many values");
  ASRN_REQUIRE(workspace && workspace_bytes >= 8 * (total + 2) && ((uintptr_t)workspace & 7) == 0,
               "asrn_clip_gradients: needs an 8-byte aligned workspace of %lld bytes (got %lld)",
               (long long)(8 * (total + 2)), (long long)workspace_bytes);
  hipStream_t st = (hipStream_t)stream;
  double* part = (double*)workspace + 2;
  float* factor = (float*)workspace;
  for (int pass = 0; pass < 2; ++pass) {               // the sums, then (with the factor known) the scaling
    int64_t done = 0;
    for (int i = 0; i < n;) {
      ClipList l;
      l.count = 0;
      int64_t b = 0;
      for (; i < n && l.count < kClipTensors; ++i) {
        if (sizes[i] == 0) continue;
        l.g[l.count] = grads[i];
        l.n[l.count] = sizes[i];
        l.first[l.count++] = (int32_t)b;
        b += clip_blocks(sizes[i]);
      }
      if (b == 0) continue;
      if (pass == 0) hipLaunchKernelGGL(k_clip_sums, dim3((unsigned)b), dim3(kClipThr), 0, st, l, part + done);
      else hipLaunchKernelGGL(k_clip_scale, dim3((unsigned)b), dim3(kClipThr), 0, st, l, factor);
      if (check_launch("asrn_clip_gradients")) return 1;
      done += b;
    }
    if (pass == 0) {
      hipLaunchKernelGGL(k_clip_norm, dim3(1), dim3(kClipThr), 0, st, part, (int)total, max_norm, loss, norm, factor,
                         skip);
      if (check_launch("asrn_clip_gradients")) return 1;
    }
  }
  return 0;
}
