// The context hash's key rows in 16 bits (asrn/nucleo.py:644-659 under autocast): from E (B, L, d) in fp32, its
// bf16 rows and the keys [E_t ; E_{t-1}] (the second half 0 at t = 0) that the context MLP's first product reads; and
// back, the three users' gradients (the word product's and the candidates' of the rows, the key's) summed in fp32 into
// dE.
//
// Both are bound by memory. One thread takes 8 channels of one token: forward, one 32-byte read and one
// 16-byte store to the rows and to each of the two keys that hold the token; backward, its four 16-byte loads (the
// next key's second half among them) and one store. As PyTorch operators (cast, zero fill, shifted copy,
// concatenation; and back two slices, a zero fill, a shifted copy, three sums and a cast) the values crossed memory
// five times each way: at 2 x 32,768 x 512, 211 us and four kernels forward, 211 us and seven backward. Here 61 and 76 us
// (335 and 403 MB, 5.4 TB/s).
#include "common.h"

namespace asrn {

constexpr int kKeyThreads = 256;

__device__ __forceinline__ uint32_t key_bf16(float x) {                         // nearest even, as the cast rounds
  const uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;                // NaN stays a (quiet) NaN
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ void key_add(const uint16_t* __restrict__ g, int64_t i, float (&s)[8]) {
  const uint4 u = *reinterpret_cast<const uint4*>(g + i);
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    s[2 * k] += __uint_as_float(w[k] << 16);
    s[2 * k + 1] += __uint_as_float(w[k] & 0xffff0000u);
  }
}

__global__ __launch_bounds__(kKeyThreads) void k_key_rows_fwd(const float* __restrict__ E, int64_t n, int64_t L, int d,
                                                               uint16_t* __restrict__ rows,
                                                               uint16_t* __restrict__ keys) {
  const int64_t e = (int64_t)blockIdx.x * kKeyThreads + threadIdx.x;
  if (e >= n) return;
  const int w = d / 8;
  const int64_t bt = e / w, t = bt % L;
  const int c = (int)(e - bt * w) * 8;
  const float4* x = reinterpret_cast<const float4*>(E + e * 8);
  const float4 a = x[0], b = x[1];
  const uint4 u = make_uint4(key_bf16(a.x) | key_bf16(a.y) << 16, key_bf16(a.z) | key_bf16(a.w) << 16,
                             key_bf16(b.x) | key_bf16(b.y) << 16, key_bf16(b.z) | key_bf16(b.w) << 16);
  uint16_t* key = keys + bt * 2 * d + c;
  *reinterpret_cast<uint4*>(rows + e * 8) = u;
  *reinterpret_cast<uint4*>(key) = u;
  if (t + 1 < L) *reinterpret_cast<uint4*>(key + 3 * (int64_t)d) = u;            // the next token's second half
  if (t == 0) *reinterpret_cast<uint4*>(key + d) = make_uint4(0u, 0u, 0u, 0u);
}

__global__ __launch_bounds__(kKeyThreads) void k_key_rows_bwd(const uint16_t* __restrict__ g1,
                                                               const uint16_t* __restrict__ g2,
                                                               const uint16_t* __restrict__ gk, int64_t n, int64_t L,
                                                               int d, float* __restrict__ dE) {
  const int64_t e = (int64_t)blockIdx.x * kKeyThreads + threadIdx.x;
  if (e >= n) return;
  const int w = d / 8;
  const int64_t bt = e / w, t = bt % L;
  const int c = (int)(e - bt * w) * 8;
  float s[8] = {};
  if (g1) key_add(g1, e * 8, s);
  if (gk) {
    const int64_t k = bt * 2 * d + c;
    key_add(gk, k, s);
    if (t + 1 < L) key_add(gk, k + 3 * (int64_t)d, s);
  }
  if (g2) key_add(g2, e * 8, s);
  float4* o = reinterpret_cast<float4*>(dE + e * 8);
  o[0] = make_float4(s[0], s[1], s[2], s[3]);
  o[1] = make_float4(s[4], s[5], s[6], s[7]);
}

static int key_sizes(const char* what, int64_t B, int64_t L, int32_t d) {
  ASRN_REQUIRE(B >= 0 && L >= 0 && d >= 8 && d % 8 == 0 && (B == 0 || L <= ((int64_t)1 << 36) / B / d),
               "%s: bad sizes B=%lld L=%lld d=%d (d a multiple of 8)", what, (long long)B, (long long)L, d);
  return 0;
}

}  // namespace asrn

using namespace asrn;

extern "C" int asrn_key_rows_fwd(const float* E, int64_t B, int64_t L, int32_t d, void* rows, void* keys,
                                 void* stream) {
  if (const int rc = key_sizes("asrn_key_rows_fwd", B, L, d)) return rc;
  ASRN_REQUIRE((((uintptr_t)E | (uintptr_t)rows | (uintptr_t)keys) & 15) == 0,
               "asrn_key_rows_fwd: E, rows and keys must be 16-byte aligned");
  const int64_t n = B * L * (d / 8);
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_key_rows_fwd, dim3((unsigned)((n + kKeyThreads - 1) / kKeyThreads)), dim3(kKeyThreads), 0,
                     (hipStream_t)stream, E, n, L, d, reinterpret_cast<uint16_t*>(rows),
                     reinterpret_cast<uint16_t*>(keys));
  return check_launch("asrn_key_rows_fwd");
}

extern "C" int asrn_key_rows_bwd(const void* drows, const void* drows2, const void* dkeys, int64_t B, int64_t L,
                                 int32_t d, float* dE, void* stream) {
  if (const int rc = key_sizes("asrn_key_rows_bwd", B, L, d)) return rc;
  ASRN_REQUIRE((((uintptr_t)drows | (uintptr_t)drows2 | (uintptr_t)dkeys | (uintptr_t)dE) & 15) == 0,
               "asrn_key_rows_bwd: the gradients must be 16-byte aligned");
  const int64_t n = B * L * (d / 8);
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_key_rows_bwd, dim3((unsigned)((n + kKeyThreads - 1) / kKeyThreads)), dim3(kKeyThreads), 0,
                     (hipStream_t)stream, reinterpret_cast<const uint16_t*>(drows),
                     reinterpret_cast<const uint16_t*>(drows2), reinterpret_cast<const uint16_t*>(dkeys), n, L, d, dE);
  return check_launch("asrn_key_rows_bwd");
}
