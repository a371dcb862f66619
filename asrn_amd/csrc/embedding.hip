// The embedding's gradient for a batch of up to 4,096 tokens: dW[v] = the sum of dE over the positions that hold token v, in
// position order, for every row of the vocabulary (0 where no position holds it). Replaces the framework's kernel for
// short batches, which walks the tokens serially (2,048 tokens, d 64, V 256: 98 us, a tenth of the small model's
// training step; here 10 us). Bound by latency: the rows of a workgroup's most frequent tokens follow one another.
//
// A workgroup owns kEmbRows rows of the vocabulary and 64 columns. It lists the positions that hold its tokens, in
// order (a scan of all ids, 8 a thread in flight, compacted by ballots), then each of its four waves adds a quarter of
// the list, in order, into its own sums in LDS (a lane owns a column, so nothing collides), 16 rows in flight; the
// quarters are added in order. No atomics.
#include "common.h"

namespace asrn {

constexpr int kEmbThr = 256, kEmbWaves = kEmbThr / kWave;
constexpr int kEmbRows = 16;
constexpr int kEmbMax = 4096;          // tokens: the list's room in LDS

__global__ __launch_bounds__(kEmbThr) void k_embedding_bwd(const float* __restrict__ dE, const int64_t* __restrict__ ids,
                                                           int n, int64_t V, int d, float* __restrict__ dW) {
  __shared__ uint16_t list[kEmbMax];                       // position << 4 | row: positions below 4,096
  __shared__ float acc[kEmbWaves][kEmbRows][kWave];
  __shared__ int counts[kEmbWaves];
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int64_t v0 = (int64_t)blockIdx.x * kEmbRows;
  const int c = blockIdx.y * kWave + lane;
  int total = 0;
  constexpr int U = 8;
  for (int i0 = 0; i0 < n; i0 += U * kEmbThr) {            // a wave takes U runs of 64 positions in a row
    int64_t id[U];
    const int p0 = i0 + wave * U * kWave + lane;
#pragma unroll
    for (int u = 0; u < U; ++u) id[u] = ids[p0 + u * kWave < n ? p0 + u * kWave : n - 1];
    uint64_t m[U];
    int mine = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      m[u] = __ballot(p0 + u * kWave < n && id[u] >= v0 && id[u] < v0 + kEmbRows);
      mine += __popcll(m[u]);
    }
    if (lane == 0) counts[wave] = mine;
    __syncthreads();
    int at = total;
    for (int w = 0; w < kEmbWaves; ++w) {
      if (w < wave) at += counts[w];
      total += counts[w];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (m[u] >> lane & 1)
        list[at + __popcll(m[u] & ((1ull << lane) - 1ull))] = (uint16_t)((p0 + u * kWave) << 4 | (int)(id[u] - v0));
      at += __popcll(m[u]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < kEmbRows; ++r) acc[wave][r][lane] = 0.f;
  const int per = (total + kEmbWaves - 1) / kEmbWaves, e0 = wave * per, e1 = e0 + per < total ? e0 + per : total;
  const float* col = dE + (c < d ? c : 0);
  constexpr int R = 16;
  for (int e = e0; e < e1; e += R) {
    float v[R];
    int row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int x = list[e + r < e1 ? e + r : e1 - 1];
      row[r] = x & (kEmbRows - 1);
      v[r] = col[(int64_t)(x >> 4) * d];
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (e + r < e1) acc[wave][row[r]][lane] += v[r];
  }
  __syncthreads();
  for (int r = wave; r < kEmbRows; r += kEmbWaves) {
    const float s = ((acc[0][r][lane] + acc[1][r][lane]) + acc[2][r][lane]) + acc[3][r][lane];
    if (c < d && v0 + r < V) dW[(v0 + r) * d + c] = s;
  }
}

}  // namespace asrn

using namespace asrn;

extern "C" int asrn_embedding_bwd(const float* dE, const int64_t* ids, int64_t n, int64_t V, int32_t d, float* dW,
                                  void* stream) {
  ASRN_REQUIRE(n >= 1 && n <= kEmbMax && V >= 1 && V < (int64_t(1) << 31) && d >= 1,
               "asrn_embedding_bwd: bad sizes n=%lld (1 to %d), V=%lld, d=%d", (long long)n, kEmbMax, (long long)V, d);
  const dim3 grid((unsigned)((V + kEmbRows - 1) / kEmbRows), (unsigned)((d + kWave - 1) / kWave));
  ASRN_REQUIRE(grid.y < 65536, "asrn_embedding_bwd: d=%d too wide", d);
  hipLaunchKernelGGL(k_embedding_bwd, grid, dim3(kEmbThr), 0, (hipStream_t)stream, dE, ids, (int)n, V, d, dW);
  return check_launch("asrn_embedding_bwd");
}
