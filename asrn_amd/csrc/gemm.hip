// Dense products on the bf16 matrix cores with fp32 results: C (M, N) = op(A) op(B) (+ C) (+ bias).
//
// fp32 operands (F32): CDNA4's fp32 matrix rate is 157 TFLOP/s, its bf16 rate 16 times that. An fp32 value from 2^-110
// on is exactly the sum of three bf16 values (24 significand bits in three parts of 8, each part the previous remainder
// rounded to nearest), so a product x y is the sum of nine bf16 products, exact in the fp32 accumulator's input. The
// three smallest (second x third and below, at most 2^-25 of x y) are left out: six bf16 products per fp32 one, an error
// below fp32's own rounding of each product, and fewer roundings of the running sum (one per 16 terms and product
// order). Measured against 64 bits (256 to 65536 terms, centred and positive operands) the products are half as far off as
// the library's fp32 ones or less. Below 2^-110 a remainder may lie under bf16's smallest subnormal, and the value enters
// rounded to a multiple of 2^-133: products of values around 1e-35 are off by 2.7e-6, around 1e-38 by 2.7e-3.
// A value that is not finite, or rounds to infinity in bf16, turns its products into NaN here; results that come out not
// finite are formed again as plain fp32 sums, so infinities and NaN are those of an fp32 product. A wave forms its rows'
// 32 by 32 blocks that hold such results again, the operands through LDS unsplit: a product that is all NaN takes 4 to 5
// times a finite one's time (768 x 3072 over 12000 tokens with one NaN token 338 us finite, 1.5 ms; one result after the
// other by its thread 62 ms), so a training step that is to be skipped stays a step.
// bf16 operands (TN only, the weight gradients): the products as they are, summed in fp32.
//
// The matrix cores drop the low bits of a sum towards minus infinity (measured: 256 terms leave results low by 1.5e-8
// of their root mean square on average, whatever their sign, against 2.4e-7 of random error), which a later sum over
// all tokens would gather. So with the tokens as rows (A not transposed) every other block of rows enters negated and
// leaves negated again, and the errors of neighbouring blocks cancel (a wave stores whole blocks: one uniform branch).
// With the tokens along K (A transposed) the running sums themselves are negated every kTurn tokens, with the values that
// enter from there on, and every other slab of K begins negated: a result's own errors cancel (768 x 3072 over
// 12000 tokens: mean error 4e-7 of the root mean square before, 1e-9 now, their own size 1.03e-6 and 0.96e-6, the
// library's 1.96e-6; 64 x 128 over 65536 2.4e-7, 1e-9, 3.6e-7, 2.7e-7, 2.8e-6). It costs 0 to 4 % (351 us either way at
// the first; 512 x 256 over 5005 with its column sums 21.1 -> 21.9), with a branch a step, the sign as a mask, or a loop for
// each sign alike.
//
// A workgroup of 4 waves forms a BM x BN tile, each wave a quarter of it from 32x32x16 MFMA tiles. Operands are loaded
// into registers one step ahead, split there and stored to LDS in units of 8 consecutive k of one row, the operand an
// MFMA lane takes; an operand stored with its rows contiguous (TA, TB) is transposed on the way, 8 k-rows per thread,
// which costs nothing in fp32 and one permute per pair in bf16. Three workgroups share a CU in fp32 (50,176 bytes of LDS
// and 112 to 164 registers a wave): one's loads, splits and barriers run under the others' MFMA.
// Products with few tiles (weight gradients: K is the token axis) are cut along K: partial products in a workspace,
// summed in order by a second launch. No atomics: the result is a function of the sizes alone.
// The weight gradient's bias gradient, the column sums of A (TA), is summed from the values a tile loads anyway.
#include "common.h"

namespace asrn {

typedef __bf16 bfx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bfx8 __attribute__((ext_vector_type(8)));
typedef float fx2 __attribute__((ext_vector_type(2)));
typedef float fx16 __attribute__((ext_vector_type(16)));

constexpr int kGemmThr = 256;
constexpr int kTurn = 256;      // k between two changes of sign

struct Gemm {
  const void* A; int64_t lda; const void* B; int64_t ldb;
  float* C; int64_t ldc;
  int M, N, K;
  const float* bias;      // (N) or null
  int accumulate;         // C += instead of C =
  float* colsum;          // (M) or null: the sums of A's columns over K (TA)
  float* part;            // splits > 1: the partial products, one row of `pstride` floats per split
  int64_t pstride;
  int splits, kper, tm, tn;
  int tail, tsplits, tkper;   // the last `tail` tiles are cut along K into tsplits slabs of tkper, summed by k_gemm_tail
};

// x, y (NEG: -x, -y) as three bf16 pairs, each the remainder's nearest
template <bool NEG>
__device__ __forceinline__ void split3(float x, float y, uint32_t (&p)[3]) {
  if (NEG) {
    x = -x;
    y = -y;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const fx2 v = {x, y};
    p[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bfx2));
    if (i < 2) {
      x -= __uint_as_float(p[i] << 16);
      y -= __uint_as_float(p[i] & 0xffff0000u);
    }
  }
}

// One operand's share of a K step: R rows (of op(A), or columns of op(B)) by BK. T: stored with the rows contiguous
// (element (k, r) at k * ld + r), else with k contiguous. A thread holds U units of 8 consecutive k.
template <int R, bool T, bool F32, int BK, int THR = kGemmThr>
struct Operand {
  static constexpr int CH = BK / 8;                          // units per row
  static constexpr int U = R * CH / THR;                     // units per thread
  static constexpr int PL = F32 ? 3 : 1;                     // bf16 planes
  // LDS unit of row r in chunk c: bank groups of 8 units. K-contiguous loads write units (c, r) with c fastest, CH to a
  // row: a chunk stride of 8 / CH mod 8 keeps 8 lanes apart. bf16 transposes write rows 4 apart: a spare unit every 8
  // rows.
  static constexpr int CS = F32 ? R + 8 / CH : R + R / 8;
  static constexpr int UNITS = PL * CH * CS;
  static __device__ __forceinline__ int at(int p, int c, int r) {
    return (p * CH + c) * CS + (F32 ? r : r + (r >> 3));
  }
  float f[F32 ? U : 1][8];          // F32: the units' values
  uint32_t w[F32 ? 1 : 8][F32 ? 1 : U / 2];   // bf16: 8 k-rows of U adjacent columns

  static __device__ __forceinline__ void where(int tid, int i, int& c, int& r) {
    if constexpr (T) {
      constexpr int G = R / U;
      c = tid / G;
      r = (tid % G) * U + i;
    } else {
      const int u = tid + THR * i;
      c = u % CH;
      r = u / CH;
    }
  }
  // rows past `rows` repeat the last ones (their results are not stored); k past k1 read as 0
  template <bool FULL>
  __device__ __forceinline__ void load(const void* X, int64_t ld, int r0, int rows, int k0, int k1, int tid) {
    int c, r;
    where(tid, 0, c, r);
    if constexpr (F32 && !T) {
      const float* x = static_cast<const float*>(X);
#pragma unroll
      for (int i = 0; i < U; ++i) {
        where(tid, i, c, r);
        const int row = r0 + r < rows ? r0 + r : rows - 1, k = k0 + 8 * c;
        const float* p = x + (int64_t)row * ld + k;
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        if (FULL || k < k1) lo = *reinterpret_cast<const float4*>(p);
        if (FULL || k + 4 < k1) hi = *reinterpret_cast<const float4*>(p + 4);
        f[i][0] = lo.x; f[i][1] = lo.y; f[i][2] = lo.z; f[i][3] = lo.w;
        f[i][4] = hi.x; f[i][5] = hi.y; f[i][6] = hi.z; f[i][7] = hi.w;
      }
    } else if constexpr (F32) {
      const float* x = static_cast<const float*>(X);
      const int col = r0 + r <= rows - U ? r0 + r : rows - U;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + 8 * c + j;
        const bool ok = FULL || k < k1;
        const float* p = x + (int64_t)(ok ? k : k1 - 1) * ld + col;
        if constexpr (U == 2) {
          const float2 v = *reinterpret_cast<const float2*>(p);
          f[0][j] = ok ? v.x : 0.f;
          f[1][j] = ok ? v.y : 0.f;
        } else {
          const float v = *p;
          f[0][j] = ok ? v : 0.f;
        }
      }
    } else {
      const uint16_t* x = static_cast<const uint16_t*>(X);
      const int col = r0 + r <= rows - U ? r0 + r : rows - U;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + 8 * c + j;
        const bool ok = FULL || k < k1;
        const uint16_t* p = x + (int64_t)(ok ? k : k1 - 1) * ld + col;
        if constexpr (U == 4) {
          const uint2 v = *reinterpret_cast<const uint2*>(p);
          w[j][0] = ok ? v.x : 0u;
          w[j][1] = ok ? v.y : 0u;
        } else {
          const uint32_t v = *reinterpret_cast<const uint32_t*>(p);
          w[j][0] = ok ? v : 0u;
        }
      }
    }
  }
  // rows of a block whose products are formed negated (k-contiguous operands: a wave's 64 / CH rows)
  static constexpr int BLOCK = kWave / CH;
  template <bool NEG>
  __device__ __forceinline__ void store(uint4* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      int c, r;
      where(tid, i, c, r);
      if constexpr (F32) {
        uint32_t q[4][3];
#pragma unroll
        for (int j = 0; j < 4; ++j) split3<NEG>(f[i][2 * j], f[i][2 * j + 1], q[j]);
#pragma unroll
        for (int p = 0; p < 3; ++p) lds[at(p, c, r)] = make_uint4(q[0][p], q[1][p], q[2][p], q[3][p]);
      } else {
        const uint32_t sel = i & 1 ? 0x07060302u : 0x05040100u;   // the high or low halves of two words
        uint32_t q[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = __builtin_amdgcn_perm(w[2 * j + 1][i / 2], w[2 * j][i / 2], sel);
        lds[at(0, c, r)] = make_uint4(q[0], q[1], q[2], q[3]);
      }
    }
  }
  // F32: the units' values as they are, row r of step column k at lds[k * R + r]
  __device__ __forceinline__ void store_raw(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      int c, r;
      where(tid, i, c, r);
#pragma unroll
      for (int j = 0; j < 8; ++j) lds[(8 * c + j) * R + r] = f[i][j];
    }
  }
  // adds this step's values to the thread's U column sums (T)
  __device__ __forceinline__ void column_sums(float (&s)[U]) const {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      float t = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (F32) t += f[i][j];
        else t += __uint_as_float(i & 1 ? w[j][i / 2] & 0xffff0000u : w[j][i / 2] << 16);
      }
      s[i] += t;
    }
  }
};

// k per step: 64 for bf16; for fp32 32, or 64 in the smallest tile, whose few steps wait for their loads
template <int BM, int BN, bool F32>
constexpr int step_k() { return !F32 || BM + BN == 128 ? 64 : 32; }

template <int BM, int BN, bool TA, bool TB, bool F32>
__global__ __launch_bounds__(kGemmThr, 2) void k_gemm(Gemm g) {
  constexpr int BK = step_k<BM, BN, F32>();
  using OA = Operand<BM, TA, F32, BK>;
  using OB = Operand<BN, TB, F32, BK>;
  constexpr int MI = BM / 64, NI = BN / 64, PL = OA::PL;
  // the waves' blocks alternate down a tile: 4 waves of BLOCK rows, then the next unit's
  constexpr bool kSigned = F32 && !TA;
  __shared__ uint4 lds[OA::UNITS + OB::UNITS];
  uint4* la = lds;
  uint4* lb = lds + OA::UNITS;
  // XCD x takes a contiguous range of tiles, n fastest, then m, then the K slabs: tiles that share rows share its L2
  const int whole = g.tm * g.tn * g.splits - g.tail;                // a multiple of the XCDs when tail > 0
  const int first = (whole + kXcdCount - 1) / kXcdCount * kXcdCount;
  const bool cut = (int)blockIdx.x >= first;                          // a slab of a tail tile
  const int total = cut ? g.tail * g.tsplits : whole, blk = (int)blockIdx.x - (cut ? first : 0);
  const int per = (total + kXcdCount - 1) / kXcdCount, t = blk % kXcdCount * per + blk / kXcdCount;
  if (t >= total) return;
  const int tiles = cut ? g.tail : g.tm * g.tn;
  const int z = t / tiles, tile = t % tiles + (cut ? whole : 0), bm = tile / g.tn, bn = tile % g.tn;
  const int kper = cut ? g.tkper : g.kper;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int m0 = bm * BM, n0 = bn * BN, ka = z * kper, kb = ka + kper < g.K ? ka + kper : g.K;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2), lr = lane & 31, lc = lane >> 5;
  const bool sums = TA && g.colsum != nullptr && bn == 0;
  float cs[OA::U];
#pragma unroll
  for (int i = 0; i < OA::U; ++i) cs[i] = 0.f;
  fx16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  OA a;
  OB b;
  auto load = [&](int k) {
    if (k + BK <= kb) {
      a.template load<true>(g.A, g.lda, m0, g.M, k, kb, tid);
      b.template load<true>(g.B, g.ldb, n0, g.N, k, kb, tid);
    } else {
      a.template load<false>(g.A, g.lda, m0, g.M, k, kb, tid);
      b.template load<false>(g.B, g.ldb, n0, g.N, k, kb, tid);
    }
  };
  constexpr bool kTurned = F32 && TA;
  bool negated = kTurned && (z & 1);              // what the sums hold; uniform
  int steps = kTurn / BK;
  if (ka < kb) load(ka);
  for (int k = ka; k < kb; k += BK) {
    __syncthreads();                              // the last step's LDS reads are done
    if constexpr (kTurned) {
      if (steps-- == 0) {
        steps = kTurn / BK - 1;
        negated = !negated;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = -acc[i][j];
      }
    }
    if ((kSigned && (wave & 1)) || (kTurned && negated)) a.template store<true>(la, tid);
    else a.template store<false>(la, tid);
    b.template store<false>(lb, tid);
    if (TA && sums) a.column_sums(cs);
    __syncthreads();
    if (k + BK < kb) load(k + BK);                // in flight under this step's products
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bfx8 fa[MI][PL], fb[NI][PL];
#pragma unroll
      for (int p = 0; p < PL; ++p) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          fa[i][p] = __builtin_bit_cast(bfx8, la[OA::at(p, 2 * kk + lc, wm + 32 * i + lr)]);
#pragma unroll
        for (int j = 0; j < NI; ++j)
          fb[j][p] = __builtin_bit_cast(bfx8, lb[OB::at(p, 2 * kk + lc, wn + 32 * j + lr)]);
      }
#pragma unroll
      for (int q = PL - 1; q >= 0; --q)           // the products of parts pa + pb = q, smallest first
#pragma unroll
        for (int pa = 0; pa <= q; ++pa)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][pa], fb[j][q - pa], acc[i][j], 0, 0, 0);
    }
  }
  float* out = cut ? g.part + ((int64_t)t * BM - m0) * BN - n0 : g.splits > 1 ? g.part + (int64_t)z * g.pstride : g.C;
  const int64_t ldo = cut ? BN : g.splits > 1 ? g.N : g.ldc;
  const bool last = g.splits == 1 && !cut;
  uint64_t bad = 0;                               // results to form again (bit (i NI + j) 16 + e)
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n0 + wn + 32 * j + lr;
      const float bias = last && g.bias && n < g.N ? g.bias[n] : 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * lc + (e & 3);
        if (m < g.M && n < g.N) {
          float v = acc[i][j][e];
          if (kSigned && ((8 * (e >> 2)) / OA::BLOCK & 1)) v = -v;     // BLOCK is 16 or 8: the block's parity
          if (kTurned && negated) v = -v;
          if (F32 && !(fabsf(v) < INFINITY)) {
            bad |= 1ull << ((i * NI + j) * 16 + e);
          } else {
            float* o = out + (int64_t)m * ldo + n;
            if (last) v += bias;
            if (last && g.accumulate) v += *o;
            *o = v;
          }
        }
      }
    }
  if constexpr (F32) {
    if (__syncthreads_or(bad != 0)) {             // uniform: once more as plain fp32 sums, k in order
      static_assert(BK * (BM + BN) * 4 <= sizeof(lds), "the values of a step fit where their parts did");
      float* ra = reinterpret_cast<float*>(lds);
      float* rb = ra + BK * BM;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
      bool some[MI];                              // whether the wave has such results in its rows' i-th 32 (uniform)
#pragma unroll
      for (int i = 0; i < MI; ++i) some[i] = __any((bad >> (i * NI * 16) & ((1ull << NI * 16) - 1)) != 0);
      load(ka);
      for (int k = ka; k < kb; k += BK) {
        __syncthreads();
        a.store_raw(ra, tid);
        b.store_raw(rb, tid);
        __syncthreads();
        if (k + BK < kb) load(k + BK);
#pragma unroll 2
        for (int kk = 0; kk < BK; ++kk) {         // past kb both operands are 0
          float y[NI];
#pragma unroll
          for (int j = 0; j < NI; ++j) y[j] = rb[kk * BN + wn + 32 * j + lr];
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            if (!some[i]) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float4 x = *reinterpret_cast<const float4*>(ra + kk * BM + wm + 32 * i + 8 * q + 4 * lc);
#pragma unroll
              for (int j = 0; j < NI; ++j) {
                acc[i][j][4 * q] = fmaf(x.x, y[j], acc[i][j][4 * q]);
                acc[i][j][4 * q + 1] = fmaf(x.y, y[j], acc[i][j][4 * q + 1]);
                acc[i][j][4 * q + 2] = fmaf(x.z, y[j], acc[i][j][4 * q + 2]);
                acc[i][j][4 * q + 3] = fmaf(x.w, y[j], acc[i][j][4 * q + 3]);
              }
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int n = n0 + wn + 32 * j + lr;
          const float bias = last && g.bias && n < g.N ? g.bias[n] : 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            if (!(bad >> ((i * NI + j) * 16 + e) & 1)) continue;     // inside the matrix, and not stored above
            const int m = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * lc + (e & 3);
            float* o = out + (int64_t)m * ldo + n;
            float v = acc[i][j][e] + bias;
            if (last && g.accumulate) v += *o;
            *o = v;
          }
        }
    }
  }
  if constexpr (TA) {
    if (sums) {                                   // uniform: the chunks' sums of a row combine in order
      float* red = reinterpret_cast<float*>(lds);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < OA::U; ++i) {
        int c, r;
        OA::where(tid, i, c, r);
        red[c * BM + r] = cs[i];
      }
      __syncthreads();
      if (tid < BM && m0 + tid < g.M) {
        float v = 0.f;
#pragma unroll
        for (int c = 0; c < OA::CH; ++c) v += red[c * BM + tid];
        (last ? g.colsum : out + (int64_t)g.M * g.N)[m0 + tid] = v;
      }
    }
  }
}

// The largest bf16 weight gradients: 256 x 256 tiles of 8 waves, 128 x 64 results each, one workgroup a CU. Wider wave
// tiles read less LDS per product (with 64 x 64 a wave's reads and the stores take longer than its MFMA), and two LDS
// buffers leave one barrier per 64 k: a step's loads are issued at its end and first waited for three quarters into the
// next one's products (the scheduling barrier: the compiler would wait at once), split and stored between the rest.
// With their sums (us, tiles of 256 x 128 or 128 x 128 / these): 768 x 3072 over 16384 tokens 134 / 120, 768 x 1536
// 82 / 72, 512 x 2048 over 65536 240 / 187; 1536 x 768 over 8192 53.3 / 52.2, over 4097 38.7 / 42.4 (too few steps a
// workgroup).
constexpr int kWideThr = 512;
__global__ __launch_bounds__(kWideThr, 2) void k_gemm_wide(Gemm g) {
  constexpr int BM = 256, BN = 256, BK = 64, HEAD = 3;    // HEAD: 16-deep products before the loads are waited for
  using O = Operand<256, true, false, BK, kWideThr>;
  constexpr int WN = 4, MI = 4, NI = BN / WN / 32;
  __shared__ uint4 lds[4 * O::UNITS];
  const int total = g.tm * g.tn * g.splits, per = (total + kXcdCount - 1) / kXcdCount;
  const int t = (int)(blockIdx.x % kXcdCount) * per + (int)(blockIdx.x / kXcdCount);
  if (t >= total) return;
  const int z = t / (g.tm * g.tn), tile = t % (g.tm * g.tn), bm = tile / g.tn, bn = tile % g.tn;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int m0 = bm * BM, n0 = bn * BN, ka = z * g.kper, kb = ka + g.kper < g.K ? ka + g.kper : g.K;
  const int wm = wave / WN * 128, wn = wave % WN * (BN / WN), lr = lane & 31, lc = lane >> 5;
  const bool sums = g.colsum != nullptr && bn == 0;
  float cs[O::U];
#pragma unroll
  for (int i = 0; i < O::U; ++i) cs[i] = 0.f;
  fx16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  auto load = [&](O& a, O& b, int k) {
    if (k + BK <= kb) {
      a.template load<true>(g.A, g.lda, m0, g.M, k, kb, tid);
      b.template load<true>(g.B, g.ldb, n0, g.N, k, kb, tid);
    } else {
      a.template load<false>(g.A, g.lda, m0, g.M, k, kb, tid);
      b.template load<false>(g.B, g.ldb, n0, g.N, k, kb, tid);
    }
  };
  uint4* l0 = lds;
  uint4* l1 = lds + 2 * O::UNITS;
  auto products = [&](int k0, int k1) {
#pragma unroll
    for (int kk = k0; kk < k1; ++kk) {
      bfx8 fa[MI], fb[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) fa[i] = __builtin_bit_cast(bfx8, l0[O::at(0, 2 * kk + lc, wm + 32 * i + lr)]);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        fb[j] = __builtin_bit_cast(bfx8, l0[O::UNITS + O::at(0, 2 * kk + lc, wn + 32 * j + lr)]);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  };
  O a, b;
  auto store = [&](uint4* l) {
    a.template store<false>(l, tid);
    b.template store<false>(l + O::UNITS, tid);
    if (sums) a.column_sums(cs);
  };
  auto swap = [&]() {
    uint4* x = l0;
    l0 = l1;
    l1 = x;
  };
  load(a, b, ka);                                 // kper > 0 and z < splits: ka < kb
  store(l0);
  if (ka + BK < kb) load(a, b, ka + BK);
  __syncthreads();
  int k = ka;
  for (; k + 3 * BK <= kb; k += BK) {             // step k's products, step k + 1 to LDS, step k + 2 on its way
    products(0, HEAD);
    __builtin_amdgcn_sched_barrier(0);
    products(HEAD, BK / 16);
    store(l1);
    a.template load<true>(g.A, g.lda, m0, g.M, k + 2 * BK, kb, tid);
    b.template load<true>(g.B, g.ldb, n0, g.N, k + 2 * BK, kb, tid);
    __syncthreads();
    swap();
  }
  for (; k + BK < kb; k += BK) {
    products(0, HEAD);
    __builtin_amdgcn_sched_barrier(0);
    products(HEAD, BK / 16);
    store(l1);
    if (k + 2 * BK < kb) load(a, b, k + 2 * BK);
    __syncthreads();
    swap();
  }
  products(0, BK / 16);
  float* out = g.splits > 1 ? g.part + (int64_t)z * g.pstride : g.C;
  const int64_t ldo = g.splits > 1 ? g.N : g.ldc;
  const bool last = g.splits == 1;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n0 + wn + 32 * j + lr;
      const float bias = last && g.bias && n < g.N ? g.bias[n] : 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * lc + (e & 3);
        if (m < g.M && n < g.N) {
          float* o = out + (int64_t)m * ldo + n;
          float v = acc[i][j][e];
          if (last) v += bias;
          if (last && g.accumulate) v += *o;
          *o = v;
        }
      }
    }
  if (sums) {                                     // uniform: the chunks' sums of a row combine in order
    float* red = reinterpret_cast<float*>(lds);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < O::U; ++i) {
      int c, r;
      O::where(tid, i, c, r);
      red[c * BM + r] = cs[i];
    }
    __syncthreads();
    if (tid < BM && m0 + tid < g.M) {
      float v = 0.f;
#pragma unroll
      for (int c = 0; c < O::CH; ++c) v += red[c * BM + tid];
      (last ? g.colsum : out + (int64_t)g.M * g.N)[m0 + tid] = v;
    }
  }
}

// C (+)= the sum of the partial products in split order (+ bias), and the column sums behind them. A workgroup takes
// 32 float4 columns by 8 lanes of splits; the lanes combine in order.
constexpr int kSumCols = 32, kSumLanes = kGemmThr / kSumCols;
__global__ __launch_bounds__(kGemmThr) void k_gemm_sum(Gemm g) {
  __shared__ float4 red[kSumLanes][kSumCols];
  const int cl = threadIdx.x % kSumCols, sl = threadIdx.x / kSumCols;
  const int64_t c = ((int64_t)blockIdx.x * kSumCols + cl) * 4, mn = (int64_t)g.M * g.N;
  const bool live = c < g.pstride;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
    const float* p = g.part + c;
    for (int z = sl; z < g.splits; z += 8 * kSumLanes) {
      float4 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int y = z + q * kSumLanes;
        v[q] = *reinterpret_cast<const float4*>(p + (int64_t)(y < g.splits ? y : z) * g.pstride);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (z + q * kSumLanes < g.splits) {
          s.x += v[q].x; s.y += v[q].y; s.z += v[q].z; s.w += v[q].w;
        }
    }
  }
  red[sl][cl] = s;
  __syncthreads();
  if (sl != 0 || !live) return;
#pragma unroll
  for (int l = 1; l < kSumLanes; ++l) {
    const float4 v = red[l][cl];
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  if (c >= mn) {
    *reinterpret_cast<float4*>(g.colsum + (c - mn)) = s;
    return;
  }
  const int64_t m = c / g.N, n = c - m * g.N;
  float* o = g.C + m * g.ldc + n;
  if (g.bias) { s.x += g.bias[n]; s.y += g.bias[n + 1]; s.z += g.bias[n + 2]; s.w += g.bias[n + 3]; }
  if (g.accumulate) {
    const float4 v = *reinterpret_cast<const float4*>(o);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  *reinterpret_cast<float4*>(o) = s;
}

// The tail tiles: C (+)= the sum of their slabs in order (+ bias), one float4 a thread.
__global__ __launch_bounds__(kGemmThr) void k_gemm_tail(Gemm g, int bm, int bn) {
  const int e = ((int)blockIdx.x * kGemmThr + (int)threadIdx.x) * 4, size = bm * bn, tl = e / size, r = e - tl * size;
  if (tl >= g.tail) return;
  const int tile = g.tm * g.tn - g.tail + tl, m = tile / g.tn * bm + r / bn, n = tile % g.tn * bn + r % bn;
  if (m >= g.M || n >= g.N) return;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  const float* p = g.part + e;
  const int64_t stride = (int64_t)g.tail * size;
#pragma unroll 4
  for (int z = 0; z < g.tsplits; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(p + z * stride);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  float* o = g.C + (int64_t)m * g.ldc + n;
  if (g.bias) { s.x += g.bias[n]; s.y += g.bias[n + 1]; s.z += g.bias[n + 2]; s.w += g.bias[n + 3]; }
  if (g.accumulate) {
    const float4 v = *reinterpret_cast<const float4*>(o);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  *reinterpret_cast<float4*>(o) = s;
}

struct Plan { int bm, bn, splits, kper, tail, tsplits, tkper; };

constexpr int kSlots = 512;     // workgroups that a plan counts on running at once, 2 a CU

// The tile and the slabs of K by the sizes. Each line with both sides measured (us, without the column sums):
// 128 x 128 in fp32 from 448 of them on: a smaller one splits its operands' values more often, but fewer large ones leave
//   slots idle. 64 / 128: 4096 x 768 x 768 (192 tiles) 45 / 49, 4096 x 1536 x 256 (384) 28.5 / 29.3, 7168 x 1024 x 256
//   (448) 34 / 30, 9600 x 768 x 768 (450) 87 / 68; at 384 to 447 tiles the long K already gain (8192 x 768 x 768 73 / 65).
//   And for weights of 768 x 768 on over 2,048 and more, whose slabs fill the slots: 768 x 768 over 1536 28 / 31, over 2048
//   33 / 32, over 4096 54 / 44, over 16384 179 / 119; just below that size 704 x 768 over 8192 92 / 69.
// 256 x 256 in bf16 from 2^20 elements on where a workgroup has steps enough: 9.6e9 multiply-adds, or twice the elements.
//   128 / 256: 1024 x 1024 over 8192 (8.6e9) 47 / 49, 768 x 1536 over 8192 (9.7e9) 52 / 52, over 10000 58 / 57, over 16384
//   80 / 72; 768 x 3072 over 4096 58 / 58, over 8192 89 / 76.
// The slabs fill the slots once (256 of the 256 x 256 tiles, one a CU): 768 x 3072 over 12000 (144 tiles) in 2, 3, 4 slabs
//   460 / 350 / 411; 768 x 1536 over 12000 (72) in 4, 7, 14 236 / 172 / 198. A slab holds at least 64 of K, and 256 past
//   K = 4096, for the sum over the slabs: 64 x 64 over 4096 in 32, 64 10.1 / 8.6; 128 x 128 over 16384 in 64, 128 15.6 /
//   16.3, 256 x 256 over 8192 in 32, 64 20 / 23, though 64 x 64 over 8192 in 32, 64 13.4 / 10.3.
// From 128 tiles on a K of up to 1,024 stays whole: 768 x 768 x 512 in 1, 3 slabs 15 / 16, 2048 x 512 x 1024 26 / 31,
//   2304 x 256 x 768 20 / 19; at 128 to 144 tiles and the longest K it would gain (1024 x 512 x 1000 in 1, 4 25 / 19).
// 64 x 128 and 128 x 64 are the caller's to ask for: between the two square ones nearly everywhere (768 x 768 over 4096 54 /
//   48 / 49 / 44), ahead of both where those are about equal (4096 x 768 x 768 39 against 45 and 49).
static Plan plan_of(int64_t M, int64_t N, int64_t K, bool f32, int tile, int splits) {
  Plan p;
  if (tile) {
    p.bm = tile >> 8;
    p.bn = tile & 255 ? tile & 255 : 256;
  } else {
    p.bm = p.bn = 64;
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    if (M > 64 && N > 64 && (t128 >= 448 || (M * N >= 768 * 768 && K >= 2048))) p.bm = p.bn = 128;
    if (!f32 && M * N >= 1 << 20 && (M * N >= 2 << 20 || (double)M * N * K >= 9.6e9)) p.bm = p.bn = 256;
  }
  const int bk = !f32 || p.bm + p.bn == 128 ? 64 : 32;
  const int64_t tiles = ((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
  int64_t s = splits;
  if (s <= 0) {
    s = (p.bn == 256 ? 256 : 512) / tiles;
    const int64_t most = K <= 4096 ? K / 64 : K / 256;
    if (s > most) s = most;
    if (tiles >= 128 && K <= 1024) s = 1;
  }
  if (s < 1) s = 1;
  const int64_t steps = (K + bk - 1) / bk;
  if (s > steps) s = steps > 0 ? steps : 1;
  p.kper = (int)((steps + s - 1) / s) * bk;
  p.splits = (int)((K + p.kper - 1) / p.kper);
  // A second round that fills less than half of the slots leaves most CUs idle: its tiles are cut along K over all of
  // them (12000 x 768 x 3072, 564 tiles: 354 -> 303 us; 12000 x 768 x 1536 178 -> 155; 9000 x 1024 x 512 68 -> 61).
  // Past two rounds it gains nothing (12000 x 1536 x 768, 1128 tiles: 162 -> 164 us).
  p.tail = p.tsplits = p.tkper = 0;
  const int64_t left = tiles % kSlots;
  if (f32 && splits == 0 && p.splits == 1 && tiles > kSlots && tiles < 2 * kSlots) {
    int64_t ts = kSlots / left;
    if (ts > K / 128) ts = K / 128;
    if (ts > 1) {
      p.tkper = (int)((steps + ts - 1) / ts) * bk;
      p.tsplits = (int)((K + p.tkper - 1) / p.tkper);
      p.tail = (int)left;
    }
  }
  return p;
}

template <int BM, int BN, bool F32>
static void launch_tile(bool ta, bool tb, const Gemm& g, unsigned grid, hipStream_t st) {
  if constexpr (!F32) {
    hipLaunchKernelGGL((k_gemm<BM, BN, true, true, false>), dim3(grid), dim3(kGemmThr), 0, st, g);
  } else {
    if (ta && tb) hipLaunchKernelGGL((k_gemm<BM, BN, true, true, true>), dim3(grid), dim3(kGemmThr), 0, st, g);
    else if (tb) hipLaunchKernelGGL((k_gemm<BM, BN, false, true, true>), dim3(grid), dim3(kGemmThr), 0, st, g);
    else hipLaunchKernelGGL((k_gemm<BM, BN, false, false, true>), dim3(grid), dim3(kGemmThr), 0, st, g);
  }
}

}  // namespace asrn

using namespace asrn;

extern "C" int64_t asrn_gemm_workspace(int64_t M, int64_t N, int64_t K, int32_t bf16, int32_t colsum, int32_t tile,
                                       int32_t splits) {
  if (M < 0 || N < 0 || K < 0) return -1;
  if (M == 0 || N == 0) return 0;
  const Plan p = plan_of(M, N, K, !bf16, tile, splits);
  if (p.tail && !colsum) return (int64_t)p.tail * p.tsplits * p.bm * p.bn * 4;
  return p.splits > 1 ? (int64_t)p.splits * (M * N + (colsum ? M : 0)) * 4 : 0;
}

extern "C" int asrn_gemm(const void* A, int64_t lda, int32_t trans_a, const void* B, int64_t ldb, int32_t trans_b,
                         int32_t bf16, float* C, int64_t ldc, int64_t M, int64_t N, int64_t K, const float* bias,
                         int32_t accumulate, float* colsum, int32_t tile, int32_t splits, void* workspace,
                         int64_t workspace_bytes, void* stream) {
  // op(A) (M, K): trans_a: stored (K, M). op(B) (K, N): trans_b: stored (N, K)
  const bool ta = trans_a != 0, rows_b = trans_b == 0;     // rows_b: B's n contiguous
  ASRN_REQUIRE(M >= 0 && N >= 0 && K >= 1 && M < (1 << 30) && N < (1 << 30) && K < (1 << 30),
               "asrn_gemm: bad sizes M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  if (M == 0 || N == 0) return 0;
  ASRN_REQUIRE(!(ta && !rows_b), "asrn_gemm: A^T B^T is not supported");
  ASRN_REQUIRE(!bf16 || (ta && rows_b), "asrn_gemm: bf16 operands are for A^T B");
  ASRN_REQUIRE(N % 4 == 0 && (!ta || M % 4 == 0) && ((ta && rows_b) || K % 4 == 0),
               "asrn_gemm: N, and M (A transposed) or K (an operand with k contiguous), must be multiples of 4");
  ASRN_REQUIRE(lda % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0 && lda >= (ta ? M : K) && ldb >= (rows_b ? N : K) &&
                   ldc >= N, "asrn_gemm: leading dimensions must be multiples of 4 that hold a row (lda=%lld ldb=%lld "
               "ldc=%lld)", (long long)lda, (long long)ldb, (long long)ldc);
  const uintptr_t al = bf16 ? 7 : 15;
  ASRN_REQUIRE(A && B && C && ((uintptr_t)A & al) == 0 && ((uintptr_t)B & al) == 0 && ((uintptr_t)C & 15) == 0 &&
                   ((uintptr_t)bias & 15) == 0 && ((uintptr_t)colsum & 15) == 0, "asrn_gemm: misaligned operand");
  ASRN_REQUIRE(colsum == nullptr || ta, "asrn_gemm: column sums are those of A^T's A");
  ASRN_REQUIRE(tile == 0 || tile == (128 << 8 | 128) || tile == (64 << 8 | 128) || tile == (128 << 8 | 64) ||
                   tile == (64 << 8 | 64) || (bf16 && tile == 256 << 8), "asrn_gemm: unknown tile %d", tile);
  Plan p = plan_of(M, N, K, !bf16, tile, splits);
  if (colsum) p.tail = 0;                                  // only whole tiles sum A's columns
  Gemm g = {A, lda, B, ldb, C, ldc, (int)M, (int)N, (int)K, bias, accumulate ? 1 : 0, colsum, (float*)workspace,
            M * N + (colsum ? M : 0), p.splits, p.kper, (int)((M + p.bm - 1) / p.bm), (int)((N + p.bn - 1) / p.bn),
            p.tail, p.tsplits, p.tkper};
  const int64_t total = (int64_t)g.tm * g.tn * g.splits;
  ASRN_REQUIRE(total < (1 << 30), "asrn_gemm: too many tiles");
  if (p.splits > 1)
    ASRN_REQUIRE(workspace && workspace_bytes >= p.splits * g.pstride * 4 && ((uintptr_t)workspace & 15) == 0,
                 "asrn_gemm: needs a 16-byte aligned workspace of %lld bytes (got %lld)",
                 (long long)(p.splits * g.pstride * 4), (long long)workspace_bytes);
  const int64_t slabs = (int64_t)p.tail * p.tsplits, slab_bytes = slabs * p.bm * p.bn * 4;
  if (p.tail)
    ASRN_REQUIRE(workspace && workspace_bytes >= slab_bytes && ((uintptr_t)workspace & 15) == 0,
                 "asrn_gemm: needs a 16-byte aligned workspace of %lld bytes (got %lld)", (long long)slab_bytes,
                 (long long)workspace_bytes);
  hipStream_t st = (hipStream_t)stream;
  auto blocks = [](int64_t n) { return (n + kXcdCount - 1) / kXcdCount * kXcdCount; };
  const unsigned grid = (unsigned)(blocks(total - p.tail) + blocks(slabs));
  if (bf16) {
    if (p.bn == 256)
      hipLaunchKernelGGL(k_gemm_wide, dim3(grid), dim3(kWideThr), 0, st, g);
    else if (p.bm == 128 && p.bn == 128) launch_tile<128, 128, false>(ta, rows_b, g, grid, st);
    else if (p.bm == 128) launch_tile<128, 64, false>(ta, rows_b, g, grid, st);
    else if (p.bn == 128) launch_tile<64, 128, false>(ta, rows_b, g, grid, st);
    else launch_tile<64, 64, false>(ta, rows_b, g, grid, st);
  } else {
    if (p.bm == 128 && p.bn == 128) launch_tile<128, 128, true>(ta, rows_b, g, grid, st);
    else if (p.bm == 128) launch_tile<128, 64, true>(ta, rows_b, g, grid, st);
    else if (p.bn == 128) launch_tile<64, 128, true>(ta, rows_b, g, grid, st);
    else launch_tile<64, 64, true>(ta, rows_b, g, grid, st);
  }
  int rc = check_launch("asrn_gemm");
  if (rc == 0 && p.tail) {
    hipLaunchKernelGGL(k_gemm_tail, dim3((unsigned)(p.tail * (p.bm * p.bn / 4 / kGemmThr))), dim3(kGemmThr), 0, st, g, p.bm,
                       p.bn);
    return check_launch("asrn_gemm");
  }
  if (rc || p.splits == 1) return rc;
  const int64_t cols = (g.pstride + 4 * kSumCols - 1) / (4 * kSumCols);
  hipLaunchKernelGGL(k_gemm_sum, dim3((unsigned)cols), dim3(kGemmThr), 0, st, g);
  return check_launch("asrn_gemm");
}
