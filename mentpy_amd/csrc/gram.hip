// Complex products of the MB-QML losses on the matrix cores (gfx950): the rows
// vec(T_b) of the sets' transfer matrices times the data matrix, with the loss
// partial sums and the seed's scale taken from the accumulators, so that the
// product itself is not stored and read again.
//
// A complex product is four real v_mfma_f32 per operand pair (Zr += Ar Br - Ai Bi,
// Zi += Ar Bi + Ai Br) in float32.  Operands go from the caches straight to
// registers, one step ahead of their products: at 32 x 32 a wave's 8 KB of operands
// per 16 k last 2048 matrix-core cycles, so the LDS would save nothing.  A lane takes
// consecutive k (any assignment of k to lanes will do, if both operands share
// it), so that A is read in runs along its rows.
#include "gram.h"

#include "device.h"

namespace mbqc {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct Operands {
  const float2* A;
  const float2* B;
  float2* C;
  float* part;
  int64_t M;
  int N, K;
  float scale;
};

// One entry of the result; returns its loss partial.
template <Product W>
__device__ __forceinline__ float finish(const Operands& g, int64_t row, int col, float2 z) {
  const int64_t at = row * g.N + col;
  if constexpr (W == Product::kOverlap) {
    if (g.C) g.C[at] = z;
    return fmaf(z.x, z.x, z.y * z.y);
  } else {
    float p = 0.0f;
    if constexpr (W == Product::kGram) {
      const float2 x = g.A[at];
      p = fmaf(x.x, z.x, x.y * z.y);
    }
    g.C[at] = cscale(z, g.scale);
    return p;
  }
}

// Many rows: a workgroup takes 64 x 64 of the result, a wave 32 x 32.  MFMA
// 32x32x2: lane l holds A[l % 32][l / 32] and B[l / 32][l % 32], the accumulator
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32], r = 0..15.  A step takes 16 k, whole
// 128-byte lines of A.  LONG (K > 64): partial sums of 64 k are added up, so that
// the rounding error of a long sum stays below that of the library products
// (gradients of 8,000 sets of a 4x4 grid against 64 bits: 6.5e-7, one sum 8.8e-7,
// library 7.6e-7); steps of 8 k leave it the registers for four waves per SIMD.
// 16,384 x 256 x 256: 82 us, LONG 91 us, of 57 us for the products alone: what is not
// hidden are the first loads and the stores, all waves being resident at once.
template <Product W, bool LONG>
__global__ __launch_bounds__(256, 4) void k_product_large(Operands g) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = l & 31, h = l >> 5;
  const int nt = (g.N + 63) / 64;
  const int tile = xcd_block(blockIdx.x, gridDim.x);
  const int64_t m0 = int64_t(tile / nt) * 64 + (w >> 1) * 32;
  const int n0 = (tile % nt) * 64 + (w & 1) * 32;
  if (m0 >= g.M || n0 >= g.N) return;
  // rows and columns past the end repeat the last one and are not stored
  const int64_t row = m0 + li < g.M ? m0 + li : g.M - 1;
  const int col = n0 + li < g.N ? n0 + li : g.N - 1;
  constexpr int KS = LONG ? 8 : 16, U = KS / 2;
  const float2* pa = g.A + row * g.K + U * h;
  const float2* pb = g.B + int64_t(U * h) * g.N + col;
  f32x16 zr, zi, sr, si;
#pragma unroll
  for (int r = 0; r < 16; ++r) zr[r] = zi[r] = sr[r] = si[r] = 0.0f;
  float2 an[U], bn[U];
  auto fetch = [&]() {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      an[j] = pa[j];
      bn[j] = pb[int64_t(j) * g.N];
    }
    pa += KS;
    pb += int64_t(KS) * g.N;
  };
  auto multiply = [&](const float2 (&a)[U], const float2 (&b)[U]) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      zr = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].x, b[j].x, zr, 0, 0, 0);
      zi = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].x, b[j].y, zi, 0, 0, 0);
      zr = __builtin_amdgcn_mfma_f32_32x32x2f32(-a[j].y, b[j].y, zr, 0, 0, 0);
      zi = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].y, b[j].x, zi, 0, 0, 0);
    }
  };
  const int steps = g.K / KS, rest = g.K % KS;
  if (steps) fetch();
  for (int i = 0; i < steps; ++i) {
    float2 a[U], b[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      a[j] = an[j];
      b[j] = bn[j];
    }
    if (i + 1 < steps) fetch();
    multiply(a, b);
    if constexpr (LONG) {
      if (i % (64 / KS) == 64 / KS - 1) {
        sr += zr;
        si += zi;
#pragma unroll
        for (int r = 0; r < 16; ++r) zr[r] = zi[r] = 0.0f;
      }
    }
  }
  if (rest) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const bool in = U * h + j < rest;
      an[j] = in ? pa[j] : make_float2(0.0f, 0.0f);
      bn[j] = in ? pb[int64_t(j) * g.N] : make_float2(0.0f, 0.0f);
    }
    multiply(an, bn);
  }
  if constexpr (LONG) {
    zr += sr;
    zi += si;
  }
  const int tiles = (g.N + 31) / 32;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t b = m0 + 8 * (r >> 2) + 4 * h + (r & 3);   // uniform over 32 lanes
    float p = 0.0f;
    if (b < g.M && n0 + li < g.N) p = finish<W>(g, b, n0 + li, make_float2(zr[r], zi[r]));
    if constexpr (W != Product::kScaled) {
      p = last_lane_sum<32>(p);
      if (li == 31 && b < g.M) g.part[b * tiles + n0 / 32] = p;
    }
  }
}

// Few rows: a workgroup takes 16 x 16, its four waves a quarter of the k's each,
// so that four times the waves hide each other's loads.  MFMA 16x16x4: lane l
// holds A[l % 16][l / 16] and B[l / 16][l % 16], the accumulator
// D[4 (l / 16) + r][l % 16], r = 0..3.  A sum has K / 8 of the k's; LONG (K > 512):
// partial sums of 64 k are added up, as in k_product_large.  (Gradients of 2,000 sets
// of a 5x4 grid with 64 inputs, K = 1,024, against 64 bits: 1.57e-9 with library
// products, 1.66e-9 in one sum, 1.49e-9 so; times level.)
template <Product W, bool LONG>
__global__ __launch_bounds__(256, 4) void k_product_small(Operands g) {
  __shared__ float2 red[4 * 16 * 17];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = l & 15, h = l >> 4;
  const int tiles = (g.N + 15) / 16;
  const int tile = xcd_block(blockIdx.x, gridDim.x);
  const int64_t m0 = int64_t(tile / tiles) * 16;
  const int n0 = (tile % tiles) * 16;
  const int64_t row = m0 + li < g.M ? m0 + li : g.M - 1;
  const int col = n0 + li < g.N ? n0 + li : g.N - 1;
  const float2* pa = g.A + row * g.K;
  const float2* pb = g.B + col;
  // two accumulators per part: shorter sums, and no product waits for the last one
  f32x4 zr[2], zi[2], sr, si;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < 2; ++i) zr[i] = zi[i] = zero;
  sr = si = zero;
  constexpr int U = 2;                       // chunks of 16 k loaded together
  [[maybe_unused]] int terms = 0;            // k's of each accumulator
  for (int k0 = 16 * w; k0 < g.K; k0 += 64 * U) {
    if constexpr (LONG) {
      if (terms == 64) {
        sr += zr[0] + zr[1];
        si += zi[0] + zi[1];
#pragma unroll
        for (int i = 0; i < 2; ++i) zr[i] = zi[i] = zero;
        terms = 0;
      }
      terms += 8 * U;
    }
    float2 a[4 * U], b[4 * U];
    if (k0 + 64 * (U - 1) + 16 <= g.K) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = k0 + 64 * u + 4 * h + j;
          a[4 * u + j] = pa[k];
          b[4 * u + j] = pb[int64_t(k) * g.N];
        }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + 64 * u + 4 * h + j;
        const bool in = k < g.K;
        a[4 * u + j] = in ? pa[k] : make_float2(0.0f, 0.0f);
        b[4 * u + j] = in ? pb[int64_t(k) * g.N] : make_float2(0.0f, 0.0f);
      }
    }
#pragma unroll
    for (int i = 0; i < 4 * U; ++i) {
      if (i % 4 == 0 && k0 + 16 * i >= g.K) break;
      const int q = i % 2;
      zr[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].x, zr[q], 0, 0, 0);
      zi[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].y, zi[q], 0, 0, 0);
      zr[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(-a[i].y, b[i].y, zr[q], 0, 0, 0);
      zi[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[i].x, zi[q], 0, 0, 0);
    }
  }
  zr[0] += zr[1];
  zi[0] += zi[1];
  if constexpr (LONG) {
    zr[0] += sr;
    zi[0] += si;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    red[(w * 16 + 4 * h + r) * 17 + li] = make_float2(zr[0][r], zi[0][r]);
  __syncthreads();
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  float2 z = red[r * 17 + c];
#pragma unroll
  for (int i = 1; i < 4; ++i) z = cadd(z, red[(i * 16 + r) * 17 + c]);
  float p = 0.0f;
  if (m0 + r < g.M && n0 + c < g.N) p = finish<W>(g, m0 + r, n0 + c, z);
  if constexpr (W != Product::kScaled) {
    p = last_lane_sum<16>(p);
    if (c == 15 && m0 + r < g.M) g.part[(m0 + r) * tiles + n0 / 16] = p;
  }
}

// In between: a workgroup takes 32 x 32, its four waves a quarter of the k's each
// (16 at a time, whole lines of A): half the operand bytes of k_product_small.
template <Product W>
__global__ __launch_bounds__(256, 2) void k_product_mid(Operands g) {
  __shared__ float2 red[4 * 32 * 33];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = l & 31, h = l >> 5;
  const int tiles = (g.N + 31) / 32;
  const int tile = xcd_block(blockIdx.x, gridDim.x);
  const int64_t m0 = int64_t(tile / tiles) * 32;
  const int n0 = (tile % tiles) * 32;
  const int64_t row = m0 + li < g.M ? m0 + li : g.M - 1;
  const int col = n0 + li < g.N ? n0 + li : g.N - 1;
  const float2* pa = g.A + row * g.K;
  const float2* pb = g.B + col;
  f32x16 zr, zi;
#pragma unroll
  for (int r = 0; r < 16; ++r) zr[r] = zi[r] = 0.0f;
  float2 an[8], bn[8];
  auto fetch = [&](int k0) {
    const int k1 = k0 + 8 * h;
    if (k0 + 16 <= g.K) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        an[j] = pa[k1 + j];
        bn[j] = pb[int64_t(k1 + j) * g.N];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool in = k1 + j < g.K;
        an[j] = in ? pa[k1 + j] : make_float2(0.0f, 0.0f);
        bn[j] = in ? pb[int64_t(k1 + j) * g.N] : make_float2(0.0f, 0.0f);
      }
    }
  };
  if (16 * w < g.K) fetch(16 * w);
  for (int k0 = 16 * w; k0 < g.K; k0 += 64) {
    float2 a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a[j] = an[j];
      b[j] = bn[j];
    }
    if (k0 + 64 < g.K) fetch(k0 + 64);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      zr = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].x, b[j].x, zr, 0, 0, 0);
      zi = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].x, b[j].y, zi, 0, 0, 0);
      zr = __builtin_amdgcn_mfma_f32_32x32x2f32(-a[j].y, b[j].y, zr, 0, 0, 0);
      zi = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j].y, b[j].x, zi, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r)
    red[(w * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * 33 + li] = make_float2(zr[r], zi[r]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (threadIdx.x >> 5) + 8 * i, c = threadIdx.x & 31;
    float2 z = red[r * 33 + c];
#pragma unroll
    for (int q = 1; q < 4; ++q) z = cadd(z, red[(q * 32 + r) * 33 + c]);
    float p = 0.0f;
    if (m0 + r < g.M && n0 + c < g.N) p = finish<W>(g, m0 + r, n0 + c, z);
    if constexpr (W != Product::kScaled) {
      p = last_lane_sum<32>(p);
      if (c == 31 && m0 + r < g.M) g.part[(m0 + r) * tiles + n0 / 32] = p;
    }
  }
}

// From 2^20 results on every SIMD has a 32 x 32 wave.  Loss and seed of the Gram form
// (K = N = 256, us, small / large): 1,024 rows 11.1 / 22, 2,048 18.9 / 23, 4,096
// 34 / 24.5, 8,192 60 / 44.5 (the one-wave 16 x 16 tiles and loss pass before: 1,024
// rows 18.0, 8,192 rows 80).
bool large(int64_t M, int N) { return M * N >= (int64_t(1) << 20); }

// From 2^18 results on a quarter of the CUs' waves is enough for 32 x 32 (seed alone, us,
// small / mid: K = N = 256, 512 rows 7.3 / 9.9, 1,024 11.1 / 10.4, 2,048 19.5 / 16.7, 3,000
// 25.7 / 22.7; K = N = 64, 12,000 rows 12.6 / 9.2; K = N = 16, 16,384 rows 6.9 / 7.9).  Not
// for K above 256: a wave takes a quarter of the k's in one sum, which would be longer
// than the 64 k that the other kernels add up in one.
bool mid(int64_t M, int N, int K) {
  return M * N >= (int64_t(1) << 18) && K >= 64 && K <= 256;
}

template <Product W>
hipError_t product_launch(const Operands& g, hipStream_t st) {
  const dim3 grid(unsigned(((g.M + 63) / 64) * ((g.N + 63) / 64)));
  if (large(g.M, g.N) && g.K > 64)
    hipLaunchKernelGGL((k_product_large<W, true>), grid, dim3(256), 0, st, g);
  else if (large(g.M, g.N))
    hipLaunchKernelGGL((k_product_large<W, false>), grid, dim3(256), 0, st, g);
  else if (mid(g.M, g.N, g.K))
    hipLaunchKernelGGL((k_product_mid<W>), dim3(unsigned(((g.M + 31) / 32) * ((g.N + 31) / 32))),
                       dim3(256), 0, st, g);
  else if (g.K > 512)
    hipLaunchKernelGGL((k_product_small<W, true>), dim3(unsigned(((g.M + 15) / 16) * ((g.N + 15) / 16))),
                       dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((k_product_small<W, false>), dim3(unsigned(((g.M + 15) / 16) * ((g.N + 15) / 16))),
                       dim3(256), 0, st, g);
  return hipGetLastError();
}

}  // namespace

int product_tile(int64_t M, int N, int K) { return large(M, N) || mid(M, N, K) ? 32 : 16; }

hipError_t launch_product(Product what, const float2* A, const float2* B, float2* C, int64_t M, int N,
                          int K, float scale, float* part, hipStream_t st) {
  const Operands g{A, B, C, part, M, N, K, scale};
  switch (what) {
    case Product::kGram: return product_launch<Product::kGram>(g, st);
    case Product::kOverlap: return product_launch<Product::kOverlap>(g, st);
    case Product::kScaled: return product_launch<Product::kScaled>(g, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace mbqc
