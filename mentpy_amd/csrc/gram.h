// Launchers of the complex matrix products of the MB-QML losses (gram.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace mbqc {

// What is done with z = A B (row-major complex, A [M][K], B [K][N]); loss partials
// part[row][tile] for tiles of product_tile(M, N, K) columns.
enum class Product {
  kGram,      // C = scale z, part = sum Re(conj(A) z)  (K = N)
  kOverlap,   // C = z (no store if null), part = sum |z|^2
  kScaled,    // C = scale z
};

int product_tile(int64_t M, int N, int K);

hipError_t launch_product(Product what, const float2* A, const float2* B, float2* C, int64_t M, int N,
                          int K, float scale, float* part, hipStream_t st);

}  // namespace mbqc
