// Density matrices of column plans (2..7 live slots) as Pauli vectors, one
// simulation spread over several lanes (gfx950).
//
// A Hermitian 2^NS x 2^NS matrix is 4^NS real coefficients Tr(rho P) over the Pauli
// strings P, half the numbers of the matrix, and a step touches them much less:
// with (I, X, Y, Z) the coefficients on the measured qubit, the projection on
// XY angle theta after the CZ with the appended |+> (coherence damping gamma)
// leaves on the appended qubit
//   I' = I,  X' = Z,  Y' = gamma (s X - c Y),  Z' = gamma (c X + s Y)
// (c, s = cos, sin theta; the factor 1/2 of the projection dropped as everywhere):
// 4 multiply-adds per quartet of real numbers where the matrix form takes 20 per
// quartet of complex ones, and the trace never changes.  The CZ of the appended
// qubit n with its other neighbour q is a signed permutation: with a Pauli as bits
// (x, z), z_n ^= x_q, z_q ^= x_n, and a minus sign where x_n x_q (z_n ^ z_q).
//
// A string is a number of NS two-bit digits (x the upper bit), the next slot to
// measure first.  The first K digits are register bits (4^K coefficients per
// lane), the others the lane.  After M <= K steps the lanes exchange through LDS so
// that the M digits just measured become the last ones.  The CZ with a neighbour
// that is the lane's last digit (first step of a later phase) waits for that
// exchange, where it is a change of the address and the sign.
//
// Input and output pass through the matrix digit by digit, the same exchanges
// carrying complex numbers.
//
// Small batches are bound by the chain of exchanges (two LDS latencies each),
// larger ones by LDS bandwidth.
#include "grids.h"
#include "wide.h"

#include <algorithm>
#include <utility>

namespace mbqc {

namespace {

template <int NS, int K>
struct Pauli {
  static constexpr int LD = NS - K;                // digits of the lane
  static constexpr int TL = 1 << (2 * LD);         // lanes per simulation
  static constexpr int T = TL > 64 ? TL : 64;      // threads per workgroup
  static constexpr int G = T / TL;                 // simulations per workgroup
  static constexpr int N = 1 << (2 * K);           // coefficients per lane
  static constexpr int P = (NS + K - 1) / K;       // phases per block
  static constexpr int CS = (64 / NS) * NS;        // steps per coefficient chunk
  // exchange buffer of 4^NS complex numbers with 2 of padding every 16 (real
  // numbers: 4 every 32, in the same space)
  static constexpr int BUF = K == NS ? 0 : (1 << (2 * NS)) + (1 << (2 * NS)) / 8;
  static constexpr int SIM = BUF + CS + (CS & 1);  // float2 of LDS per simulation
  static constexpr int len(int p) { return NS / P + (p < NS % P ? 1 : 0); }
  static constexpr int first(int p) {
    int f = 0;
    for (int i = 0; i < p; ++i) f += len(i);
    return f;
  }
};

__device__ __forceinline__ int pad_real(int a) { return a + 4 * (a >> 5); }
__device__ __forceinline__ int pad_complex(int a) { return a + 2 * (a >> 4); }

// Place of register r of lane `lane` after a rotation by M digits.
template <int NS, int K, int M>
__device__ __forceinline__ int rotated(int r, int lane) {
  constexpr int LOW = 2 * (K - M);
  return ((r & ((1 << LOW) - 1)) << (2 * (NS - K + M))) | (lane << (2 * M)) | (r >> LOW);
}

// Steps FIRST + S on register digit S (and, for S > 0, the CZ with digit S - 1).
template <int K, int S>
__device__ __forceinline__ void pauli_step(float (&t)[1 << (2 * K)], float gc, float gs) {
  constexpr int N = 1 << (2 * K), SH = 2 * (K - 1 - S);
  float n[N];
#pragma unroll
  for (int b = 0; b < N; ++b) {
    if ((b >> SH) & 3) continue;
    const float pi = t[b], pz = t[b | (1 << SH)], px = t[b | (2 << SH)], py = t[b | (3 << SH)];
    const float v[4] = {pi, fmaf(gs, py, gc * px), pz, fmaf(-gc, py, gs * px)};   // I, Z, X, Y
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      int to = b | (d << SH);
      bool neg = false;
      if constexpr (S > 0) {
        const int x = d >> 1, z = d & 1, q = (b >> (SH + 2)) & 3, xq = q >> 1, zq = q & 1;
        to ^= (xq << SH) | (x << (SH + 2));
        neg = x && xq && (z ^ zq);
      }
      n[to] = neg ? -v[d] : v[d];
    }
  }
#pragma unroll
  for (int b = 0; b < N; ++b) t[b] = n[b];
}

// Rotation by M digits.  CZ: with the CZ between the phase's first digit and the
// lane's last one.
template <int NS, int K, int M, bool CZ>
__device__ __forceinline__ void pauli_rotate(float (&t)[1 << (2 * K)], float* buf, int lane) {
  using W = Pauli<NS, K>;
  if constexpr (K == NS) return;
  lanes_sync<W::TL>();
  constexpr int LOW = 2 * (K - M);                 // registers of one vector: digit M - 1
  const int xq = CZ ? (lane >> 1) & 1 : 0, zq = CZ ? lane & 1 : 0;
  // sign of the first digit's X (z = 0) and Y (z = 1) coefficients
  const uint32_t neg0 = uint32_t(xq & zq) << 31, neg1 = uint32_t(xq & ~zq) << 31;
#pragma unroll
  for (int r = 0; r < W::N; ++r) {
    if ((r >> LOW) & 3) continue;
    float v[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) v[d] = t[r | (d << LOW)];
    if constexpr (!CZ) {
      *reinterpret_cast<float4*>(buf + pad_real(rotated<NS, K, M>(r, lane))) =
          make_float4(v[0], v[1], v[2], v[3]);
    } else if constexpr (M == 1) {
      // the vector is the first digit: I, Z stay in this lane's place, X, Y go to
      // the lane with the other z; within each pair z changes where xq
      const float i0 = xq ? v[1] : v[0], i1 = xq ? v[0] : v[1];
      const float x = __uint_as_float(__float_as_uint(v[2]) ^ neg0);
      const float y = __uint_as_float(__float_as_uint(v[3]) ^ neg1);
      *reinterpret_cast<float2*>(buf + pad_real(rotated<NS, K, M>(r, lane))) = make_float2(i0, i1);
      *reinterpret_cast<float2*>(buf + pad_real(rotated<NS, K, M>(r, lane ^ 1)) + 2) =
          make_float2(xq ? y : x, xq ? x : y);
    } else {
      constexpr int ZB = 2 * (K - 1);              // z bit of the first digit
      const int z0 = (r >> ZB) & 1, x0 = (r >> (ZB + 1)) & 1;
      if (x0) {
        const uint32_t sg = z0 ? neg1 : neg0;
#pragma unroll
        for (int d = 0; d < 4; ++d) v[d] = __uint_as_float(__float_as_uint(v[d]) ^ sg);
      }
      // changing z0 moves the place by 4^(M-1), within one padding interval
      constexpr int D = 1 << (2 * (M - 1));
      static_assert(D <= 16, "padding interval");
      const int at = pad_real(rotated<NS, K, M>(r, x0 ? lane ^ 1 : lane)) + (z0 ? -xq : xq) * D;
      *reinterpret_cast<float4*>(buf + at) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
  lanes_sync<W::TL>();
#pragma unroll
  for (int r = 0; r < W::N; ++r) t[r] = buf[pad_real((r << (2 * W::LD)) | lane)];
}

template <int NS, int K, int M>
__device__ __forceinline__ void complex_rotate(float2 (&t)[1 << (2 * K)], float2* buf, int lane) {
  using W = Pauli<NS, K>;
  if constexpr (K == NS) return;
  lanes_sync<W::TL>();
  constexpr int LOW = 2 * (K - M);
#pragma unroll
  for (int r = 0; r < W::N; ++r) {
    if ((r >> LOW) & 1) continue;
    const float2 u = t[r], v = t[r | (1 << LOW)];
    *reinterpret_cast<float4*>(buf + pad_complex(rotated<NS, K, M>(r, lane))) =
        make_float4(u.x, u.y, v.x, v.y);
  }
  lanes_sync<W::TL>();
#pragma unroll
  for (int r = 0; r < W::N; ++r) t[r] = buf[pad_complex((r << (2 * W::LD)) | lane)];
}

// Digit S from matrix bits (row, column) to Pauli bits:
//   I = B00 + B11, Z = B00 - B11, X = B01 + B10, Y = i (B01 - B10).
template <int K, int S>
__device__ __forceinline__ void to_pauli(float2 (&t)[1 << (2 * K)]) {
  constexpr int SH = 2 * (K - 1 - S);
#pragma unroll
  for (int b = 0; b < (1 << (2 * K)); ++b) {
    if ((b >> SH) & 3) continue;
    const float2 b00 = t[b], b01 = t[b | (1 << SH)], b10 = t[b | (2 << SH)], b11 = t[b | (3 << SH)];
    t[b] = cadd(b00, b11);
    t[b | (1 << SH)] = csub(b00, b11);
    t[b | (2 << SH)] = cadd(b01, b10);
    const float2 d = csub(b01, b10);
    t[b | (3 << SH)] = make_float2(-d.y, d.x);
  }
}

// The way back (times 2) and the output channel on the qubit:
//   B00, B11 = I +- Z, B01, B10 = X -+ i Y.
template <int K, int S>
__device__ __forceinline__ void to_matrix(float2 (&t)[1 << (2 * K)], const DmNoise& nz) {
  constexpr int SH = 2 * (K - 1 - S);
#pragma unroll
  for (int b = 0; b < (1 << (2 * K)); ++b) {
    if ((b >> SH) & 3) continue;
    const float2 pi = t[b], pz = t[b | (1 << SH)], px = t[b | (2 << SH)], py = t[b | (3 << SH)];
    float2 b00 = cadd(pi, pz), b11 = csub(pi, pz);
    float2 b01 = make_float2(px.x + py.y, px.y - py.x), b10 = make_float2(px.x - py.y, px.y + py.x);
    if (nz.out_noise) {
      const float2 u = b00, v = b11;
      b00 = make_float2(fmaf(nz.d00, u.x, nz.d01 * v.x), fmaf(nz.d00, u.y, nz.d01 * v.y));
      b11 = make_float2(fmaf(nz.d10, u.x, nz.d11 * v.x), fmaf(nz.d10, u.y, nz.d11 * v.y));
      b01 = cscale(b01, nz.coh);
      b10 = cscale(b10, nz.coh);
    }
    t[b] = b00;
    t[b | (1 << SH)] = b01;
    t[b | (2 << SH)] = b10;
    t[b | (3 << SH)] = b11;
  }
}

template <int NS, int K, int P, int... SS>
__device__ __forceinline__ void in_phase(float2 (&t)[1 << (2 * K)], float2* buf, int lane,
                                         std::integer_sequence<int, SS...>) {
  (to_pauli<K, SS>(t), ...);
  complex_rotate<NS, K, Pauli<NS, K>::len(P)>(t, buf, lane);
}

template <int NS, int K, int P, int... SS>
__device__ __forceinline__ void step_phase(float (&t)[1 << (2 * K)], float* buf, const float2* bs,
                                           int lane, std::integer_sequence<int, SS...>) {
  using W = Pauli<NS, K>;
  (pauli_step<K, SS>(t, bs[W::first(P) + SS].x, -bs[W::first(P) + SS].y), ...);
  pauli_rotate<NS, K, W::len(P), (P > 0)>(t, buf, lane);
}

template <int NS, int K, int P, int... SS>
__device__ __forceinline__ void out_phase(float2 (&t)[1 << (2 * K)], float2* buf, int lane,
                                          const DmNoise& nz, std::integer_sequence<int, SS...>) {
  (to_matrix<K, SS>(t, nz), ...);
  complex_rotate<NS, K, Pauli<NS, K>::len(P)>(t, buf, lane);
}

// Row and column of the matrix entry with digits v (row bits the upper ones).
__device__ __forceinline__ int every_second_bit(int v) {
  v &= 0x5555;
  v = (v | (v >> 1)) & 0x3333;
  v = (v | (v >> 2)) & 0x0f0f;
  return (v | (v >> 4)) & 0x00ff;
}

template <int NS, int K, int... PS>
__device__ __forceinline__ void pauli_sim(const Job& J, int64_t g, bool active, const DmNoise& nz,
                                          int pad_slots, uint32_t flags, float2* buf, float2* bs,
                                          int lane, std::integer_sequence<int, PS...>) {
  using W = Pauli<NS, K>;
  const int64_t gg = active ? g : J.total - 1;
  int64_t bi, si;
  split_sim(J, gg, &bi, &si);
  const float* ang = J.angles + bi * J.angle_stride;
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  const int32_t* in_index = J.tab + J.off_in;
  const int32_t* sign = J.tab + J.off_sign;
  const int32_t* out_pos = J.tab + J.off_out;
  const float2* psi = J.psi + si * J.in_stride;
  const int n = J.n_steps;
  float t[W::N];
  {
    float2 m[W::N];
    float2 va[1 << K], vb[1 << K];
    const int la = every_second_bit(lane >> 1), lb = every_second_bit(lane);
#pragma unroll
    for (int i = 0; i < (1 << K); ++i) {
      const int a = (i << W::LD) | la, b = (i << W::LD) | lb;
      va[i] = flip(psi[in_index[a]], sign[a] ? 0x80000000u : 0u);
      vb[i] = flip(psi[in_index[b]], sign[b] ? 0x80000000u : 0u);
    }
#pragma unroll
    for (int r = 0; r < W::N; ++r)
      m[r] = cmul(va[every_second_bit(r >> 1)], cconj(vb[every_second_bit(r)]));
    (in_phase<NS, K, PS>(m, buf, lane, std::make_integer_sequence<int, W::len(PS)>{}), ...);
#pragma unroll
    for (int r = 0; r < W::N; ++r) t[r] = m[r].x;   // Hermitian: the coefficients are real
  }
  const float trace = t[0];   // of lane 0: the coefficient of I...I, constant from here on
  for (int kc = 0; kc < n; kc += W::CS) {
    lanes_sync<W::TL>();      // the previous chunk's reads are done
#pragma unroll 1
    for (int i = lane; i < W::CS; i += W::TL) {
      const int k = kc + i;
      if (k < n) bs[i] = cscale(exp_minus_i(step_angle(steps[k], ang, J.angle_stride_a)), nz.gamma);
    }
    lanes_sync<W::TL>();
    const int ke = kc + W::CS < n ? kc + W::CS : n;
    for (int k0 = kc; k0 < ke; k0 += NS)
      (step_phase<NS, K, PS>(t, reinterpret_cast<float*>(buf), bs + (k0 - kc), lane,
                             std::make_integer_sequence<int, W::len(PS)>{}),
       ...);
  }
  float2 m[W::N];
#pragma unroll
  for (int r = 0; r < W::N; ++r) m[r] = make_float2(t[r], 0.0f);
  (out_phase<NS, K, PS>(m, buf, lane, nz, std::make_integer_sequence<int, W::len(PS)>{}), ...);
  float scale = ldexpf(1.0f, -NS - pad_slots);
  if (flags & MBQC_FLAG_RENORMALIZE) {
    // lane 0's trace to all lanes
    float tr = trace;
    if constexpr (W::TL > 64) {
      if (lane == 0) bs[0].x = tr;
      __syncthreads();
      tr = bs[0].x;
    } else {
      tr = __shfl(tr, 0, W::TL);
    }
    scale = ldexpf(1.0f, -NS) / tr;
  }
  const int64_t d = int64_t(1) << J.n_out;
  float2* o = J.out + g * d * d;
  if constexpr (K == NS) {
    if (!active) return;
#pragma unroll
    for (int r = 0; r < W::N; ++r)
      o[int64_t(out_pos[every_second_bit(r >> 1)]) * d + out_pos[every_second_bit(r)]] =
          cscale(m[r], scale);
  } else {
    // rows of the matrix through LDS, so that stores are contiguous
    lanes_sync<W::TL>();
#pragma unroll
    for (int r = 0; r < W::N; ++r) {
      const int v = (r << (2 * W::LD)) | lane;
      buf[pad_complex((every_second_bit(v >> 1) << NS) | every_second_bit(v))] = m[r];
    }
    lanes_sync<W::TL>();
    if (!active) return;
#pragma unroll
    for (int r = 0; r < W::N; ++r) {
      const int e = r * W::TL + lane;
      o[int64_t(out_pos[e >> NS]) * d + out_pos[e & ((1 << NS) - 1)]] =
          cscale(buf[pad_complex(e)], scale);
    }
  }
}

template <int NS, int K>
__global__ __launch_bounds__((Pauli<NS, K>::T)) void k_dm_pauli(Job J, DmNoise nz, int pad_slots,
                                                               uint32_t flags) {
  using W = Pauli<NS, K>;
  __shared__ __align__(16) float2 lds[W::G * W::SIM];
  const int sub = threadIdx.x / W::TL, lane = threadIdx.x % W::TL;
  float2* buf = lds + sub * W::SIM;
  const int64_t g = int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  pauli_sim<NS, K>(J, g, g < J.total, nz, pad_slots, flags, buf, buf + W::BUF, lane,
                   std::make_integer_sequence<int, W::P>{});
}

// ------------------------------------------------------------ angle gradients
//
// The steps of a column plan are unitary up to their scale, so the gradient needs
// neither the states nor the cotangents of the steps in between, only
//   G = sum over columns of |out><seed|   (2^NS x 2^NS),
// taken backwards through the steps, G -> U^-1 G U: with outputs
// out_c = U_n ... U_1 in_c and dL = Re sum conj(seed) d(out) the derivative by the
// angle of step k is Im Tr(P1 G_k), P1 = (1 - Z) / 2 on the measured qubit and
// G_k before the step's butterfly.  The imaginary parts of Tr(G P) are 4^NS real
// numbers that evolve among themselves, so a step backwards is the transpose of a
// density matrix step: per parameter set 4^NS multiply-adds where the sweep of
// states and cotangents takes 9 C 2^NS for C columns, no checkpoints, and the
// derivative of a step is two coefficients, (I - Z) / 2.
//
// Bound by the digit exchanges through LDS (many sets: about half of the issue slots)
// or by the chain of steps and exchanges (few).  The transfer matrix's columns,
// against the sweeps with checkpoints: 4x20 grid, 16,384 sets 131 -> 54 us, 4x16
// grid, 1,024 sets 20.4 -> 11.7 us, 5x10 grid, 4,096 sets 101 -> 49 us.

// The inverse of pauli_rotate.
template <int NS, int K, int M, bool CZ>
__device__ __forceinline__ void pauli_unrotate(float (&t)[1 << (2 * K)], float* buf, int lane) {
  using W = Pauli<NS, K>;
  if constexpr (K == NS) return;
  lanes_sync<W::TL>();
#pragma unroll
  for (int r = 0; r < W::N; ++r) buf[pad_real((r << (2 * W::LD)) | lane)] = t[r];
  lanes_sync<W::TL>();
  constexpr int LOW = 2 * (K - M);
  const int xq = CZ ? (lane >> 1) & 1 : 0, zq = CZ ? lane & 1 : 0;
  const uint32_t neg0 = uint32_t(xq & zq) << 31, neg1 = uint32_t(xq & ~zq) << 31;
#pragma unroll
  for (int r = 0; r < W::N; ++r) {
    if ((r >> LOW) & 3) continue;
    float v[4];
    if constexpr (CZ && M == 1) {
      const float2 a = *reinterpret_cast<const float2*>(buf + pad_real(rotated<NS, K, M>(r, lane)));
      const float2 b =
          *reinterpret_cast<const float2*>(buf + pad_real(rotated<NS, K, M>(r, lane ^ 1)) + 2);
      v[0] = xq ? a.y : a.x;
      v[1] = xq ? a.x : a.y;
      v[2] = __uint_as_float(__float_as_uint(xq ? b.y : b.x) ^ neg0);
      v[3] = __uint_as_float(__float_as_uint(xq ? b.x : b.y) ^ neg1);
    } else {
      int at = pad_real(rotated<NS, K, M>(r, lane));
      uint32_t sg = 0;
      if constexpr (CZ) {
        constexpr int ZB = 2 * (K - 1), D = 1 << (2 * (M - 1));
        const int z0 = (r >> ZB) & 1, x0 = (r >> (ZB + 1)) & 1;
        if (x0) {
          at = pad_real(rotated<NS, K, M>(r, lane ^ 1));
          sg = z0 ? neg1 : neg0;
        }
        at += (z0 ? -xq : xq) * D;
      }
      const float4 u = *reinterpret_cast<const float4*>(buf + at);
      const float w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] = __uint_as_float(__float_as_uint(w[d]) ^ sg);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) t[r | (d << LOW)] = v[d];
  }
}

// The inverse of pauli_step (gamma = 1); returns the Z coefficient of the digit
// alone (lane 0's), which the phase before it leaves as it is.
template <int K, int S>
__device__ __forceinline__ float pauli_unstep(float (&t)[1 << (2 * K)], float c, float s) {
  constexpr int N = 1 << (2 * K), SH = 2 * (K - 1 - S);
  float n[N];
#pragma unroll
  for (int b = 0; b < N; ++b) {
    if ((b >> SH) & 3) continue;
    float v[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      int to = b | (d << SH);
      bool neg = false;
      if constexpr (S > 0) {
        const int x = d >> 1, z = d & 1, q = (b >> (SH + 2)) & 3, xq = q >> 1, zq = q & 1;
        to ^= (xq << SH) | (x << (SH + 2));
        neg = x && xq && (z ^ zq);
      }
      v[d] = neg ? -t[to] : t[to];
    }
    n[b] = v[0];
    n[b | (1 << SH)] = v[2];
    n[b | (2 << SH)] = fmaf(s, v[3], c * v[1]);
    n[b | (3 << SH)] = fmaf(-c, v[3], s * v[1]);
  }
#pragma unroll
  for (int b = 0; b < N; ++b) t[b] = n[b];
  return t[1 << SH];
}

template <int NS, int K, int P, int... SS>
__device__ __forceinline__ void unstep_phase(float (&t)[1 << (2 * K)], float* buf, const float2* bs,
                                             float (&z)[NS], int lane,
                                             std::integer_sequence<int, SS...>) {
  using W = Pauli<NS, K>;
  constexpr int F = W::first(P), M = W::len(P);
  pauli_unrotate<NS, K, M, (P > 0)>(t, buf, lane);
  ((z[F + M - 1 - SS] = pauli_unstep<K, M - 1 - SS>(t, bs[F + M - 1 - SS].x, -bs[F + M - 1 - SS].y)),
   ...);
}

// m += a conj(b)
__device__ __forceinline__ void cmul_conj_add(float2& m, float2 a, float2 b) {
  m.x = fmaf(a.x, b.x, fmaf(a.y, b.y, m.x));
  m.y = fmaf(a.y, b.x, fmaf(-a.x, b.y, m.y));
}

template <int NS, int K, int... PS>
__device__ __forceinline__ void pauli_gradient(const Job& J, const float2* out, const float2* seed,
                                               int64_t bi, bool active, int C, int n_angles, float* loss,
                                               float* grad, float2* buf, float2* bs, int lane,
                                               std::integer_sequence<int, PS...>) {
  using W = Pauli<NS, K>;
  const float* ang = J.angles + bi * J.angle_stride;
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  const Constant<int32_t> aidx = constant(J.tab + J.off_aidx);
  const int32_t* out_pos = J.tab + J.off_out;
  const int n = J.n_steps;
  float t[W::N];
  {
    float2 m[W::N];
    const int la = every_second_bit(lane >> 1), lb = every_second_bit(lane);
    const float2* pa[1 << K];
    const float2* pb[1 << K];
#pragma unroll
    for (int i = 0; i < (1 << K); ++i) {
      pa[i] = out + ((bi * C) << NS) + out_pos[(i << W::LD) | la];
      pb[i] = seed + ((bi * C) << NS) + out_pos[(i << W::LD) | lb];
    }
#pragma unroll
    for (int r = 0; r < W::N; ++r) m[r] = make_float2(0.0f, 0.0f);
#pragma unroll 8
    for (int c = 0; c < C; ++c) {
      float2 va[1 << K], vb[1 << K];
#pragma unroll
      for (int i = 0; i < (1 << K); ++i) {
        va[i] = pa[i][int64_t(c) << NS];
        vb[i] = pb[i][int64_t(c) << NS];
      }
#pragma unroll
      for (int r = 0; r < W::N; ++r)
        cmul_conj_add(m[r], va[every_second_bit(r >> 1)], vb[every_second_bit(r)]);
    }
    (in_phase<NS, K, PS>(m, buf, lane, std::make_integer_sequence<int, W::len(PS)>{}), ...);
#pragma unroll
    for (int r = 0; r < W::N; ++r) t[r] = m[r].y;
    if (loss && active && lane == 0) loss[bi] = fmaf(0.5f, m[0].x, 1.0f);
  }
  const float all = t[0];     // of lane 0: the coefficient of I...I, constant from here on
  const bool writer = active && lane == 0;
  float* gp = grad + bi * n_angles;
  for (int kc = ((n - 1) / W::CS) * W::CS; kc >= 0; kc -= W::CS) {
    lanes_sync<W::TL>();      // the previous chunk's reads are done
#pragma unroll 1
    for (int i = lane; i < W::CS; i += W::TL) {
      const int k = kc + i;
      if (k < n) bs[i] = exp_minus_i(step_angle(steps[k], ang, J.angle_stride_a));
    }
    lanes_sync<W::TL>();
    const int ke = kc + W::CS < n ? kc + W::CS : n;
    for (int k0 = ke - NS; k0 >= kc; k0 -= NS) {
      float2 b[NS];
      float z[NS];
      int ai[NS];
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        b[k] = bs[k0 - kc + k];
        ai[k] = aidx[k0 + k];
      }
      (unstep_phase<NS, K, W::P - 1 - PS>(t, reinterpret_cast<float*>(buf), b, z, lane,
                                          std::make_integer_sequence<int, W::len(W::P - 1 - PS)>{}),
       ...);
      if (writer) {
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (ai[k] >= 0) gp[ai[k]] = 0.5f * (all - z[k]);
      }
    }
  }
}

template <int NS, int K>
__global__ __launch_bounds__((Pauli<NS, K>::T)) void k_pauli_gradient(
    Job J, const float2* __restrict__ out, const float2* __restrict__ seed, int64_t B, int C,
    int n_angles, float* __restrict__ loss, float* __restrict__ grad) {
  using W = Pauli<NS, K>;
  __shared__ __align__(16) float2 lds[W::G * W::SIM];
  const int sub = threadIdx.x / W::TL, lane = threadIdx.x % W::TL;
  float2* buf = lds + sub * W::SIM;
  const int64_t g = int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  const bool active = g < B;
  pauli_gradient<NS, K>(J, out, seed, active ? g : B - 1, active, C, n_angles, loss, grad, buf,
                        buf + W::BUF, lane, std::make_integer_sequence<int, W::P>{});
}

// Register digits K: one keeps many lanes on a simulation and the chain of a step
// short, two halve the exchanges.  Measured (us per replayed launch, the matrix
// kernels before / K = 1 / K = 2): 3 slots (12 columns) 1,024 sims 10.2 / 6.7 /
// 13.2, 4,096 12.7 / 8.0 / 13.5, 1M 727 / 509 / 661; 4 slots (10) 1,024 13.0 / 7.8 /
// 10.6, 4,096 25.6 / 15.2 / 14.8, 16,384 82.5 / 45.8 / 35.1; 5 slots (8) 1,024
// 25.4 / 17.5 / 16.3, 16,384 273 / 162 / 106; 6 slots (8) 1,024 95.6 / 36.0 / 35.9;
// 7 slots (8) 256 212 / 47.6 / 47.5.  Three digits are slower from 3 slots on (30 us
// for 4,096 sims of 3: registers and too few waves).
constexpr int64_t kDm4OneDigitMaxSims = 2048;

template <int NS, int K>
hipError_t dm_launch(const Job& J, const DmNoise& nz, int pad_slots, uint32_t flags,
                     hipStream_t st) {
  using W = Pauli<NS, K>;
  return in_parts(J.total / J.S, J.S, max_grid(W::T) * W::G, hipSuccess,
                  [&](int64_t b, int64_t sets, int64_t s, int64_t inputs) {
    Job part = J;
    part.angles = J.angles + b * J.angle_stride;
    part.psi = J.psi + s * J.in_stride;
    part.out = J.out + ((b * J.S + s) << (2 * J.n_out));
    part.S = inputs;
    part.total = sets * inputs;
    hipLaunchKernelGGL((k_dm_pauli<NS, K>), dim3(unsigned((part.total + W::G - 1) / W::G)), dim3(W::T),
                       0, st, part, nz, pad_slots, flags);
    return hipGetLastError();
  });
}

template <int NS, int K>
hipError_t gradient_launch(const Job& J, const float2* out, const float2* seed, int64_t B, int64_t C,
                           int n_angles, float* loss, float* grad, hipStream_t st) {
  using W = Pauli<NS, K>;
  return in_grids((B + W::G - 1) / W::G, W::T, hipSuccess, [&](int64_t first, int64_t count) {
    const int64_t b = first * W::G, rows = (b * C) << NS;
    Job part = J;
    part.angles = J.angles + b * J.angle_stride;
    hipLaunchKernelGGL((k_pauli_gradient<NS, K>), dim3(unsigned(count)), dim3(W::T), 0, st, part,
                       out + rows, seed + rows, std::min(B - b, count * W::G), int(C), n_angles,
                       loss ? loss + b : nullptr, grad + b * n_angles);
    return hipGetLastError();
  });
}

}  // namespace

// Register digits, us per replayed launch with the transfer matrix's columns, K = 1 /
// K = 2: 2x12 grid, 16,384 sets 8.6 / 12.9; 3x12 grid, 16 sets 7.3 / 12.4, 16,384
// 14.6 / 18.3; 4x16 grid, 1,024 sets 12.0 / 14.9, 4,096 22.4 / 18.1; 5x10 grid,
// 1,024 sets 29.0 / 19.9.
hipError_t launch_pauli_gradient(const Job& J, const float2* out, const float2* seed, int64_t B,
                                 int64_t C, int n_angles, float* loss, float* grad,
                                 hipStream_t st) {
  switch (J.ns) {
    case 2: return gradient_launch<2, 1>(J, out, seed, B, C, n_angles, loss, grad, st);
    case 3: return gradient_launch<3, 1>(J, out, seed, B, C, n_angles, loss, grad, st);
    case 4:
      return B <= kDm4OneDigitMaxSims
                 ? gradient_launch<4, 1>(J, out, seed, B, C, n_angles, loss, grad, st)
                 : gradient_launch<4, 2>(J, out, seed, B, C, n_angles, loss, grad, st);
    case 5: return gradient_launch<5, 2>(J, out, seed, B, C, n_angles, loss, grad, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_dm_pauli(const Job& J, const DmNoise& nz, int pad_slots, uint32_t flags,
                           hipStream_t st) {
  switch (J.ns) {
    case 2: return dm_launch<2, 1>(J, nz, pad_slots, flags, st);
    case 3: return dm_launch<3, 1>(J, nz, pad_slots, flags, st);
    case 4:
      return J.total <= kDm4OneDigitMaxSims ? dm_launch<4, 1>(J, nz, pad_slots, flags, st)
                                            : dm_launch<4, 2>(J, nz, pad_slots, flags, st);
    case 5: return dm_launch<5, 2>(J, nz, pad_slots, flags, st);
    case 6: return dm_launch<6, 2>(J, nz, pad_slots, flags, st);
    case 7: return dm_launch<7, 2>(J, nz, pad_slots, flags, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mbqc
