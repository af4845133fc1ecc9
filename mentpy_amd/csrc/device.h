// Device code shared by the kernel sources: complex arithmetic, sine and cosine,
// the reference's global phase, the job description, the sampled-outcome draws
// and small workgroup helpers.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "plan.h"

namespace mbqc {

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// flip the sign of both components when sbit == 0x80000000
__device__ __forceinline__ float2 flip(float2 v, uint32_t sbit) {
  return make_float2(__uint_as_float(__float_as_uint(v.x) ^ sbit),
                     __uint_as_float(__float_as_uint(v.y) ^ sbit));
}
// CZ sign of slot-index j against the neighbour mask: parity(j & mask) << 31
__device__ __forceinline__ uint32_t czbit(uint32_t j, uint32_t mask) {
  return uint32_t(__builtin_popcount(j & mask) & 1) << 31;
}

// Round-to-nearest-even integer of v (|v| < 2^22) by the 1.5 * 2^23 shifter:
// fl(v + 1.5 * 2^23) has a unit last mantissa bit, so its lowest bit is the
// parity of rint(v).  With the shifter added in an FMA, v = a * c is rounded
// once (no rounding of a * c first).
constexpr float kShifter = 12582912.0f;      // 1.5 * 2^23

// sin and cos of x for |x| up to a few thousand: x = k pi + r with a two-term
// Cody-Waite split of pi (hi part the nearest float), |r| <= pi/2, then
// polynomials fitted for minimum maximum error on [-pi/2, pi/2] (odd degree 9
// for sin, even degree 10 for cos; fitted in double by linear programming on
// 4,000 Chebyshev points, approximation error below 5e-10, float evaluation
// error about 1e-7), and the sign (-1)^k on both.
__device__ __forceinline__ void sincos_poly(float x, float* sn, float* cs) {
  const float kb = fmaf(x, 0.318309886183790671538f, kShifter);
  const float k = kb - kShifter;
  float r = fmaf(-k, 3.14159274101257324219f, x);
  r = fmaf(-k, -8.74227800037248e-8f, r);
  const float r2 = r * r;
  float ps = fmaf(r2, 2.601407004e-6f, -1.980598900e-4f);
  ps = fmaf(r2, ps, 8.332983591e-3f);
  ps = fmaf(r2, ps, -1.666665375e-1f);
  const float sr = fmaf(r * r2, ps, r);
  float pc = fmaf(r2, -2.650938882e-7f, 2.479057366e-5f);
  pc = fmaf(r2, pc, -1.388906501e-3f);
  pc = fmaf(r2, pc, 4.166670144e-2f);
  pc = fmaf(r2, pc, -0.5f);
  const float cr = fmaf(r2, pc, 1.0f);
  const uint32_t sgn = __float_as_uint(kb) << 31;
  *sn = __uint_as_float(__float_as_uint(sr) ^ sgn);
  *cs = __uint_as_float(__float_as_uint(cr) ^ sgn);
}

// (cos a, sin a) rounded from double arithmetic, |a| up to a few thousand:
// a = k pi/2 + r, |r| <= pi/4, Taylor series to r^13 and r^14 (remainders below
// 3e-14, so the floats are the nearest ones but for very rare near-ties).
__device__ __forceinline__ float2 cis_f64(double a) {
  const double k = rint(a * 0.63661977236758134308);
  double r = fma(-k, 1.57079632679489661923, a);
  r = fma(-k, 6.12323399573676603587e-17, r);
  const double r2 = r * r;
  double ps = fma(r2, 1.0 / 6227020800.0, -1.0 / 39916800.0);
  ps = fma(r2, ps, 1.0 / 362880.0);
  ps = fma(r2, ps, -1.0 / 5040.0);
  ps = fma(r2, ps, 1.0 / 120.0);
  ps = fma(r2, ps, -1.0 / 6.0);
  const float s = float(fma(r * r2, ps, r));
  double pc = fma(r2, -1.0 / 87178291200.0, 1.0 / 479001600.0);
  pc = fma(r2, pc, -1.0 / 3628800.0);
  pc = fma(r2, pc, 1.0 / 40320.0);
  pc = fma(r2, pc, -1.0 / 720.0);
  pc = fma(r2, pc, 1.0 / 24.0);
  pc = fma(r2, pc, -0.5);
  const float c = float(fma(r2, pc, 1.0));
  const int q = int(k) & 3;
  const float cs = (q & 1) ? s : c, sn = (q & 1) ? c : s;
  return make_float2(((q + 1) & 2) ? -cs : cs, (q & 2) ? -sn : sn);
}

// e^{-i x} for kernels that evaluate a step's coefficient once per simulation,
// where double arithmetic costs nothing next to the amplitudes.  (The float
// polynomials above leave about 1e-7 in every coefficient, an error that all
// amplitudes share and that adds up over the steps.)
__device__ __forceinline__ float2 exp_minus_i(float x) { return cis_f64(-double(x)); }

// The reference's global phase, prod_k sgn(cos(theta_k/2)) e^{i theta_k/2}
// (the factor its amplitude-sum partial trace introduces,
// mentpy/calculator/state_ops.py:68-73).  With m_k = rint(theta_k / 2 pi),
// theta_k/2 - pi m_k lies in [-pi/2, pi/2], so sgn(cos(theta_k/2)) = (-1)^m_k
// and the product is exp(i (sum_k theta_k / 2 - pi sum_k m_k)).  The angles
// are summed in double (full-rate on this GPU) and the integers m_k in int32,
// and the phase is formed once at the end.
// m_k must be exact for every float32 angle, also the ones next to an odd
// multiple of pi where cos(theta/2) changes sign (float32(pi) itself lies
// 8.7e-8 above pi: m = 1, phase -i).  A float32 product with fl32(1/2pi),
// 4e-8 too small relative to 1/2pi, rounds those down, so m_k is rounded in
// double: fma(theta, fl64(1/2pi), 1.5 * 2^52) rounds the exact product to an
// integer (ties to even) held in the low word of its bits, with a relative
// error of 1.1e-16 that can only matter within 1e-13 of a half-integer;
// no float32 angle below 2^12 comes that close (the nearest lies more than
// 1e-9 away, checked exhaustively on the CPU).
constexpr double kShifter64 = 6755399441055744.0;   // 1.5 * 2^52
struct RefPhase {
  double th_sum = 0.0;
  int32_t m_sum = 0;
  __device__ __forceinline__ void add(float th) {
    const double d = double(th);
    const double mb = fma(d, 0.15915494309189533577, kShifter64);
    m_sum += int32_t(uint32_t(__double_as_longlong(mb)));
    th_sum += d;
  }
  // add(th) where `on`, nothing elsewhere
  __device__ __forceinline__ void add_if(float th, bool on) {
    const double d = on ? double(th) : 0.0;
    const double mb = fma(d, 0.15915494309189533577, kShifter64);
    m_sum += int32_t(uint32_t(__double_as_longlong(mb)));
    th_sum += d;
  }
  __device__ __forceinline__ float2 value() const {
    // at most pi/2 per step: small enough for cis_f64's reduction
    return cis_f64(fma(-3.14159265358979323846, double(m_sum), 0.5 * th_sum));
  }
};

// b = e^{-i theta}; with REF the step's reference phase is accumulated too.
template <bool REF>
__device__ __forceinline__ float2 step_coeff(float th, RefPhase* ph) {
  if constexpr (REF) ph->add(th);
  float s, c;
  sincos_poly(th, &s, &c);
  return make_float2(c, -s);
}

// Job description shared by the SV / DM / adjoint kernels (passed by value
// or read from global memory by the persistent kernel).
struct Job {
  const int32_t* tab;       // packed device tables of the plan
  int32_t off_in, off_sign, off_out, off_svres, off_dmres, e_sv, e_dm;
  int32_t ns, n_steps, n_out, live_mask, off_coef;
  int32_t off_aidx, off_run;  // contiguous angle indices, stretch ends
  // 1: no step has a fixed angle and every angle offset angle_index *
  // angle_stride_a fits in 32 bits (the statevector kernels' short fetch)
  int32_t fast_fetch;
  const float* angles;
  int64_t angle_stride;     // elements between angle vectors (0: shared)
  int64_t angle_stride_a;   // elements between the angles of one vector
  const float2* psi;
  int64_t in_stride;
  float2* out;
  float2* phase_out;
  int64_t S, total;
};

// Plan tables as constant memory, for loads at uniform addresses: they become
// scalar loads, also in kernels whose memory fences (the lanes' LDS exchanges)
// keep the compiler from proving that nothing writes the tables.  A per-lane load
// in their place costs every wave its full latency.
template <typename T>
using Constant = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ Constant<T> constant(const T* p) {
  return (Constant<T>)p;
}

// Angle vector and input of simulation g: g / S and g % S, in 32 bits where the
// batch allows it (a 64-bit division is over a hundred instructions).
__device__ __forceinline__ void split_sim(const Job& J, int64_t g, int64_t* bi, int64_t* si) {
  if (J.S == 1) {
    *bi = g;
    *si = 0;
  } else if (J.total <= 0xffffffffll) {
    const uint32_t q = uint32_t(g) / uint32_t(J.S);
    *bi = q;
    *si = uint32_t(g) - q * uint32_t(J.S);
  } else {
    *bi = g / J.S;
    *si = g - *bi * J.S;
  }
}

// Single-qubit noise of the density-matrix path.  Every supported channel is
// phase covariant: on a qubit's 2x2 blocks it maps the diagonal pair
// (r00, r11) -> (d00 r00 + d01 r11, d10 r00 + d11 r11) and scales both
// off-diagonal blocks by the real factor coh.  A measured qubit only shows
// the trace (preserved) and coh to its XY projection, so its noise (and the
// readout flip) folds into gamma = coh (1 - 2 p_readout); output qubits get the
// full map at the end.
struct DmNoise {
  float gamma;
  float d00, d01, d10, d11, coh;
  int32_t out_noise;  // 0: the output map is the identity
  float flip;         // 1 - 2 p_readout
};

// Identity modifier of the per-step projection coefficient b = e^{-i theta}.
struct NoModify {
  __device__ __forceinline__ float2 operator()(int, float2 b) const { return b; }
};

__device__ __forceinline__ float sv_final_scale(int e) {
  float s = ldexpf(1.0f, -(e >> 1));
  return (e & 1) ? s * 0.70710678118654752440f : s;
}

// 32 pseudo-random bits per (seed, simulation, block of 32 steps): the
// splitmix64 finaliser (Steele, Lea, Flood, "Fast splittable pseudorandom
// number generators", OOPSLA 2014) applied to a Weyl-sequence key.
__device__ __forceinline__ uint32_t draw32(uint64_t seed, uint64_t sim, uint64_t block) {
  uint64_t z = seed + sim * 0x9E3779B97F4A7C15ull + (block + 1) * 0xD1B54A32D192ED03ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return uint32_t(z ^ (z >> 31));
}

// Per-lane Pauli frame and outcome draw of the sampled mode.  Before step k,
// bit 0 of fx / fz is the X / Z frame of schedule[k]: the node is measured at
// (-1)^x theta, the drawn projection m' (probability 1/2 each) is onto
// |+/- theta'>, and the physical outcome is m' xor z.  An outcome 1 flips the
// frames of the flow successor and of its later neighbours (xmask/zmask).
// Frames are 32-bit: a plan that samples has every offset below 32 (the plan
// compiler checks it).
struct SampleMod {
  uint32_t fx = 0, fz = 0;
  uint64_t seed = 0, sim = 0;
  Constant<uint64_t> xm;
  Constant<uint64_t> zm;
  int32_t* out_words;   // this simulation's outcome words (null for inactive lanes)
  int n;
  uint32_t rbits = 0, word = 0;
  __device__ __forceinline__ float2 operator()(int k, float2 b) {
    const int kb = k & 31;
    if (kb == 0) rbits = draw32(seed, sim, uint64_t(k >> 5));
    const uint32_t mprime = (rbits >> kb) & 1u;
    const uint32_t xk = fx & 1u, zk = fz & 1u;
    const uint32_t mk = mprime ^ zk;
    word |= mk << kb;
    if (kb == 31 || k == n - 1) {
      if (out_words) out_words[k >> 5] = int32_t(word);
      word = 0;
    }
    const uint32_t sel = 0u - mk;
    fx = (fx ^ (uint32_t(xm[k]) & sel)) >> 1;
    fz = (fz ^ (uint32_t(zm[k]) & sel)) >> 1;
    float2 bb = xk ? cconj(b) : b;
    return mprime ? make_float2(-bb.x, -bb.y) : bb;
  }
};

// Workgroups are dealt to the chip's kXcds XCDs round-robin (workgroup b runs
// on XCD b % kXcds), each XCD with its own L2.  xcd_block maps workgroup b of
// n to a logical block so that every XCD takes a contiguous run of logical
// blocks (a bijection of [0, n)): neighbouring simulations, which share cache
// lines of the angle table, then meet in one L2 instead of each XCD fetching
// the line.
constexpr unsigned kXcds = 8;
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned n) {
  const unsigned q = n / kXcds, r = n % kXcds, x = b % kXcds;
  return x * q + (x < r ? x : r) + b / kXcds;
}

__device__ __forceinline__ int insert_zero(int v, int q) {
  return ((v >> q) << (q + 1)) | (v & ((1 << q) - 1));
}

// Sum over the T threads of a workgroup (T a power of two); a workgroup of
// fewer than 64 threads only exchanges among its own lanes.
template <int T>
__device__ __forceinline__ float block_sum(float v, float* red) {
  constexpr int first = T >= 64 ? 32 : T / 2;
  for (int m = first; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  if constexpr (T > 64) {
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    v = 0.0f;
#pragma unroll
    for (int i = 0; i < T / 64; ++i) v += red[i];
  }
  return v;
}

// Makes the LDS writes of a simulation's lanes visible to all of them: a
// barrier where it spans several waves, else only an order within the wave.
template <int T>
__device__ __forceinline__ void lanes_sync() {
  if constexpr (T > 64) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// Sum over L neighbouring lanes; `red`: LDS of L / 64 values, used where they
// span several waves (then the whole workgroup).
template <int L, typename V>
__device__ __forceinline__ V lanes_sum(V v, V* red) {
#pragma unroll
  for (int m = (L < 64 ? L : 64) / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  if constexpr (L > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < L / 64; ++i) v += red[i];
  }
  return v;
}

// The angle of step k of this simulation (its angle-vector entry or its fixed angle).
__device__ __forceinline__ float step_angle(const mbqc_step& st, const float* ang, int64_t sa) {
  return st.angle_index >= 0 ? ang[int64_t(st.angle_index) * sa] : st.fixed_angle;
}

// Work item of the batched kernels.
struct BatchItem {
  int32_t job;
  int32_t count;   // simulations in this item
  int64_t first;   // first simulation index within the job
};

// A Job read from device memory (rather than passed as a kernel argument)
// holds generic pointers: loads and stores through them compile to flat
// instructions, and the plan-table loads could not be proven free of the
// kernel's own stores, so they would all be per-lane vector loads.  The same
// layout with the pointers typed as global memory, and the read-only plan
// tables as constant memory, restores global vector instructions and scalar
// table loads.
struct GlobalJob {
  const __attribute__((address_space(4))) int32_t* tab;
  int32_t off_in, off_sign, off_out, off_svres, off_dmres, e_sv, e_dm;
  int32_t ns, n_steps, n_out, live_mask, off_coef;
  int32_t off_aidx, off_run;
  int32_t fast_fetch;
  const __attribute__((address_space(1))) float* angles;
  int64_t angle_stride;
  int64_t angle_stride_a;
  const __attribute__((address_space(1))) float2* psi;
  int64_t in_stride;
  __attribute__((address_space(1))) float2* out;
  __attribute__((address_space(1))) float2* phase_out;
  int64_t S, total;
};
static_assert(sizeof(GlobalJob) == sizeof(Job), "GlobalJob mirrors Job");

__device__ __forceinline__ Job load_job(const Job* jobs, int i) {
  const GlobalJob g = reinterpret_cast<const GlobalJob*>(jobs)[i];
  Job j;
  j.tab = (const int32_t*)g.tab;
  j.off_in = g.off_in;
  j.off_sign = g.off_sign;
  j.off_out = g.off_out;
  j.off_svres = g.off_svres;
  j.off_dmres = g.off_dmres;
  j.e_sv = g.e_sv;
  j.e_dm = g.e_dm;
  j.ns = g.ns;
  j.n_steps = g.n_steps;
  j.n_out = g.n_out;
  j.live_mask = g.live_mask;
  j.off_coef = g.off_coef;
  j.off_aidx = g.off_aidx;
  j.off_run = g.off_run;
  j.fast_fetch = g.fast_fetch;
  j.angles = (const float*)g.angles;
  j.angle_stride = g.angle_stride;
  j.angle_stride_a = g.angle_stride_a;
  j.psi = (const float2*)g.psi;
  j.in_stride = g.in_stride;
  j.out = (float2*)g.out;
  j.phase_out = (float2*)g.phase_out;
  j.S = g.S;
  j.total = g.total;
  return j;
}

// group counters live kCounterStride ints apart (separate cache lines)
constexpr int kCounterStride = 64;

// Sum over the TL lanes of a group, in its last lane at least.
template <int CTRL, int ROWS>
__device__ __forceinline__ float add_dpp(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}
template <int TL>
__device__ __forceinline__ float last_lane_sum(float v) {
  if constexpr (TL > 1) v = add_dpp<0xB1, 0xf>(v);     // quad_perm [1,0,3,2]
  if constexpr (TL > 2) v = add_dpp<0x4E, 0xf>(v);     // quad_perm [2,3,0,1]
  if constexpr (TL > 4) v = add_dpp<0x141, 0xf>(v);    // row_half_mirror
  if constexpr (TL > 8) v = add_dpp<0x140, 0xf>(v);    // row_mirror
  if constexpr (TL > 16) v = add_dpp<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  if constexpr (TL > 32) v = add_dpp<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
  return v;
}

}  // namespace mbqc
