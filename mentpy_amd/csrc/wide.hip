// Statevector kernels that spread one simulation over several lanes (gfx950):
// live windows of 7 slots and more, and small batches of narrower ones.
//
// The state of one simulation is spread over TL = 2^(NS - R) lanes with 2^R
// amplitudes each in registers: amplitude v = r * TL + lane, r the register.
// A block of NS steps measures the slots from the most significant to the
// least, so the first steps of a block pair amplitudes of one lane: they are
// register-only butterflies.  After M <= R of them the lanes exchange through
// LDS so that the M slots just measured become the least significant bits
// (v -> rotate-left(v, M)) and the next slots to measure are register bits
// again.  A block is ceil(NS / R) such phases; after it the rotation is back
// at slot order.  The LDS then carries every amplitude once per phase instead
// of once per step, and a barrier (only where a simulation spans more than
// one wave) stands between phases, not between steps.
//
// Sine, cosine and the reference phase are evaluated once per step, one step
// per lane, for a chunk of whole blocks at a time, and read back as LDS
// broadcasts.
//
// Bound by LDS bandwidth and VALU issue about equally: a block of the 9-slot
// loop is 232 VALU and 41 LDS instructions per wave.  9x10 grid, 4,099
// simulations: 103.6 us with one LDS pass and one barrier per step, 28.4 us so.
#include "grids.h"
#include "wide.h"

#include <algorithm>
#include <utility>

namespace mbqc {

namespace {

// Register bits R by window size.  More of them mean fewer exchanges, fewer
// mean more lanes per simulation and more waves in flight.  Measured (us per
// call of 4,096 simulations of a 10-column grid, R = 2 / 3 / 4 / 5): 9 slots
// 43 / 31 / 33 / 40, 10 slots 79 / 62 / 53 / 54, 11 slots (6 columns) 112 / 75 /
// 63 / 74; from 12 slots on 4 is at least as good as 5.
constexpr int wide_reg_bits(int ns) { return ns <= 9 ? 3 : 4; }

// NS amplitude bits over lanes and registers, M of them measured per block
// (all of them except in a pass over tiles of a larger state).  SPARE: log2 of
// the lanes per amplitude lane; the spare ones share the coefficient work and
// repeat the state's.
template <int NS, int R, int M = NS, int SPARE = 0>
struct Wide {
  static constexpr int TL = 1 << (NS - R);        // lanes per simulation
  static constexpr int CL = TL << SPARE;          // lanes that evaluate its coefficients
  static constexpr int T = CL > 64 ? CL : 64;     // threads per workgroup
  static constexpr int G = T / CL;                // simulations per workgroup
  static constexpr int NR = 1 << R;               // amplitudes per lane
  static constexpr int P = (M + R - 1) / R;       // phases per block
  static constexpr int CS = M == NS ? (64 / NS) * NS : M;   // steps per coefficient chunk
  static constexpr int BUF = (1 << NS) + (1 << NS) / 16;   // padded exchange buffer
  static constexpr int SIM = BUF + CS;            // float2 of LDS per simulation
  static constexpr int len(int p) { return M / P + (p < M % P ? 1 : 0); }
  static constexpr int first(int p) {
    int f = 0;
    for (int i = 0; i < p; ++i) f += len(i);
    return f;
  }
};

__device__ __forceinline__ int padded(int a) { return a + (a >> 4); }

// CZ neighbours of the qubit appended by a step, as a mask over the amplitude
// bits at the block's start, and the sign (bit 31) that amplitude bits outside
// the workgroup's tile contribute.
struct StepSigns {
  uint32_t mask, outer;
};
struct SlotSigns {
  __device__ __forceinline__ StepSigns operator()(const mbqc_step& st) const { return {st.nmask, 0u}; }
};

// Step FIRST + S of a block on its phase's register bit R - 1 - S.
template <int NS, int R, int FIRST, int S, bool COLUMN, typename Signs>
__device__ __forceinline__ void wide_step(float2 (&t)[1 << R], float2 b, const mbqc_step* steps,
                                          int k, int lane, bool top, const Signs& signs) {
  constexpr int NR = 1 << R, QB = 1 << (R - 1 - S);
  constexpr int TL = 1 << (NS - R);
  if constexpr (COLUMN) {
    // the appended qubit's other neighbour is the one appended a step
    // earlier: no one at the column's first step (`top`), lane bit 0 at the
    // first step of a later phase, else the register bit above the measured one
    const float sg = (S == 0 && !top && (lane & 1)) ? -1.0f : 1.0f;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (r & QB) continue;
      const float2 x = t[r], y = t[r | QB];
      float2 u0;
      u0.x = fmaf(-b.y, y.y, fmaf(b.x, y.x, x.x));
      u0.y = fmaf(b.x, y.y, fmaf(b.y, y.x, x.y));
      t[r] = u0;
      if constexpr (S == 0) {
        const float be = 2.0f * sg;
        t[r | QB] = make_float2(fmaf(be, x.x, -sg * u0.x), fmaf(be, x.y, -sg * u0.y));
      } else if (r & (QB << 1)) {
        t[r | QB] = make_float2(fmaf(-2.0f, x.x, u0.x), fmaf(-2.0f, x.y, u0.y));
      } else {
        t[r | QB] = make_float2(fmaf(2.0f, x.x, -u0.x), fmaf(2.0f, x.y, -u0.y));
      }
    }
  } else {
    const Constant<uint32_t> row = constant(reinterpret_cast<const uint32_t*>(steps + k));
    mbqc_step st{};
    st.flags = row[1];
    st.nmask = row[2];
    const float s = (st.flags & 2u) ? -1.0f : 1.0f;
    const float app = (st.flags & 1u) ? 1.0f : 0.0f;
    // the neighbour mask in the phase's amplitude order (rotated by FIRST)
    const StepSigns z = signs(st);
    const uint32_t m = ((z.mask << FIRST) | (z.mask >> (NS - FIRST))) & ((1u << NS) - 1);
    const uint32_t lane_sign = czbit(uint32_t(lane), m & uint32_t(TL - 1)) ^ z.outer;
    const uint32_t mr = m >> (NS - R);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (r & QB) continue;
      const float c = __uint_as_float(__float_as_uint(app) ^ lane_sign ^ czbit(uint32_t(r), mr));
      const float al = c * s, be = c * (1.0f - s);
      const float2 x = t[r], y = t[r | QB];
      float2 u0;
      u0.x = fmaf(-b.y, y.y, fmaf(b.x, y.x, x.x));
      u0.y = fmaf(b.x, y.y, fmaf(b.y, y.x, x.y));
      t[r] = u0;
      t[r | QB] = make_float2(fmaf(al, u0.x, be * x.x), fmaf(al, u0.y, be * x.y));
    }
  }
}

// v -> rotate-left(v, M): the top M bits of v (register bits) become the lowest.
template <int NS, int R, int M, int T>
__device__ __forceinline__ void wide_rotate(float2 (&t)[1 << R], float2* buf, int lane) {
  constexpr int NR = 1 << R;
  lanes_sync<T>();   // earlier reads of the buffer are done
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int top = r >> (R - M), low = r & ((1 << (R - M)) - 1);
    buf[padded((low << (NS - R + M)) | (lane << M) | top)] = t[r];
  }
  lanes_sync<T>();
#pragma unroll
  for (int r = 0; r < NR; ++r) t[r] = buf[padded((r << (NS - R)) | lane)];
}

// `top`: the block starts a column (a compile-time fact except in tile passes).
template <int NS, int R, int M, int P, bool COLUMN, typename Mod, typename Signs, int... SS>
__device__ __forceinline__ void wide_phase(float2 (&t)[1 << R], float2* buf, const float2* bs,
                                           const mbqc_step* steps, int k0, int n, int lane, bool top,
                                           Mod& mod, const Signs& signs,
                                           std::integer_sequence<int, SS...>) {
  using W = Wide<NS, R, M>;
  constexpr int F = W::first(P);
  // a column plan has only full blocks
  ((COLUMN || k0 + F + SS < n
        ? wide_step<NS, R, F, SS, COLUMN>(t, mod(k0 + F + SS, bs[F + SS]), steps, k0 + F + SS, lane,
                                          F == 0 && top, signs)
        : void()),
   ...);
  wide_rotate<NS, R, W::len(P), W::T>(t, buf, lane);
}

template <int NS, int R, int M, bool COLUMN, typename Mod, typename Signs, int... PS>
__device__ __forceinline__ void wide_block(float2 (&t)[1 << R], float2* buf, const float2* bs,
                                           const mbqc_step* steps, int k0, int n, int lane, bool top,
                                           Mod& mod, const Signs& signs,
                                           std::integer_sequence<int, PS...>) {
  (wide_phase<NS, R, M, PS, COLUMN>(t, buf, bs, steps, k0, n, lane, top, mod, signs,
                                    std::make_integer_sequence<int, Wide<NS, R, M>::len(PS)>{}),
   ...);
}

// e^{-i theta} of the chunk of steps [k0, k0 + CS), one step per lane.
// (cl: the lane's place among the `clanes` lanes that evaluate them.)  POLY: from
// the float polynomials of the one-simulation-per-lane kernels, bit for bit.
template <int CS, bool REF, bool POLY = false>
__device__ __forceinline__ void wide_coeffs(float2* bs, const mbqc_step* steps, const float* ang,
                                            int64_t sa, int k0, int n, int cl, int clanes,
                                            RefPhase* ph) {
#pragma unroll 1
  for (int i = cl; i < CS; i += clanes) {
    const int k = k0 + i;
    if (k < n) {
      const float th = step_angle(steps[k], ang, sa);
      if constexpr (REF) ph->add(th);
      bs[i] = POLY ? step_coeff<false>(th, nullptr) : exp_minus_i(th);
    }
  }
}

// All steps of one simulation; `on_end(blk, t)` runs after every block.
template <int NS, int R, bool REF, bool COLUMN, bool POLY = false, typename OnEnd, typename Mod>
__device__ __forceinline__ void wide_run(float2 (&t)[1 << R], const Job& J, const float* ang,
                                         float2* buf, float2* bs, int cl, int clanes,
                                         RefPhase* ph, OnEnd on_end, Mod&& mod) {
  using W = Wide<NS, R>;
  const int lane = cl & (W::TL - 1);
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  const Constant<int32_t> resc = constant(J.tab + J.off_svres);
  const int n = J.n_steps;
  for (int kc = 0; kc < n; kc += W::CS) {
    // the previous chunk's last read came before its last exchange
    wide_coeffs<W::CS, REF, POLY>(bs, steps, ang, J.angle_stride_a, kc, n, cl, clanes, ph);
    lanes_sync<W::T>();
    const int ke = kc + W::CS < n ? kc + W::CS : n;
    for (int k0 = kc; k0 < ke; k0 += NS) {
      if (resc[k0 / NS]) {
#pragma unroll
        for (int r = 0; r < W::NR; ++r) t[r] = cscale(t[r], 0x1p-32f);
      }
      wide_block<NS, R, NS, COLUMN>(t, buf, bs + (k0 - kc), steps, k0, n, lane, true, mod,
                                    SlotSigns(), std::make_integer_sequence<int, W::P>{});
      on_end(k0 / NS, t);
    }
  }
}

template <int NS, int R>
__device__ __forceinline__ void wide_load(float2 (&t)[1 << R], const Job& J, int64_t si, int lane) {
  const int32_t* in_index = J.tab + J.off_in;
  const int32_t* sign = J.tab + J.off_sign;
  const float2* psi = J.psi + si * J.in_stride;
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    const int j = (r << (NS - R)) | lane;
    t[r] = flip(psi[in_index[j]], sign[j] ? 0x80000000u : 0u);
  }
}

// 1 / norm of the state over the output amplitudes (those with out_pos >= 0).
template <int NS, int R>
__device__ __forceinline__ float wide_inv_norm(const float2 (&t)[1 << R], const int32_t* out_pos,
                                               int lane, void* red) {
  float n2 = 0.0f;
#pragma unroll
  for (int r = 0; r < (1 << R); ++r)
    if (out_pos[(r << (NS - R)) | lane] >= 0) n2 = fmaf(t[r].x, t[r].x, fmaf(t[r].y, t[r].y, n2));
  return 1.0f / sqrtf(lanes_sum<Wide<NS, R>::TL>(n2, static_cast<float*>(red)));
}

// The same with the squares added in amplitude order on every lane, as the
// one-simulation-per-lane kernels add them (small states only).
template <int NS, int R>
__device__ __forceinline__ float wide_inv_norm_in_order(const float2 (&t)[1 << R],
                                                        const int32_t* out_pos, float2* buf,
                                                        int lane) {
  float n2 = 0.0f;
  if constexpr (R == NS) {
#pragma unroll
    for (int j = 0; j < (1 << NS); ++j)
      if (out_pos[j] >= 0) n2 = fmaf(t[j].x, t[j].x, fmaf(t[j].y, t[j].y, n2));
  } else {
    lanes_sync<Wide<NS, R>::TL>();
#pragma unroll
    for (int r = 0; r < (1 << R); ++r) buf[padded((r << (NS - R)) | lane)] = t[r];
    lanes_sync<Wide<NS, R>::TL>();
#pragma unroll
    for (int j = 0; j < (1 << NS); ++j) {
      const float2 v = buf[padded(j)];
      if (out_pos[j] >= 0) n2 = fmaf(v.x, v.x, fmaf(v.y, v.y, n2));
    }
  }
  return 1.0f / sqrtf(n2);
}

// Simulation g of job J on the lanes of one group (inactive groups run the
// last simulation and store nothing).  cl: the lane's place among the `clanes`
// lanes that share coefficients.
template <int NS, int R, bool REF, bool COLUMN, int SPARE = 0>
__device__ __forceinline__ void wide_sim(const Job& J, int64_t g, bool active, uint32_t flags,
                                         float2* buf, float2* bs, int cl,
                                         int clanes = Wide<NS, R, NS, SPARE>::CL) {
  using W = Wide<NS, R, NS, SPARE>;
  const int lane = cl & (W::TL - 1);
  const int64_t gg = active ? g : J.total - 1;
  int64_t bi, si;
  split_sim(J, gg, &bi, &si);
  float2 t[W::NR];
  wide_load<NS, R>(t, J, si, lane);
  RefPhase rp;
  constexpr bool kLaneKernelToo = NS <= 6;   // then equal to it bit for bit
  wide_run<NS, R, REF, COLUMN, kLaneKernelToo>(
      t, J, J.angles + bi * J.angle_stride, buf, bs, cl, clanes, &rp, [](int, const float2 (&)[W::NR]) {},
      NoModify());
  if constexpr (REF) {
    rp.m_sum = lanes_sum<W::CL>(rp.m_sum, reinterpret_cast<int32_t*>(bs));
    rp.th_sum = lanes_sum<W::CL>(rp.th_sum, reinterpret_cast<double*>(bs));
  }
  const float2 ph = REF ? rp.value() : make_float2(1.0f, 0.0f);
  const int32_t* out_pos = J.tab + J.off_out;
  float scale;
  if (!(flags & MBQC_FLAG_RENORMALIZE)) scale = sv_final_scale(J.e_sv);
  else if constexpr (kLaneKernelToo) scale = wide_inv_norm_in_order<NS, R>(t, out_pos, buf, lane);
  else scale = wide_inv_norm<NS, R>(t, out_pos, lane, bs);
  const float2 f = cscale(ph, scale);
  if (active && (SPARE == 0 || cl < W::TL)) {
    float2* o = J.out + g * (int64_t(1) << J.n_out);
#pragma unroll
    for (int r = 0; r < W::NR; ++r) {
      const int p = out_pos[(r << (NS - R)) | lane];
      if (p >= 0) o[p] = cmul(t[r], f);
    }
    if (lane == 0 && (flags & MBQC_FLAG_WRITE_PHASE) && J.phase_out) J.phase_out[g] = ph;
  }
}

template <int NS, int R, bool REF, bool COLUMN, int SPARE = 0>
__global__ __launch_bounds__((Wide<NS, R, NS, SPARE>::T)) void k_wide_sv(Job J, int64_t g0,
                                                                       uint32_t flags) {
  using W = Wide<NS, R, NS, SPARE>;
  __shared__ float2 lds[W::G * W::SIM];
  const int sub = threadIdx.x / W::CL, cl = threadIdx.x % W::CL;
  float2* buf = lds + sub * W::SIM;
  const int64_t g = g0 + int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  wide_sim<NS, R, REF, COLUMN, SPARE>(J, g, g < J.total, flags, buf, buf + W::BUF, cl);
}

// Lanes that evaluate one set of coefficients for simulations of `lanes` lanes,
// `same` of which in a row have the same angles: at most a wave.
inline int shared_lanes(int lanes, int64_t same) {
  for (; lanes < 64 && same % 2 == 0; same /= 2) lanes *= 2;
  return lanes;
}

// The same without the reference phase (whose sums stay with a simulation) for
// simulations that share their angles in groups of clanes / TL, at least 4 of them:
// no lanes are spent on coefficients alone.
template <int NS, int R, bool COLUMN>
__global__ __launch_bounds__((Wide<NS, R>::T)) void k_wide_sv_shared(Job J, uint32_t flags,
                                                                     int clanes) {
  using W = Wide<NS, R>;
  constexpr int SETS = (W::T + 63) / 64 * (W::TL >= 16 ? 1 : 64 / (4 * W::TL));
  __shared__ float2 lds[W::G * W::BUF + SETS * W::CS];
  const int sub = threadIdx.x / W::TL;
  const int64_t g = int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  wide_sim<NS, R, false, COLUMN>(J, g, g < J.total, flags, lds + sub * W::BUF,
                                 lds + W::G * W::BUF + int(threadIdx.x) / clanes * W::CS,
                                 int(threadIdx.x) % clanes, clanes);
}

// Sampled outcomes: the frame and draws of SampleMod, evaluated identically by
// every lane of a simulation; one lane writes the outcome words.
template <int NS, int R, bool COLUMN>
__global__ __launch_bounds__((Wide<NS, R>::T)) void k_wide_sample(
    Job J, const uint64_t* __restrict__ xm, const uint64_t* __restrict__ zm,
    const int32_t* __restrict__ out_off, int32_t* __restrict__ outcomes, int32_t words,
    uint64_t seed, int64_t g0) {
  using W = Wide<NS, R>;
  __shared__ float2 lds[W::G * W::SIM];
  const int sub = threadIdx.x / W::TL, lane = threadIdx.x % W::TL;
  float2* buf = lds + sub * W::SIM;
  float2* bs = buf + W::BUF;
  const int64_t g = g0 + int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  const bool active = g < J.total;
  const int64_t gg = active ? g : J.total - 1;
  int64_t bi, si;
  split_sim(J, gg, &bi, &si);
  float2 t[W::NR];
  wide_load<NS, R>(t, J, si, lane);
  int32_t* row = outcomes + gg * (words + 2);
  SampleMod mod;
  mod.seed = seed;
  mod.sim = uint64_t(gg);
  mod.xm = constant(xm);
  mod.zm = constant(zm);
  mod.n = J.n_steps;
  mod.out_words = active && lane == 0 ? row : nullptr;
  RefPhase ph;
  wide_run<NS, R, false, COLUMN>(t, J, J.angles + bi * J.angle_stride, buf, bs, lane, W::TL, &ph,
                                 [](int, const float2 (&)[W::NR]) {}, mod);
  uint32_t xo = 0, zo = 0;
  for (int m = 0; m < J.n_out; ++m) {
    const int off = out_off[m];
    xo |= ((mod.fx >> off) & 1u) << (J.n_out - 1 - m);
    zo |= ((mod.fz >> off) & 1u) << (J.n_out - 1 - m);
  }
  const int32_t* out_pos = J.tab + J.off_out;
  const float scale = wide_inv_norm<NS, R>(t, out_pos, lane, bs);
  if (!active) return;
  float2* o = J.out + g * (int64_t(1) << J.n_out);
#pragma unroll
  for (int r = 0; r < W::NR; ++r) {
    const int p = out_pos[(r << (NS - R)) | lane];
    if (p >= 0) {
      const uint32_t q = uint32_t(p) ^ xo;
      o[q] = flip(cscale(t[r], scale), czbit(q, zo));
    }
  }
  if (lane == 0) {
    row[words] = int32_t(xo);
    row[words + 1] = int32_t(zo);
  }
}

// Batched groups: a persistent workgroup pulls items from the group's counter
// and runs their simulations, G at a time.  Every thread reads the item index
// from LDS, so all leave the loop together once the counter passes n_items.
template <int NS, int R, bool REF, bool COLUMN>
__global__ __launch_bounds__((Wide<NS, R>::T)) void k_wide_batch(
    const Job* __restrict__ jobs, const BatchItem* __restrict__ items, int64_t n_items, int* counter,
    uint32_t flags) {
  using W = Wide<NS, R>;
  __shared__ float2 lds[W::G * W::SIM];
  __shared__ int item_s;
  const int sub = threadIdx.x / W::TL, lane = threadIdx.x % W::TL;
  float2* buf = lds + sub * W::SIM;
  for (;;) {
    __syncthreads();   // the previous item's last reads of item_s and the buffers are done
    if (threadIdx.x == 0) item_s = atomicAdd(counter, 1);
    __syncthreads();
    const int it = item_s;
    if (it >= n_items) break;
    const BatchItem I = items[it];
    const Job J = load_job(jobs, I.job);
    const int64_t end = std::min<int64_t>(I.first + I.count, J.total);
    for (int64_t g = I.first; g < end; g += W::G) {
      __syncthreads();
      wide_sim<NS, R, REF, COLUMN>(J, g + sub, g + sub < end, flags, buf, buf + W::BUF, lane);
    }
  }
}

// ---------------------------------------------------------------- adjoint
// Adjoint sweeps of column plans.  Every step of a column plan is invertible:
// new0 = x + b y, new1 = c (x - b y) with c the CZ sign, so
//   2x = new0 + c new1,   2 b y = new0 - c new1,
// and the backward sweep runs the state back from a checkpoint at the end of a
// group of ck blocks instead of recomputing it forward from the group's start
// and keeping every step's measured half.  With h = lam0 - c lam1 the cotangent of
// new0 (L real, dL = Re sum conj(lam) d(new)):
//   lam_x = lam0 + c lam1,   lam_y = conj(b) h,
//   dL/dtheta += Im(sum b y conj(h)).
// The factors 2 of the state are powers of two carried per block, so they round
// nothing; a state is at most ck blocks of steps away from its checkpoint.
// Bound by VALU issue (18 FMA-rate instructions per pair and step, two states
// in registers) and the two exchanges per phase.  8x6 grid, 509 sets x 4
// columns: backward 172 -> 20 us against one workgroup per row with the states
// and the measured halves in LDS and a barrier per step, forward 22.7 -> 14.2.
// Gradient error against 64 bits 3.6e-7 -> 3.0e-7 (the running back costs
// about 8%, the correctly rounded coefficients gain more: over 4 to 14
// rows, patterns of two measured columns are level with the recomputing sweeps, of
// three mostly 5 to 10% below them, of five 15 to 25%).
// Columns of one parameter set have the same angles: groups of `clanes` lanes
// (TL times a power of two of columns, at most a wave) evaluate one set of
// coefficients for their simulations.
template <int NS, int R>
struct AdjWide {
  using W = Wide<NS, R>;
  // float2 of LDS for `groups` simulations: `states` exchange buffers each, then
  // the coefficients
  __host__ __device__ static constexpr int lds(int groups, int states, int clanes) {
    return groups * states * W::BUF + (groups * W::TL + clanes - 1) / clanes * W::CS;
  }
  static int clanes(int64_t columns) { return shared_lanes(W::TL, columns); }
};

template <int NS, int R>
__global__ __launch_bounds__((Wide<NS, R>::T)) void k_wide_adj_forward(Job J,
                                                                       float2* __restrict__ ckpt,
                                                                       int ck, int clanes) {
  using W = Wide<NS, R>;
  extern __shared__ float2 lds[];
  const int sub = threadIdx.x / W::TL, lane = threadIdx.x % W::TL;
  const int64_t g = int64_t(xcd_block(blockIdx.x, gridDim.x)) * W::G + sub;
  const bool active = g < J.total;
  const int64_t gg = active ? g : J.total - 1;
  int64_t bi, si;
  split_sim(J, gg, &bi, &si);
  float2 t[W::NR];
  wide_load<NS, R>(t, J, si, lane);
  const int nblk = (J.n_steps + NS - 1) / NS;
  RefPhase ph;
  wide_run<NS, R, false, true>(
      t, J, J.angles + bi * J.angle_stride, lds + sub * W::BUF,
      lds + W::G * W::BUF + int(threadIdx.x) / clanes * W::CS, int(threadIdx.x) % clanes, clanes, &ph,
      [&](int blk, const float2 (&tt)[W::NR]) {
        if (((blk + 1) & (ck - 1)) != 0 && blk + 1 != nblk) return;   // ck: 1 or 2
        // inactive groups repeat the last simulation's stores
        float2* cp = ckpt + ((int64_t(blk >> (ck - 1)) * J.total + gg) << NS) + lane;
#pragma unroll
        for (int r = 0; r < W::NR; ++r) cp[r << (NS - R)] = tt[r];
      },
      NoModify());
  if (!active) return;
  const int32_t* out_pos = J.tab + J.off_out;
  const float scale = sv_final_scale(J.e_sv);
  float2* o = J.out + g * (int64_t(1) << J.n_out);
#pragma unroll
  for (int r = 0; r < W::NR; ++r) {
    const int p = out_pos[(r << (NS - R)) | lane];
    if (p >= 0) o[p] = cscale(t[r], scale);
  }
}

// The inverse exchange: v -> rotate-right(v, M), of the state and the cotangent.
// Up to 9 slots they have a buffer each and exchange at once; above, where a
// buffer is 8 KB and more, one after the other.
constexpr bool adj_two_buffers(int ns) { return ns <= 9; }

template <int NS, int R>
__device__ __forceinline__ void put_rows(const float2 (&t)[1 << R], float2* buf, int lane) {
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) buf[padded((r << (NS - R)) | lane)] = t[r];
}
template <int NS, int R, int M>
__device__ __forceinline__ void get_rotated(float2 (&t)[1 << R], const float2* buf, int lane) {
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    const int top = r >> (R - M), low = r & ((1 << (R - M)) - 1);
    t[r] = buf[padded((low << (NS - R + M)) | (lane << M) | top)];
  }
}
template <int NS, int R, int M, int TL>
__device__ __forceinline__ void wide_unrotate(float2 (&t)[1 << R], float2 (&lam)[1 << R], float2* buf,
                                              int lane) {
  lanes_sync<TL>();
  put_rows<NS, R>(t, buf, lane);
  if constexpr (adj_two_buffers(NS)) {
    float2* second = buf + Wide<NS, R>::BUF;
    put_rows<NS, R>(lam, second, lane);
    lanes_sync<TL>();
    get_rotated<NS, R, M>(t, buf, lane);
    get_rotated<NS, R, M>(lam, second, lane);
  } else {
    lanes_sync<TL>();
    get_rotated<NS, R, M>(t, buf, lane);
    lanes_sync<TL>();
    put_rows<NS, R>(lam, buf, lane);
    lanes_sync<TL>();
    get_rotated<NS, R, M>(lam, buf, lane);
  }
}

// Step FIRST + S backwards on state t (scaled by a power of two: doubled by
// each step) and cotangent lam; returns this lane's Im(sum 2 b y conj(h)).
template <int NS, int R, int FIRST, int S>
__device__ __forceinline__ float wide_unstep(float2 (&t)[1 << R], float2 (&lam)[1 << R], float2 b,
                                             int lane) {
  constexpr int NR = 1 << R, QB = 1 << (R - 1 - S);
  const float2 bc = cconj(b);
  const float lc = (S == 0 && FIRST > 0 && (lane & 1)) ? -1.0f : 1.0f;
  float d = 0.0f;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & QB) continue;
    const float c = S == 0 ? lc : ((r & (QB << 1)) ? -1.0f : 1.0f);
    const float2 u0 = t[r], u1 = t[r | QB], l0 = lam[r], l1 = lam[r | QB];
    const float2 y = make_float2(fmaf(-c, u1.x, u0.x), fmaf(-c, u1.y, u0.y));
    const float2 h = make_float2(fmaf(-c, l1.x, l0.x), fmaf(-c, l1.y, l0.y));
    d = fmaf(y.y, h.x, fmaf(-y.x, h.y, d));
    t[r] = make_float2(fmaf(c, u1.x, u0.x), fmaf(c, u1.y, u0.y));
    lam[r] = make_float2(fmaf(c, l1.x, l0.x), fmaf(c, l1.y, l0.y));
    t[r | QB] = cmul(bc, y);
    lam[r | QB] = cmul(bc, h);
  }
  return d;
}

// Where a lane puts the gradient entries of its simulation: acc[angle index]
// in LDS, one writer per simulation and wave (waves: entry stride n_angles).
struct GradSlot {
  float* acc;
  bool writer, first;
};

template <int NS, int R, int P, int... SS>
__device__ __forceinline__ void wide_unphase(float2 (&t)[1 << R], float2 (&lam)[1 << R], float2* buf,
                                             const float2 (&b)[NS], float (&d)[NS], int lane,
                                             std::integer_sequence<int, SS...>) {
  using W = Wide<NS, R>;
  constexpr int F = W::first(P), M = W::len(P);
  wide_unrotate<NS, R, M, W::TL>(t, lam, buf, lane);
  ((d[F + M - 1 - SS] = wide_unstep<NS, R, F, M - 1 - SS>(t, lam, b[F + M - 1 - SS], lane)), ...);
}

// A block backwards.  Its coefficients are read at the start and its gradient
// entries written at the end, so that the steps between have no LDS latency or
// branch of their own.  With few simulations the sweep is its chain of steps
// (16 sets of a 4x16 grid, 60 steps: 16.5 us, 29.4 us with one lane per
// simulation), with many the LDS exchanges and the adds across lanes (4096 sets:
// 40 us, one lane 41 us).
template <int NS, int R, int... PS>
__device__ __forceinline__ void wide_unblock(float2 (&t)[1 << R], float2 (&lam)[1 << R], float2* buf,
                                             const float2* bs, Constant<int32_t> aidx, int lane,
                                             const GradSlot& slot,
                                             std::integer_sequence<int, PS...>) {
  using W = Wide<NS, R>;
  float2 b[NS];
  float d[NS];
  int ai[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    b[k] = bs[k];
    ai[k] = aidx[k];
  }
  (wide_unphase<NS, R, W::P - 1 - PS>(t, lam, buf, b, d, lane,
                                      std::make_integer_sequence<int, W::len(W::P - 1 - PS)>{}),
   ...);
  // the state was doubled by each of the steps after step k
#pragma unroll
  for (int k = 0; k < NS; ++k)
    d[k] = last_lane_sum<(W::TL < 64 ? W::TL : 64)>(d[k]) * (1.0f / float(1 << (NS - k)));
  if (slot.writer) {
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (ai[k] >= 0) slot.acc[ai[k]] = slot.first ? d[k] : slot.acc[ai[k]] + d[k];
  }
}

// Backward sweep of a column plan: a workgroup holds N = blockDim / TL
// simulations at a time.  Rows of `red` <= N columns that are reduced together
// take `red` neighbouring groups (N / red rows per workgroup), longer ones
// run in red / N rounds.  Per-angle sums stay in LDS (one row of n_angles per
// group and wave of it) and are added up once at the end.
template <int NS, int R>
__global__ __launch_bounds__((Wide<NS, R>::TL > 256 ? Wide<NS, R>::TL : 256)) void k_wide_adj_backward(
    Job J, const float2* __restrict__ ckpt, const float2* __restrict__ seed, WideAdjoint A,
    int clanes, float* __restrict__ gpart) {
  using W = Wide<NS, R>;
  using AW = AdjWide<NS, R>;
  constexpr int TL = W::TL;
  constexpr int WV = TL > 64 ? TL / 64 : 1;       // waves of one simulation
  extern __shared__ float2 dyn[];
  const int N = blockDim.x / TL;
  const int sub = threadIdx.x / TL, lane = threadIdx.x % TL;
  constexpr int BUFS = adj_two_buffers(NS) ? 2 : 1;
  float2* buf = dyn + sub * BUFS * W::BUF;
  float2* bs = dyn + N * BUFS * W::BUF + int(threadIdx.x) / clanes * W::CS;
  const int cl = int(threadIdx.x) % clanes;
  float* accs = reinterpret_cast<float*>(dyn + AW::lds(N, BUFS, clanes));
  const int wave = TL > 64 ? lane >> 6 : 0;
  const int per = A.red < N ? A.red : N;          // columns of a row held at once
  const int rows = N / per;                       // rows of this workgroup
  const int64_t n_rows = (J.total / A.C) * A.P;
  const int64_t row0 = int64_t(xcd_block(blockIdx.x, gridDim.x)) * rows;
  const int64_t row = row0 + sub / per;
  const bool active = row < n_rows;
  const int64_t rr = active ? row : n_rows - 1;
  const int64_t bi = rr / A.P, r0 = rr - bi * A.P;
  const float* ang = J.angles + bi * J.angle_stride;
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  const Constant<int32_t> resc = constant(J.tab + J.off_svres);
  const int32_t* out_pos = J.tab + J.off_out;
  const Constant<int32_t> aidx = constant(J.tab + J.off_aidx);
  const float scale = sv_final_scale(J.e_sv);
  const int n = J.n_steps, nblk = n / NS;
  for (int a = threadIdx.x; a < N * WV * A.n_angles; a += blockDim.x) accs[a] = 0.0f;
  __syncthreads();
  GradSlot slot;
  slot.acc = accs + (sub * WV + wave) * A.n_angles;
  slot.writer = (threadIdx.x & ((TL < 64 ? TL : 64) - 1)) == (TL < 64 ? TL : 64) - 1;
  for (int c0 = 0; c0 < A.red; c0 += per) {
    slot.first = c0 == 0;
    const int64_t g = bi * A.C + r0 * A.red + c0 + sub % per;
    const float2* sd = seed + g * (int64_t(1) << J.n_out);
    float2 t[W::NR], lam[W::NR];
#pragma unroll
    for (int r = 0; r < W::NR; ++r) {
      const int p = out_pos[(r << (NS - R)) | lane];
      lam[r] = cscale(sd[p >= 0 ? p : 0], p >= 0 ? scale : 0.0f);
    }
    // the next checkpoint is on its way while a block runs (a load at the block's
    // start left every block waiting for it)
    constexpr bool kPrefetch = R <= 3;
    float2 ahead[kPrefetch ? W::NR : 1];
    auto load_ckpt = [&](int blk, auto& to) {
      const float2* cp = ckpt + ((int64_t(blk >> (A.ck - 1)) * J.total + g) << NS) + lane;
#pragma unroll
      for (int r = 0; r < W::NR; ++r) to[r] = cp[r << (NS - R)];
    };
    if constexpr (kPrefetch) load_ckpt(nblk - 1, ahead);
    for (int kc = ((n - 1) / W::CS) * W::CS; kc >= 0; kc -= W::CS) {
      lanes_sync<TL>();   // the previous chunk's reads are done
      wide_coeffs<W::CS, false>(bs, steps, ang, J.angle_stride_a, kc, n, cl, clanes, nullptr);
      lanes_sync<TL>();
      const int ke = kc + W::CS < n ? kc + W::CS : n;
      for (int blk = ke / NS - 1; blk * NS >= kc; --blk) {
        const bool at_ckpt = blk + 1 == nblk || ((blk + 1) & (A.ck - 1)) == 0;   // ck: 1 or 2
        if constexpr (kPrefetch) {
          if (at_ckpt) {
#pragma unroll
            for (int r = 0; r < W::NR; ++r) t[r] = ahead[r];
          }
          if (blk > 0 && (blk & (A.ck - 1)) == 0) load_ckpt(blk - 1, ahead);
        } else if (at_ckpt) {
          load_ckpt(blk, t);
        }
        wide_unblock<NS, R>(t, lam, buf, bs + (blk * NS - kc), aidx + blk * NS, lane, slot,
                            std::make_integer_sequence<int, W::P>{});
        // the block's doublings and rescale undone; the cotangent takes the rescale
        const bool rs = resc[blk] != 0;
        const float f = (rs ? 0x1p32f : 1.0f) / float(1 << NS);
#pragma unroll
        for (int r = 0; r < W::NR; ++r) t[r] = cscale(t[r], f);
        if (rs) {
#pragma unroll
          for (int r = 0; r < W::NR; ++r) lam[r] = cscale(lam[r], 0x1p-32f);
        }
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < rows * A.n_angles; i += blockDim.x) {
    const int q = i / A.n_angles, a = i - q * A.n_angles;
    float v = 0.0f;
    for (int c = 0; c < per * WV; ++c) v += accs[(q * per * WV + c) * A.n_angles + a];
    if (row0 + q < n_rows) gpart[(row0 + q) * A.n_angles + a] = v;
  }
}

// Register bits of the adjoint sweeps (two states).
constexpr int adj_reg_bits(int ns) { return ns <= 5 ? 2 : wide_reg_bits(ns); }

// Simulations per workgroup of the backward sweep: a row's columns together, up
// to 256 threads, in whole waves, as far as the LDS allows.  The LDS is taken
// for unshared coefficients, so that the choice depends on the plan and the
// columns per row only.
template <int NS>
size_t adj_backward_lds(int N, int n_angles, int clanes) {
  using A = AdjWide<NS, adj_reg_bits(NS)>;
  const int WV = A::W::TL > 64 ? A::W::TL / 64 : 1;
  return size_t(A::lds(N, adj_two_buffers(NS) ? 2 : 1, clanes)) * sizeof(float2) +
         size_t(N) * WV * n_angles * sizeof(float);
}

template <int NS>
int adj_backward_groups(int red, int n_angles) {
  constexpr int TL = Wide<NS, adj_reg_bits(NS)>::TL;
  int N = TL >= 256 ? 1 : std::min(256 / TL, red);
  if (N * TL < 64) N = 64 / TL;
  while (N > 1 && N * TL > 64 && adj_backward_lds<NS>(N, n_angles, TL) > kWideMaxLds / 2) N /= 2;
  return N;
}

template <int NS>
hipError_t adj_forward_launch(const Job& J, float2* ckpt, int ck, hipStream_t st) {
  constexpr int R = adj_reg_bits(NS);
  using W = Wide<NS, R>;
  const int clanes = AdjWide<NS, R>::clanes(J.S);
  const size_t lds = size_t(AdjWide<NS, R>::lds(W::G, 1, clanes)) * sizeof(float2);
  const void* kern = reinterpret_cast<const void*>(&k_wide_adj_forward<NS, R>);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_wide_adj_forward<NS, R>), dim3(unsigned((J.total + W::G - 1) / W::G)),
                     dim3(W::T), lds, st, J, ckpt, ck, clanes);
  return hipGetLastError();
}

template <int NS>
hipError_t adj_backward_launch(const Job& J, const float2* ckpt, const float2* seed,
                               const WideAdjoint& A, float* gpart, hipStream_t st) {
  constexpr int R = adj_reg_bits(NS);
  constexpr int TL = Wide<NS, R>::TL;
  const int N = adj_backward_groups<NS>(A.red, A.n_angles);
  // neighbouring groups are columns of one row as far as the row goes
  const int clanes = AdjWide<NS, R>::clanes(std::min(A.red, N));
  const size_t lds = adj_backward_lds<NS>(N, A.n_angles, clanes);
  const void* kern = reinterpret_cast<const void*>(&k_wide_adj_backward<NS, R>);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
  }
  const int rows = N / std::min(A.red, N);
  const int64_t n_rows = (J.total / A.C) * A.P;
  hipLaunchKernelGGL((k_wide_adj_backward<NS, R>), dim3(unsigned((n_rows + rows - 1) / rows)),
                     dim3(unsigned(N * TL)), lds, st, J, ckpt, seed, A, clanes, gpart);
  return hipGetLastError();
}

// ---------------------------------------------------------------- tile passes
// Windows of 15..20 slots: the state is cut into tiles of 2^kTileBits
// amplitudes and a pass runs M steps on every tile, one workgroup each, so
// that a single simulation already spreads over 2^(ns - kTileBits) workgroups
// (one workgroup walking the whole state is bound by its own memory latency).
// With v the amplitude in the current rotation (the next slots to measure are
// its top bits) a tile holds all values of the top M bits and of the lowest
// kTileBits - M bits; the other bits (`mid`) name the tile.  It reads runs of
// 2^(kTileBits - M) amplitudes and, as rotate-left(v, M) puts the measured
// bits lowest, writes one contiguous run.  The passes alternate between two
// buffers; the first reads the input, the last leaves the output unscaled and
// one partial norm per tile, which k_tile_finish applies.  With few simulations
// the passes are bound by their own launch and memory latency (5-9 us each, six
// of them for three columns of 16 slots): 16x4 grid, 4 simulations, 1,470 us
// with one workgroup per simulation, 61 us so.
constexpr int kTileBits = 12;
constexpr int kTileRegBits = 4;

struct TileSigns {
  int ns, m, sub;
  uint32_t mid;
  __device__ __forceinline__ StepSigns operator()(const mbqc_step& st) const {
    const int c = kTileBits - m;
    const uint32_t all = (1u << ns) - 1;
    const uint32_t v = sub ? ((st.nmask << sub) | (st.nmask >> (ns - sub))) & all : st.nmask;
    const uint32_t low = v & ((1u << c) - 1), top = v >> (ns - m);
    const uint32_t outer = (v >> c) & ((1u << (ns - kTileBits)) - 1);
    return {(top << c) | low, czbit(mid, outer)};
  }
};

// One pass: steps [k0, k0 + M) of simulation g of J, whose state is the l-th of the
// buffers; `sub`: the rotation before it (k0 % ns).  in == nullptr: the first pass
// (the input state); `last`: the output and its partial norms.
template <int M, bool COLUMN>
__device__ __forceinline__ void tile_pass(const Job& J, int64_t g, int64_t l,
                                          const float2* __restrict__ in, float2* __restrict__ out,
                                          float* __restrict__ norms, int k0, int sub, bool last) {
  using W = Wide<kTileBits, kTileRegBits, M>;
  constexpr int C = kTileBits - M;
  __shared__ float2 buf[W::BUF];
  __shared__ float2 bs[M];
  __shared__ float red[W::T / 64];
  const int lane = threadIdx.x;
  const uint32_t mid = blockIdx.x & ((1u << (J.ns - kTileBits)) - 1);
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  const Constant<int32_t> resc = constant(J.tab + J.off_svres);
  int64_t bi, si;
  split_sim(J, g, &bi, &si);
  float2 t[W::NR];
  const int64_t state = l << J.ns;
#pragma unroll
  for (int r = 0; r < W::NR; ++r) {
    const int u = r * W::TL + lane;
    const int v = ((u >> C) << (J.ns - M)) | int(mid << C) | (u & ((1 << C) - 1));
    if (in) {
      t[r] = in[state + v];
    } else {
      const int32_t* in_index = J.tab + J.off_in;
      const int32_t* sign = J.tab + J.off_sign;
      t[r] = flip(J.psi[si * J.in_stride + in_index[v]], sign[v] ? 0x80000000u : 0u);
    }
  }
  wide_coeffs<M, false>(bs, steps, J.angles + bi * J.angle_stride, J.angle_stride_a, k0, J.n_steps,
                        lane, W::T, nullptr);
  __syncthreads();
  if (sub == 0 && resc[k0 / J.ns]) {
#pragma unroll
    for (int r = 0; r < W::NR; ++r) t[r] = cscale(t[r], 0x1p-32f);
  }
  NoModify mod;
  wide_block<kTileBits, kTileRegBits, M, COLUMN>(t, buf, bs, steps, k0, J.n_steps, lane, sub == 0,
                                                 mod, TileSigns{J.ns, M, sub, mid},
                                                 std::make_integer_sequence<int, W::P>{});
  const int base = int(mid << kTileBits);
  if (!last) {
#pragma unroll
    for (int r = 0; r < W::NR; ++r) out[state + base + r * W::TL + lane] = t[r];
    return;
  }
  const int32_t* out_pos = J.tab + J.off_out;
  float2* o = J.out + g * (int64_t(1) << J.n_out);
  float n2 = 0.0f;
#pragma unroll
  for (int r = 0; r < W::NR; ++r) {
    const int p = out_pos[base + r * W::TL + lane];
    if (p >= 0) {
      o[p] = t[r];
      n2 = fmaf(t[r].x, t[r].x, fmaf(t[r].y, t[r].y, n2));
    }
  }
  n2 = lanes_sum<256>(n2, red);
  if (lane == 0) norms[blockIdx.x] = n2;
}

// Workgroup b runs tile b % tiles of simulation b / tiles: simulations g0, g0 + 1, ...
// of one job, or (batches) those that a list names, of several jobs.
template <int M, bool COLUMN>
__global__ __launch_bounds__((Wide<kTileBits, kTileRegBits>::T)) void k_tile_pass(
    Job J, const float2* __restrict__ in, float2* __restrict__ out, float* __restrict__ norms,
    int64_t g0, int k0, int sub, int last) {
  const int64_t l = int64_t(blockIdx.x) >> (J.ns - kTileBits);
  tile_pass<M, COLUMN>(J, g0 + l, l, in, out, norms, k0, sub, last);
}

template <int M, bool COLUMN>
__global__ __launch_bounds__((Wide<kTileBits, kTileRegBits>::T)) void k_tile_pass_jobs(
    const Job* __restrict__ jobs, const BatchItem* __restrict__ sims, int ns,
    const float2* __restrict__ in, float2* __restrict__ out, float* __restrict__ norms, int k0,
    int sub, int block_end) {
  const int64_t l = int64_t(blockIdx.x) >> (ns - kTileBits);
  const BatchItem I = sims[l];
  const Job J = load_job(jobs, I.job);
  // a job is done with the block that holds its last step
  const bool last = block_end && k0 - sub + ns >= J.n_steps;
  tile_pass<M, COLUMN>(J, I.first, l, in, out, norms, k0, sub, last);
}

// Phase and scale of the outputs a last pass left: workgroup (x, y) takes
// 1,024 amplitudes of the y-th simulation.
__device__ __forceinline__ void tile_finish(const Job& J, int64_t g, int64_t l,
                                            const float* __restrict__ norms, uint32_t flags) {
  __shared__ float red_f[4];
  __shared__ double red_d[4];
  __shared__ int32_t red_i[4];
  const int64_t dout = int64_t(1) << J.n_out;
  const int64_t e0 = int64_t(blockIdx.x) * 1024;
  if (e0 >= dout) return;
  const int tid = threadIdx.x;
  const int tiles = 1 << (J.ns - kTileBits);
  const mbqc_step* steps = reinterpret_cast<const mbqc_step*>(J.tab);
  float2 ph = make_float2(1.0f, 0.0f);
  if (flags & MBQC_FLAG_REF_PHASE) {
    int64_t bi, si;
    split_sim(J, g, &bi, &si);
    const float* ang = J.angles + bi * J.angle_stride;
    RefPhase rp;
    for (int k = tid; k < J.n_steps; k += 256) rp.add(step_angle(steps[k], ang, J.angle_stride_a));
    rp.m_sum = lanes_sum<256>(rp.m_sum, red_i);
    rp.th_sum = lanes_sum<256>(rp.th_sum, red_d);
    ph = rp.value();
  }
  float scale = sv_final_scale(J.e_sv);
  if (flags & MBQC_FLAG_RENORMALIZE) {
    float n2 = 0.0f;
    for (int i = tid; i < tiles; i += 256) n2 += norms[l * tiles + i];
    scale = 1.0f / sqrtf(lanes_sum<256>(n2, red_f));
  }
  const float2 f = cscale(ph, scale);
  float2* o = J.out + g * dout;
  for (int64_t e = e0 + tid; e < e0 + 1024 && e < dout; e += 256) o[e] = cmul(o[e], f);
  if (blockIdx.x == 0 && tid == 0 && (flags & MBQC_FLAG_WRITE_PHASE) && J.phase_out)
    J.phase_out[g] = ph;
}

__global__ __launch_bounds__(256) void k_tile_finish(Job J, const float* __restrict__ norms,
                                                     int64_t g0, uint32_t flags) {
  tile_finish(J, g0 + blockIdx.y, blockIdx.y, norms, flags);
}

__global__ __launch_bounds__(256) void k_tile_finish_jobs(const Job* __restrict__ jobs,
                                                          const BatchItem* __restrict__ sims,
                                                          const float* __restrict__ norms,
                                                          uint32_t flags) {
  const BatchItem I = sims[blockIdx.y];
  tile_finish(load_job(jobs, I.job), I.first, blockIdx.y, norms, flags);
}

// The passes of patterns of up to `blocks` blocks: at most 8 steps each, of near equal
// length within a block.  pass(std::integral_constant<int, M>, block, k0, sub,
// block_end): after a block's last pass the rotation is back at slot order.
template <typename Pass>
hipError_t tile_passes(int ns, int blocks, Pass&& pass) {
  const int per = (ns + 7) / 8;
  for (int blk = 0; blk < blocks; ++blk) {
    int sub = 0;
    for (int p = 0; p < per; ++p) {
      const int m = ns / per + (p < ns % per ? 1 : 0);
      const int k0 = blk * ns + sub;
      const bool end = p + 1 == per;
      switch (m) {
        case 5: pass(std::integral_constant<int, 5>{}, blk, k0, sub, end); break;
        case 6: pass(std::integral_constant<int, 6>{}, blk, k0, sub, end); break;
        case 7: pass(std::integral_constant<int, 7>{}, blk, k0, sub, end); break;
        case 8: pass(std::integral_constant<int, 8>{}, blk, k0, sub, end); break;
        default: return hipErrorInvalidValue;
      }
      sub += m;
    }
  }
  return hipSuccess;
}

// launch(grid, g0) over all simulations.  (13 and 14 slots take 512 and 1,024 threads per
// simulation: 8,388,608 and 4,194,304 of them are more than one launch has.)
template <typename W, typename Launch>
hipError_t in_sim_grids(int64_t total, Launch&& launch) {
  return in_grids((total + W::G - 1) / W::G, W::T, hipSuccess, [&](int64_t first, int64_t count) {
    launch(dim3(unsigned(count)), first * W::G);
    return hipGetLastError();
  });
}

template <int NS>
hipError_t sv_launch(const Job& J, bool column, uint32_t flags, hipStream_t st) {
  constexpr int R = wide_reg_bits(NS);
  using W = Wide<NS, R>;
  const bool ref = flags & MBQC_FLAG_REF_PHASE;
  return in_sim_grids<W>(J.total, [&](dim3 grid, int64_t g0) {
    const dim3 block(W::T);
    if (column) {
      if (ref) hipLaunchKernelGGL((k_wide_sv<NS, R, true, true>), grid, block, 0, st, J, g0, flags);
      else hipLaunchKernelGGL((k_wide_sv<NS, R, false, true>), grid, block, 0, st, J, g0, flags);
    } else {
      if (ref) hipLaunchKernelGGL((k_wide_sv<NS, R, true, false>), grid, block, 0, st, J, g0, flags);
      else hipLaunchKernelGGL((k_wide_sv<NS, R, false, false>), grid, block, 0, st, J, g0, flags);
    }
  });
}

// Windows of 1..6 slots with too few simulations to fill the chip at one per
// lane, where a launch takes as long as one lane's chain of steps: here the
// lanes of a group share a simulation's coefficients (one step per lane) and,
// from 4 slots on, its amplitudes, 4 per lane.  A group is a whole wave up to
// 1,024 simulations (one wave per SIMD), else 8 lanes (6 slots: 16).
constexpr int narrow_reg_bits(int ns) { return ns <= 3 ? ns : 2; }

// Most simulations that run so.  Measured in replayed graphs, us per launch (one lane
// per simulation / this), angle-major angles: 2 slots, 40 columns, 16 sims 9.7 / 8.9,
// 512 10.1 / 9.7, 768 10.1 / 10.6, 4,096 10.3 / 13.0; 3 slots, 40 columns, 16 sims
// 16.5 / 14.5, 512 17.1 / 15.1, 640 17.0 / 17.6, 2,048 17.1 / 19.0 (rows of angles: 2
// slots, 2,048 sims 11.6 / 11.4, 3 slots 17.5 / 18.5; 4 and 80 columns cross at the
// same sizes).  30-column grids: 4 slots 64 22.4 / 11.2, 8,192 23.6 / 20.4, 16,384
// 24.0 / 23.8, 32,768 24.8 / 38.5; 5 slots 64 45.5 / 14.1, 16,384 48.0 / 32.4,
// 32,768 49.9 / 54.2; 6 slots 64 86 / 14.7, 32,768 94.7 / 75.6.  One slot: no gain.
constexpr int64_t kNarrowMaxSims[7] = {0, 0, 512, 512, 16384, 16384, 32768};

template <int NS, int SPARE>
hipError_t narrow_launch(const Job& J, bool column, uint32_t flags, hipStream_t st) {
  constexpr int R = narrow_reg_bits(NS);
  using W = Wide<NS, R, NS, SPARE>;
  const dim3 grid(unsigned((J.total + W::G - 1) / W::G)), block(W::T);
  const bool ref = flags & MBQC_FLAG_REF_PHASE;
#define MBQC_NARROW(REF, COL) \
  hipLaunchKernelGGL((k_wide_sv<NS, R, REF, COL, SPARE>), grid, block, 0, st, J, int64_t(0), flags)
  if (column) {
    if (ref) MBQC_NARROW(true, true);
    else MBQC_NARROW(false, true);
  } else {
    if (ref) MBQC_NARROW(true, false);
    else MBQC_NARROW(false, false);
  }
#undef MBQC_NARROW
  return hipGetLastError();
}

template <int NS>
hipError_t shared_launch(const Job& J, bool column, uint32_t flags, hipStream_t st) {
  constexpr int R = narrow_reg_bits(NS);
  using W = Wide<NS, R>;
  const dim3 grid(unsigned((J.total + W::G - 1) / W::G)), block(W::T);
  const int clanes = shared_lanes(W::TL, J.S);
  if (column)
    hipLaunchKernelGGL((k_wide_sv_shared<NS, R, true>), grid, block, 0, st, J, flags, clanes);
  else
    hipLaunchKernelGGL((k_wide_sv_shared<NS, R, false>), grid, block, 0, st, J, flags, clanes);
  return hipGetLastError();
}

template <int NS>
hipError_t narrow_launch(const Job& J, bool column, uint32_t flags, hipStream_t st) {
  constexpr int lane_bits = NS - narrow_reg_bits(NS);
  if constexpr (kNarrowMaxSims[NS] <= 1024) return narrow_launch<NS, 6 - lane_bits>(J, column, flags, st);
  else if (J.total <= 1024) return narrow_launch<NS, 6 - lane_bits>(J, column, flags, st);
  else return narrow_launch<NS, (lane_bits < 3 ? 3 - lane_bits : 0)>(J, column, flags, st);
}

// One simulation whose angles and input come with the kernel's arguments and
// whose output goes to memory that the host reads: a whole call is one launch,
// with no copies before or after it.  The arguments are staged in LDS, from
// where a wave runs the simulation as narrow_launch's whole-wave form does.
// Bound by the launch and the wait for it: a 2x5 grid's call takes 22 us, 74 us
// with tensors made, copied and read back around the launch.
template <int NS, bool REF, bool COLUMN>
__global__ __launch_bounds__(64) void k_run_one(Job J, HostInputs in, uint32_t flags) {
  constexpr int R = narrow_reg_bits(NS), SPARE = 6 - (NS - R);
  using W = Wide<NS, R, NS, SPARE>;
  __shared__ float2 lds[W::SIM];
  __shared__ __align__(8) uint32_t staged[kHostInputWords];
  for (int i = threadIdx.x; i < in.n_words; i += 64) staged[i] = in.word[i];
  lanes_sync<64>();
  J.psi = reinterpret_cast<const float2*>(staged);
  J.angles = reinterpret_cast<const float*>(staged + in.first_angle);
  wide_sim<NS, R, REF, COLUMN, SPARE>(J, 0, true, flags, lds, lds + W::BUF, threadIdx.x);
}

template <int NS>
hipError_t run_one_launch(const Job& J, const HostInputs& in, bool column, uint32_t flags,
                          hipStream_t st) {
  const bool ref = flags & MBQC_FLAG_REF_PHASE;
#define MBQC_RUN_ONE(REF, COL) \
  hipLaunchKernelGGL((k_run_one<NS, REF, COL>), dim3(1), dim3(64), 0, st, J, in, flags)
  if (column) {
    if (ref) MBQC_RUN_ONE(true, true);
    else MBQC_RUN_ONE(false, true);
  } else {
    if (ref) MBQC_RUN_ONE(true, false);
    else MBQC_RUN_ONE(false, false);
  }
#undef MBQC_RUN_ONE
  return hipGetLastError();
}

template <int NS>
hipError_t sample_launch(const Job& J, bool column, const uint64_t* xm, const uint64_t* zm,
                         const int32_t* out_off, int32_t* outcomes, int32_t words, uint64_t seed,
                         hipStream_t st) {
  constexpr int R = wide_reg_bits(NS);
  using W = Wide<NS, R>;
  return in_sim_grids<W>(J.total, [&](dim3 grid, int64_t g0) {
    const dim3 block(W::T);
    if (column)
      hipLaunchKernelGGL((k_wide_sample<NS, R, true>), grid, block, 0, st, J, xm, zm, out_off, outcomes,
                         words, seed, g0);
    else
      hipLaunchKernelGGL((k_wide_sample<NS, R, false>), grid, block, 0, st, J, xm, zm, out_off,
                         outcomes, words, seed, g0);
  });
}

template <int NS>
hipError_t batch_launch(bool column, int64_t waves, const Job* jobs, const BatchItem* items,
                        int64_t n_items, int* counter, uint32_t flags, hipStream_t st) {
  constexpr int R = wide_reg_bits(NS);
  using W = Wide<NS, R>;
  const int64_t wgs = std::max<int64_t>(1, std::min<int64_t>(waves / (W::T / 64), n_items));
  const dim3 grid{unsigned(wgs)}, block(W::T);
  const bool ref = flags & MBQC_FLAG_REF_PHASE;
#define MBQC_WIDE_BATCH(REF, COL)                                                                \
  hipLaunchKernelGGL((k_wide_batch<NS, R, REF, COL>), grid, block, 0, st, jobs, items, n_items, \
                     counter, flags)
  if (column) {
    if (ref) MBQC_WIDE_BATCH(true, true);
    else MBQC_WIDE_BATCH(false, true);
  } else {
    if (ref) MBQC_WIDE_BATCH(true, false);
    else MBQC_WIDE_BATCH(false, false);
  }
#undef MBQC_WIDE_BATCH
  return hipGetLastError();
}

}  // namespace

#define MBQC_WIDE_SWITCH(ns, CALL)        \
  switch (ns) {                           \
    case 7: return CALL(7);               \
    case 8: return CALL(8);               \
    case 9: return CALL(9);               \
    case 10: return CALL(10);             \
    case 11: return CALL(11);             \
    case 12: return CALL(12);             \
    case 13: return CALL(13);             \
    case 14: return CALL(14);             \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_run_one(const Job& J, const HostInputs& in, bool column, uint32_t flags,
                          hipStream_t st) {
  switch (J.ns) {
    case 1: return run_one_launch<1>(J, in, column, flags, st);
    case 2: return run_one_launch<2>(J, in, column, flags, st);
    case 3: return run_one_launch<3>(J, in, column, flags, st);
    case 4: return run_one_launch<4>(J, in, column, flags, st);
    case 5: return run_one_launch<5>(J, in, column, flags, st);
    case 6: return run_one_launch<6>(J, in, column, flags, st);
    default: return hipErrorInvalidValue;
  }
}

// Most simulations that run with their angles' coefficients shared (raw phase, inputs a
// multiple of 4).  Both forms take time in proportion to the steps, but the one with
// one simulation per lane waits for the same memory latencies whatever the steps, so
// that the line lies higher for short patterns.  Replayed graphs, us (one simulation
// per lane / shared), 4 inputs: 4 slots, 33 columns, 32,768 sims 27.2 / 26.7; 80
// columns, 28,672 sims 55.2 / 54.1, 32,768 55.1 / 57.4; 5 slots, 26 columns, 32,768 sims
// 44.7 / 41.7; 80 columns, 28,672 sims 105.4 / 103.6, 32,768 105.5 / 115.6; 6 slots, 13
// columns, 131,072 sims 110 / 98; 20 columns, 49,152 sims 74.6 / 61.5, 131,072 112 / 150;
// 41 columns, 49,152 sims 127.7 / 122.5, 65,536 131 / 159; 80 columns, 40,960 sims
// 219 / 199, 49,152 (16 inputs) 218 / 236.
static int64_t shared_max(const Job& J, uint32_t flags) {
  if (J.S % 4 != 0 || (flags & MBQC_FLAG_REF_PHASE)) return 0;
  switch (J.ns) {
    case 4:
    case 5: return J.n_steps <= 128 ? 32768 : 28672;
    case 6: return J.n_steps <= 72 ? 131072 : J.n_steps <= 240 ? 49152 : 40960;
    default: return 0;
  }
}

bool narrow_sv(const Job& J, uint32_t flags) {
  return J.ns <= 6 && J.total <= std::max(kNarrowMaxSims[J.ns], shared_max(J, flags));
}

hipError_t launch_narrow_sv(const Job& J, bool column, uint32_t flags, hipStream_t st) {
  if (J.total > 1024 && J.total <= shared_max(J, flags)) {
    if (J.ns == 4) return shared_launch<4>(J, column, flags, st);
    if (J.ns == 5) return shared_launch<5>(J, column, flags, st);
    return shared_launch<6>(J, column, flags, st);
  }
  switch (J.ns) {
    case 2: return narrow_launch<2>(J, column, flags, st);
    case 3: return narrow_launch<3>(J, column, flags, st);
    case 4: return narrow_launch<4>(J, column, flags, st);
    case 5: return narrow_launch<5>(J, column, flags, st);
    case 6: return narrow_launch<6>(J, column, flags, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_wide_sv(const Job& J, bool column, uint32_t flags, hipStream_t st) {
#define MBQC_CALL(NS) sv_launch<NS>(J, column, flags, st)
  MBQC_WIDE_SWITCH(J.ns, MBQC_CALL)
#undef MBQC_CALL
}

size_t wide_tile_bytes(int ns) {
  return 2 * (sizeof(float2) << ns) + (sizeof(float) << (ns - kTileBits));
}

hipError_t launch_wide_tiles(const Job& J, bool column, uint32_t flags, void* ws, int64_t g0,
                             int64_t n, hipStream_t st) {
  float2* a = static_cast<float2*>(ws);
  float2* b = a + (n << J.ns);
  float* norms = reinterpret_cast<float*>(b + (n << J.ns));
  const float2* in = nullptr;
  const dim3 grid(unsigned(n << (J.ns - kTileBits))), block(Wide<kTileBits, kTileRegBits>::T);
  const int blocks = (J.n_steps + J.ns - 1) / J.ns;
  const hipError_t e = tile_passes(J.ns, blocks, [&](auto m, int blk, int k0, int sub, bool end) {
    constexpr int M = decltype(m)::value;
    const int last = end && blk + 1 == blocks;
    float2* out = in == a ? b : a;
    if (column)
      hipLaunchKernelGGL((k_tile_pass<M, true>), grid, block, 0, st, J, in, out, norms, g0, k0, sub,
                         last);
    else
      hipLaunchKernelGGL((k_tile_pass<M, false>), grid, block, 0, st, J, in, out, norms, g0, k0, sub,
                         last);
    in = out;
  });
  if (e != hipSuccess) return e;
  const unsigned chunks = unsigned(((int64_t(1) << J.n_out) + 1023) / 1024);
  for (int64_t y = 0; y < n; y += 65535) {   // grid rows are limited to 65,535
    const unsigned ny = unsigned(std::min<int64_t>(n - y, 65535));
    hipLaunchKernelGGL(k_tile_finish, dim3(chunks, ny), dim3(256), 0, st, J,
                       norms + (y << (J.ns - kTileBits)), g0 + y, flags);
  }
  return hipGetLastError();
}

hipError_t launch_wide_tiles_jobs(int ns, bool column, uint32_t flags, const Job* jobs,
                                  const BatchItem* sims, int64_t n, const int64_t* active, int blocks,
                                  int max_out, void* ws, hipStream_t st) {
  float2* a = static_cast<float2*>(ws);
  float2* b = a + (n << ns);
  float* norms = reinterpret_cast<float*>(b + (n << ns));
  const float2* in = nullptr;
  const dim3 block(Wide<kTileBits, kTileRegBits>::T);
  const hipError_t e = tile_passes(ns, blocks, [&](auto m, int blk, int k0, int sub, bool end) {
    constexpr int M = decltype(m)::value;
    const dim3 grid(unsigned(active[blk] << (ns - kTileBits)));
    float2* out = in == a ? b : a;
    if (column)
      hipLaunchKernelGGL((k_tile_pass_jobs<M, true>), grid, block, 0, st, jobs, sims, ns, in, out,
                         norms, k0, sub, int(end));
    else
      hipLaunchKernelGGL((k_tile_pass_jobs<M, false>), grid, block, 0, st, jobs, sims, ns, in, out,
                         norms, k0, sub, int(end));
    in = out;
  });
  if (e != hipSuccess) return e;
  const unsigned chunks = unsigned(((int64_t(1) << max_out) + 1023) / 1024);
  hipLaunchKernelGGL(k_tile_finish_jobs, dim3(chunks, unsigned(n)), dim3(256), 0, st, jobs, sims, norms,
                     flags);
  return hipGetLastError();
}

hipError_t launch_wide_sample(const Job& J, bool column, const uint64_t* xm, const uint64_t* zm,
                              const int32_t* out_off, int32_t* outcomes, int32_t words,
                              uint64_t seed, hipStream_t st) {
#define MBQC_CALL(NS) sample_launch<NS>(J, column, xm, zm, out_off, outcomes, words, seed, st)
  MBQC_WIDE_SWITCH(J.ns, MBQC_CALL)
#undef MBQC_CALL
}

hipError_t launch_wide_batch(int ns, bool column, int64_t waves, const Job* jobs,
                             const BatchItem* items, int64_t n_items, int* counter, uint32_t flags,
                             hipStream_t st) {
#define MBQC_CALL(NS) batch_launch<NS>(column, waves, jobs, items, n_items, counter, flags, st)
  MBQC_WIDE_SWITCH(ns, MBQC_CALL)
#undef MBQC_CALL
}

bool wide_adjoint_fits(int ns, int red, int n_angles) {
#define MBQC_CALL(NS)                                                                          \
  adj_backward_lds<NS>(adj_backward_groups<NS>(red, n_angles), n_angles,                       \
                       Wide<NS, adj_reg_bits(NS)>::TL) <= kWideMaxLds
  switch (ns) {
    case 4: return MBQC_CALL(4);
    case 5: return MBQC_CALL(5);
    case 6: return MBQC_CALL(6);
    case 7: return MBQC_CALL(7);
    case 8: return MBQC_CALL(8);
    case 9: return MBQC_CALL(9);
    case 10: return MBQC_CALL(10);
    case 11: return MBQC_CALL(11);
    case 12: return MBQC_CALL(12);
    case 13: return MBQC_CALL(13);
    case 14: return MBQC_CALL(14);
    default: return false;
  }
#undef MBQC_CALL
}

#define MBQC_ADJ_SWITCH(ns, CALL)         \
  switch (ns) {                           \
    case 4: return CALL(4);               \
    case 5: return CALL(5);               \
    case 6: return CALL(6);               \
    case 7: return CALL(7);               \
    case 8: return CALL(8);               \
    case 9: return CALL(9);               \
    case 10: return CALL(10);             \
    case 11: return CALL(11);             \
    case 12: return CALL(12);             \
    case 13: return CALL(13);             \
    case 14: return CALL(14);             \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_wide_adj_forward(const Job& J, float2* ckpt, int ck, hipStream_t st) {
#define MBQC_CALL(NS) adj_forward_launch<NS>(J, ckpt, ck, st)
  MBQC_ADJ_SWITCH(J.ns, MBQC_CALL)
#undef MBQC_CALL
}

hipError_t launch_wide_adj_backward(const Job& J, const float2* ckpt, const float2* seed,
                                    const WideAdjoint& A, float* gpart, hipStream_t st) {
#define MBQC_CALL(NS) adj_backward_launch<NS>(J, ckpt, seed, A, gpart, st)
  MBQC_ADJ_SWITCH(J.ns, MBQC_CALL)
#undef MBQC_CALL
}

}  // namespace mbqc
