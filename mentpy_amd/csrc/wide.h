// Launchers of the register-blocked kernels (wide.hip): live windows of 7..20
// slots, small batches of narrower ones, adjoint sweeps.  They need a plan whose
// measured slots follow the rotation (Plan::rotating).
#pragma once
#include "device.h"

namespace mbqc {

// `column`: every step is that of a grid in column order (Plan::column_steps),
// so the CZ signs are compile-time constants.
hipError_t launch_wide_sv(const Job& J, bool column, uint32_t flags, hipStream_t st);
// The same for windows of 2..6 slots, where narrow_sv says that the batch is
// too small for one simulation per lane.
bool narrow_sv(const Job& J, uint32_t flags);
hipError_t launch_narrow_sv(const Job& J, bool column, uint32_t flags, hipStream_t st);
// One simulation of a window of 1..6 slots, its input state (2^n_in amplitudes,
// from word 0) and angles (from word first_angle) passed by value.
constexpr int kHostInputWords = 896;   // with the Job within the 4 KiB of kernel arguments
struct HostInputs {
  int32_t n_words, first_angle;
  uint32_t word[kHostInputWords];
};
hipError_t launch_run_one(const Job& J, const HostInputs& in, bool column, uint32_t flags,
                          hipStream_t st);
// Windows of 15..20 slots: simulations [g0, g0 + n) in passes over tiles of
// their states, in a workspace of n * wide_tile_bytes(ns) bytes.
size_t wide_tile_bytes(int ns);
hipError_t launch_wide_tiles(const Job& J, bool column, uint32_t flags, void* ws, int64_t g0,
                             int64_t n, hipStream_t st);
// The same for n <= 65,535 simulations of several jobs of window size ns, named by
// (job, first) of `sims` in order of decreasing steps: active[b] of them have steps
// in block b of `blocks`; max_out: most output qubits of their jobs.
hipError_t launch_wide_tiles_jobs(int ns, bool column, uint32_t flags, const Job* jobs,
                                  const BatchItem* sims, int64_t n, const int64_t* active, int blocks,
                                  int max_out, void* ws, hipStream_t st);
hipError_t launch_wide_sample(const Job& J, bool column, const uint64_t* xm, const uint64_t* zm,
                              const int32_t* out_off, int32_t* outcomes, int32_t words,
                              uint64_t seed, hipStream_t st);
// One persistent launch over a batch's work items of window size ns with
// `waves` resident wavefronts.
hipError_t launch_wide_batch(int ns, bool column, int64_t waves, const Job* jobs,
                             const BatchItem* items, int64_t n_items, int* counter, uint32_t flags,
                             hipStream_t st);

// Adjoint sweeps of column plans with 4..14 slots.  Checkpoints: the state after
// every ck-th block and after the last, ckpt[(block / ck) * total + g] each
// 2^ns amplitudes.
struct WideAdjoint {
  int64_t C;          // columns per parameter set
  int32_t P, red;     // partial-sum rows per set, columns per row
  int32_t ck;         // blocks per checkpoint
  int32_t n_angles;
};
constexpr size_t kWideMaxLds = 160 * 1024 - 256;   // gfx950: 160 KiB per workgroup
bool wide_adjoint_fits(int ns, int red, int n_angles);
hipError_t launch_wide_adj_forward(const Job& J, float2* ckpt, int ck, hipStream_t st);
hipError_t launch_wide_adj_backward(const Job& J, const float2* ckpt, const float2* seed,
                                    const WideAdjoint& A, float* gpart, hipStream_t st);

// Angle gradients of a column plan of 2..5 slots whose slots are all outputs, from
// outputs and seed [B][C][2^ns] alone, into grad[B][n_angles]; with `loss`, also loss[B] =
// 1 + Re sum conj(seed) out / 2.
hipError_t launch_pauli_gradient(const Job& J, const float2* out, const float2* seed, int64_t B,
                                 int64_t C, int n_angles, float* loss, float* grad,
                                 hipStream_t st);

// Density matrices of column plans with 2..7 slots (wide_dm.hip); pad_slots:
// slots that start as |+> padding (n_slots - n_inputs).
hipError_t launch_dm_pauli(const Job& J, const DmNoise& nz, int pad_slots, uint32_t flags,
                           hipStream_t st);

}  // namespace mbqc
