// Launches of many workgroups.  A launch has less than 2^32 threads; the runtime drops
// workgroups of a larger one without an error.
#pragma once
#include <cstdint>

namespace mbqc {

// Most workgroups of `threads` threads in one launch.
constexpr int64_t max_grid(int64_t threads) { return ((int64_t(1) << 32) - 1) / threads; }

// launch(first, count) for runs of the `blocks` workgroups of `threads` threads that
// one launch can take each, until one returns something else than `ok`.
template <typename Status, typename Launch>
Status in_grids(int64_t blocks, int64_t threads, Status ok, Launch&& launch) {
  const int64_t most = max_grid(threads);
  Status s = ok;
  for (int64_t first = 0; first < blocks && s == ok; first += most)
    s = launch(first, blocks - first < most ? blocks - first : most);
  return s;
}

// launch(b, n_sets, s, n_inputs) for parts of sets x inputs simulations of at most `most`
// each: whole sets, or runs of one set's inputs where those alone are too many.
template <typename Status, typename Launch>
Status in_parts(int64_t sets, int64_t inputs, int64_t most, Status ok, Launch&& launch) {
  const int64_t per_b = inputs < most ? most / inputs : 1, per_s = inputs < most ? inputs : most;
  Status st = ok;
  for (int64_t b = 0; b < sets && st == ok; b += per_b)
    for (int64_t s = 0; s < inputs && st == ok; s += per_s)
      st = launch(b, sets - b < per_b ? sets - b : per_b, s, inputs - s < per_s ? inputs - s : per_s);
  return st;
}

}  // namespace mbqc
