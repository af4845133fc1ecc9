// Launches of many workgroups.  A launch has less than 2^32 threads; the runtime drops
// workgroups of a larger one without an error.
#pragma once
#include <cstdint>

namespace mbqc {

// launch(first, count) for runs of the `blocks` workgroups of `threads` threads that
// one launch can take each, until one returns something else than `ok`.
template <typename Status, typename Launch>
Status in_grids(int64_t blocks, int64_t threads, Status ok, Launch&& launch) {
  const int64_t most = ((int64_t(1) << 32) - 1) / threads;
  Status s = ok;
  for (int64_t first = 0; first < blocks && s == ok; first += most)
    s = launch(first, blocks - first < most ? blocks - first : most);
  return s;
}

}  // namespace mbqc
