// Branches of one launch on side streams: forked from the caller's stream, joined
// back into it whether or not every launch succeeded, so that work already on a
// branch never outlives the call's place in the caller's stream (and a stream
// capture is left with no open branch).  Api: the runtime's calls (kernels.hip).
#pragma once

namespace mbqc {

template <typename Api, int MAX>
class SideStreams {
 public:
  using Stream = typename Api::Stream;
  using Event = typename Api::Event;
  using Error = typename Api::Error;

  // `fork`, side[i] and join[i] belong to the caller and are used in branch i.
  SideStreams(Stream main, Event fork, const Stream* side, const Event* join)
      : main_(main), fork_(fork), side_(side), join_(join) {}

  Error fork() { return Api::record(fork_, main_); }

  // Branch i begins: what follows on side[i] comes after the fork.
  Error begin(int i) {
    const Error e = Api::wait(side_[i], fork_);
    if (e == Api::kOk) begun_[i] = true;
    return e;
  }

  // Joins every branch that began; the first error, all of them tried.
  Error join() {
    Error first = Api::kOk;
    for (int i = 0; i < MAX; ++i) {
      if (!begun_[i]) continue;
      begun_[i] = false;
      Error e = Api::record(join_[i], side_[i]);
      if (e == Api::kOk) e = Api::wait(main_, join_[i]);
      if (first == Api::kOk) first = e;
    }
    return first;
  }

 private:
  Stream main_;
  Event fork_;
  const Stream* side_;
  const Event* join_;
  bool begun_[MAX] = {};
};

}  // namespace mbqc
