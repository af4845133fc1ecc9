"""The fork and join of a launch's side streams (mentpy_amd/csrc/side_streams.h) with a
runtime that records its calls and fails on demand: every branch that began is
joined, also after a failed launch or a failed call."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mentpy_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include "side_streams.h"
static int calls = 0, fail_at = -1;
static int step(const char* what, int a, int b) {
  const bool bad = calls++ == fail_at;
  std::printf("%s%d,%d%s ", what, a, b, bad ? "!" : "");
  return bad ? 7 : 0;
}
struct Api {
  using Stream = int; using Event = int; using Error = int;
  static constexpr int kOk = 0;
  static int record(int ev, int st) { return step("record", ev, st); }
  static int wait(int st, int ev) { return step("wait", st, ev); }
};
int main(int argc, char** argv) {
  int launch_fails_at = -1;
  for (int i = 1; i + 1 < argc; i += 2)
    std::sscanf(argv[i + 1], "%d", std::strcmp(argv[i], "call") ? &launch_fails_at : &fail_at);
  const int side[4] = {10, 11, 12, 13}, join[4] = {20, 21, 22, 23};
  mbqc::SideStreams<Api, 4> s(1, 2, side, join);
  int e = s.fork();
  for (int i = 3; i >= 1 && !e; --i) {
    e = s.begin(i);
    if (e) break;
    std::printf("launch%d ", i);
    if (i == launch_fails_at) e = 9;
  }
  const int ej = s.join();
  std::printf("= %d", e ? e : ej);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("side_streams")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-I", str(CSRC), str(d / "p.cpp"), "-o", str(d / "p")], check=True)
    return d / "p"


JOIN = {i: f"record2{i},1{i} wait1,2{i} " for i in (1, 2, 3)}


@pytest.mark.parametrize("args,want", [
    ((), "record2,1 wait13,2 launch3 wait12,2 launch2 wait11,2 launch1 " + JOIN[1] + JOIN[2] + JOIN[3] + "= 0"),
    # the second launch fails: both branches that began are joined
    (("launch", "2"), "record2,1 wait13,2 launch3 wait12,2 launch2 " + JOIN[2] + JOIN[3] + "= 9"),
    # a branch that could not begin is not joined, the one before it is
    (("call", "2"), "record2,1 wait13,2 launch3 wait12,2! " + JOIN[3] + "= 7"),
    # a failed join does not keep the other branches from theirs
    (("call", "4"), "record2,1 wait13,2 launch3 wait12,2 launch2 wait11,2 launch1 record21,11! "
     + JOIN[2] + JOIN[3] + "= 7"),
])
def test_every_branch_that_began_is_joined(program, args, want):
    out = subprocess.run([str(program), *args], capture_output=True, text=True, check=True).stdout
    assert out == want
