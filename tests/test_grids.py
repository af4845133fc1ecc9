"""The cutting of launches into grids that one launch can take (mentpy_amd/csrc/grids.h):
every workgroup once, in order, fewer than 2^32 threads each, and a stop at an error."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mentpy_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "grids.h"
int main(int, char** argv) {
  const int64_t blocks = std::atoll(argv[1]), threads = std::atoll(argv[2]), fails = std::atoll(argv[3]);
  int n = 0;
  const int e = mbqc::in_grids(blocks, threads, 0, [&](int64_t first, int64_t count) {
    std::printf("%lld+%lld ", (long long)first, (long long)count);
    return ++n == fails ? 5 : 0;
  });
  std::printf("= %d", e);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("grids")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-I", str(CSRC), str(d / "p.cpp"), "-o", str(d / "p")], check=True)
    return d / "p"


@pytest.mark.parametrize("blocks,threads,fails,want", [
    (0, 64, 0, "= 0"), (1, 64, 0, "0+1 = 0"), (67108863, 64, 0, "0+67108863 = 0"),
    (67108864, 64, 0, "0+67108863 67108863+1 = 0"),
    (4194304, 1024, 0, "0+4194303 4194303+1 = 0"),
    (10000000, 1024, 0, "0+4194303 4194303+4194303 8388606+1611394 = 0"),
    (10000000, 1024, 2, "0+4194303 4194303+4194303 = 5"),
    (3, 0xffffff * 256, 0, "0+1 1+1 2+1 = 0"),
])
def test_every_workgroup_in_some_launch(program, blocks, threads, fails, want):
    out = subprocess.run([str(program), str(blocks), str(threads), str(fails)], capture_output=True,
                         text=True, check=True).stdout
    assert out == want
