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
int main(int argc, char** argv) {
  if (argc == 5) {   // sets inputs most fails
    int n = 0;
    const int fails = std::atoi(argv[4]);
    const int e = mbqc::in_parts(std::atoll(argv[1]), std::atoll(argv[2]), std::atoll(argv[3]), 0,
                                 [&](int64_t b, int64_t nb, int64_t s, int64_t ns) {
      std::printf("%lld+%lldx%lld+%lld ", (long long)b, (long long)nb, (long long)s, (long long)ns);
      return ++n == fails ? 5 : 0;
    });
    std::printf("= %d", e);
    return 0;
  }
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


@pytest.mark.parametrize("sets,inputs,most,fails,want", [
    (5, 3, 100, 0, "0+5x0+3 = 0"), (5, 3, 7, 0, "0+2x0+3 2+2x0+3 4+1x0+3 = 0"),
    (2, 8, 8, 0, "0+1x0+8 1+1x0+8 = 0"), (2, 9, 8, 0, "0+1x0+8 0+1x8+1 1+1x0+8 1+1x8+1 = 0"),
    (2, 9, 8, 2, "0+1x0+8 0+1x8+1 = 5"), (1, 20, 8, 0, "0+1x0+8 0+1x8+8 0+1x16+4 = 0"),
    (0, 3, 8, 0, "= 0")])
def test_every_simulation_in_some_part(program, sets, inputs, most, fails, want):
    out = subprocess.run([str(program), *map(str, (sets, inputs, most, fails))], capture_output=True,
                         text=True, check=True).stdout
    assert out == want
