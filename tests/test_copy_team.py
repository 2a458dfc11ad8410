"""The threads that copy large results to the caller (csrc/copy_team.h), on the
CPU: every byte of results of one chunk, several, and a ragged last one arrives;
a team that is given up before its first chunk leaves the caller's buffer as it
was; and its helpers sleep while the first chunk is being computed."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include <stdio.h>
#include <stdlib.h>
#include <time.h>
#include <chrono>
#include "copy_team.h"
using rtg::CopyTeam;
static char value(size_t i) { return (char)(i * 2654435761u >> 13); }
static int copies(size_t bytes, size_t chunk) {
  std::vector<char> dst(bytes + 64, 'x'), b0(chunk), b1(chunk);
  {
    CopyTeam team(dst.data(), bytes, chunk, b0.data(), b1.data());
    team.touch();
    for (size_t i = 0; i < team.count(); ++i) {
      for (size_t k = 0; k < team.size(i); ++k) (i & 1 ? b1 : b0)[k] = value(i * chunk + k);
      team.copy(i);
    }
  }
  for (size_t i = 0; i < bytes; ++i)
    if (dst[i] != value(i)) return printf("byte %zu of %zu (chunks of %zu) is wrong\n", i, bytes, chunk), 1;
  for (size_t i = bytes; i < dst.size(); ++i)
    if (dst[i] != 'x') return printf("written past %zu bytes\n", bytes), 1;
  return 0;
}
static int given_up() {
  const size_t n = 1 << 22, chunk = 1 << 20;
  std::vector<char> dst(n, 'x'), b0(chunk), b1(chunk);
  clock_t t0;
  {
    CopyTeam team(dst.data(), n, chunk, b0.data(), b1.data());
    team.touch();
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    t0 = clock();
    std::this_thread::sleep_for(std::chrono::milliseconds(400));
    t0 = clock() - t0;
  }
  for (size_t i = 0; i < n; ++i)
    if (dst[i] != 'x') return printf("byte %zu was overwritten\n", i), 1;
  const double busy = (double)t0 / CLOCKS_PER_SEC;
  if (busy > 0.1) return printf("the helpers ran for %.2f s of 0.4 s\n", busy), 1;
  return 0;
}
int main(int argc, char** argv) {
  if (argc > 1) return given_up();
  for (size_t bytes : {1, 4, 4095, 4096, 16384, 65536, 65540, 1000000, 1048576})
    for (size_t chunk : {4096, 65536, 262144})
      if (copies(bytes, chunk)) return 1;
  return 0;
}
'''


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("copy_team")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "rusttorch_amd", "csrc"), "-o",
                    str(d / "t"), str(d / "t.cpp")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("args", [[], ["given up"]], ids=["copies", "given up"])
def test_copy_team(program, args):
    r = subprocess.run([program, *args], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
