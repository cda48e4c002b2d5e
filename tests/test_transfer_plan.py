"""The chunks of a transfer on the CPU: for every size, in either direction and
through the buffers of a context made for a larger grid, the buffers stay
inside the pool, the chunks cover the transfer, and the sizes are those that
the header's measurements ask for."""
import os
import subprocess

import pytest

from evora_amd import build

SRC = """
#include <cstdio>
#include <cstdlib>
#include "transfer.h"
using namespace evh;
static int bad = 0;
static void check(bool ok, const char *what, long long a, long long b) {
  if (!ok && bad++ < 10) std::printf("%s: %lld of %lld\\n", what, a, b);
}
static void size(long long n, long long most) {
  const long long pool = pool_bytes(most);
  check(pool >= kCellBytes && pool <= kPoolBytes, "pool", n, most);
  for (int bytes : {48, 8})
    for (int up = 0; up < 2; up++) {
      const ChunkPlan c = chunk_plan(n, bytes, up, pool);
      check(c.units >= 1 && c.buffers >= 1 && c.buffers <= kBuffers, "plan", n, most);
      check(c.units * bytes * c.buffers <= pool, "buffers", n, most);
      check(c.units * c.buffers >= n || c.buffers >= 2, "one buffer", n, most);
      if (bytes == 48 && up && n == most && n * 48 <= 10 << 20) check(c.units >= n, "one piece", n, most);
      if (bytes == 48 && n == most && n * 48 > 64 << 20) check(c.units * bytes >= 8 << 20, "short chunks", n, most);
      if (bytes == 48 && n == most) check((n + c.units - 1) / c.units <= (n * 48 >> 20) / 24 + 25, "chunks", n, most);
    }
}
int main() {
  for (long long n = 1; n < 3000; n++) size(n, n);
  for (long long n = 3000; n < 3LL << 30; n += n / 97) {
    size(n, n);
    for (long long m = n; m < 3LL << 30; m = m * 5 / 3 + 1) size(n, m);
  }
  for (int n = 2; n < 600; n++) size((long long)n * n * n, (long long)n * n * n);
  std::printf("%d wrong\\n", bad);
  return bad != 0;
}
"""


def test_chunks_and_buffers(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    (tmp_path / "plan.hip").write_text(SRC)
    exe = tmp_path / "plan"
    r = subprocess.run([build.HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function", "-I", build.CSRC,
                        str(tmp_path / "plan.hip"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
