"""The host threads behind copies to pageable memory, without a device: what
they copy, and the processor time they take while they wait for a part."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "ibfs_amd" / "csrc"

PROGRAM = r"""
#include <sys/resource.h>

#include <chrono>
#include <cstdio>

#include "copy_pool.h"

using ibfs::CopyPool;

static double cpu_s() {
  rusage r;
  getrusage(RUSAGE_SELF, &r);
  return r.ru_utime.tv_sec + r.ru_stime.tv_sec + 1e-6 * (r.ru_utime.tv_usec + r.ru_stime.tv_usec);
}

int main() {
  CopyPool pool;
  const size_t n = 3, bytes = (1 << 20) + 5;
  std::vector<char> src(n * bytes), dst(n * bytes);
  for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 7 + i / 251);
  for (bool spin : {true, false}) {
    std::fill(dst.begin(), dst.end(), 0);
    std::vector<CopyPool::Part> parts(n);
    for (size_t j = 0; j < n; ++j) {
      parts[j].dst = dst.data() + j * bytes;
      parts[j].src = src.data() + j * bytes;
      parts[j].bytes = bytes;
    }
    pool.begin(parts.data(), (int)n, spin);
    double waited = 0;
    for (size_t j = 0; j < n; ++j) {  // every part arrives 100 ms after the one before
      const double c0 = cpu_s();
      std::this_thread::sleep_for(std::chrono::milliseconds(100));
      waited += cpu_s() - c0;
      pool.ready((int)j + 1);
      pool.wait_part((int)j);
    }
    pool.end();
    if (src != dst) return 2;
    std::printf("spin=%d cpu=%.4f\n", spin, waited);
  }
  // a transfer that ends early: the parts never ready are left alone
  std::fill(dst.begin(), dst.end(), 0);
  std::vector<CopyPool::Part> parts(2);
  for (size_t j = 0; j < 2; ++j) {
    parts[j].dst = dst.data() + j * bytes;
    parts[j].src = src.data() + j * bytes;
    parts[j].bytes = bytes;
  }
  pool.begin(parts.data(), 2, false);
  pool.ready(1);
  pool.wait_part(0);
  std::this_thread::sleep_for(std::chrono::milliseconds(20));
  pool.end();
  if (!std::equal(dst.begin(), dst.begin() + bytes, src.begin()) || dst[bytes] != 0) return 3;
  // many short transfers, parts ready at once or as they are taken
  for (int k = 0; k < 2000; ++k) {
    std::vector<CopyPool::Part> p(3);
    for (size_t j = 0; j < 3; ++j) {
      p[j].dst = dst.data() + j * 1000;
      p[j].src = src.data() + (j + k % 5) * 1000;
      p[j].bytes = 999;
    }
    pool.begin(p.data(), 3, (k & 1) != 0);
    for (int j = 1; j <= 3; ++j) {
      pool.ready(j);
      if (k % 3) pool.wait_part(j - 1);
    }
    for (int j = 0; j < 3; ++j) pool.wait_part(j);
    pool.end();
    for (size_t j = 0; j < 3; ++j)
      if (std::memcmp(p[j].dst, p[j].src, 999) != 0) return 4;
  }
  std::puts("done");
  std::fflush(stdout);
  std::_Exit(0);  // the pool's threads live as long as the process
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_waiting_threads_take_no_processor_time(tmp_path):
    """Parts that arrive 100 ms apart: eight threads that poll for them would
    take up to 2.4 s; they poll for 1 ms a part at most (24 ms in all) and then
    sleep, and sleep at once in a transfer of whole chunks."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-pthread", "-I", str(CSRC), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    lines = r.stdout.split("\n")
    cpu = {l.split()[0]: float(l.split("cpu=")[1]) for l in lines if "cpu=" in l}
    assert "done" in lines and len(cpu) == 2
    assert cpu["spin=1"] < 0.15 and cpu["spin=0"] < 0.05, cpu
