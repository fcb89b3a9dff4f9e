"""Chunks of a download handed over by several threads (hg_rows.hpp), on the
CPU: every chunk once and only after it has arrived, threads that start with
the first chunk, a thread that cannot be had, and a transfer that fails."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hormone_amd",
                    "csrc")
MAIN = """
#include "hg_rows.hpp"
#include <cstdio>
#include <new>
#include <system_error>
#include <vector>
static int made, limit, kind;
static std::atomic<long> arrived;
struct Thread {  // the limit-th one cannot be had
  std::thread t;
  Thread() = default;
  template <class F> explicit Thread(F &f) {
    if (arrived.load() < 1) std::puts("a thread before the first chunk"), std::exit(3);
    if (made++ == limit) {
      if (kind == 0) throw std::bad_alloc();
      throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    }
    t = std::thread(std::ref(f));
  }
  Thread &operator=(Thread &&o) = default;
  void join() { t.join(); }
};
int main() {
  for (kind = 0; kind < 2; ++kind)
    for (limit = 0; limit < 9; ++limit)
      for (long n : {1, 2, 3, 8, 31, 32})
        for (long fail : {-1L, 0L, n / 2, n - 1}) {
          made = 0;
          arrived = 0;
          std::vector<std::atomic<int>> seen(n);
          for (auto &x : seen) x = 0;
          const bool ok = hg::hand_over_chunks<Thread>(
              n, 7,
              [&](long q) {
                if (q == fail) return false;
                arrived = q + 1;
                return true;
              },
              [&](long q) {
                if (arrived.load() <= q) std::puts("a chunk before it arrived"), std::exit(4);
                ++seen[q];
              });
          if (ok != (fail < 0)) return 5;
          for (auto &x : seen)
            if (ok ? x != 1 : x > 1) return 6;
        }
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_chunks_are_handed_over_once(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "rows"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-I", CSRC, "-o", str(exe),
                    str(tmp_path / "main.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
