"""The parts of the host-device copies that need no GPU (csrc/host_parts.hpp), compiled as they are."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, body):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text('#include "host_parts.hpp"\n#include <atomic>\n#include <cstdio>\n#include <set>\n#include <system_error>\n'
                   '#define CHECK(x) do { if (!(x)) { std::printf("%d: %s\\n", __LINE__, #x); return 1; } } while (0)\n'
                   + body)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "npeff_ref_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.parametrize("threads", [0, 1, 3, 7])
def test_shares_run_without_threads(tmp_path, threads):
    """As many threads as can be made, every share once."""
    _run(tmp_path, """
int main() {
  for (int n = 1; n <= 8; n++) {
    std::atomic<int> ran[8] = {};
    int made = 0;
    auto spawn = [&](auto f) {
      if (made == %d) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
      made++;
      return std::thread(f);
    };
    dn::run_shares(n, [&](int t) { ran[t]++; }, spawn);
    for (int t = 0; t < n; t++) CHECK(ran[t] == 1);
    for (int t = n; t < 8; t++) CHECK(ran[t] == 0);
  }
}
""" % threads)


def test_idle_objects_stay_with_their_device(tmp_path):
    _run(tmp_path, """
int main() {
  dn::idle_by_device<int> idle;
  int x = -1;
  CHECK(!idle.take(0, &x));
  for (int k = 0; k < 4; k++) CHECK(idle.give(0, 10 + k, 4));
  CHECK(!idle.give(0, 14, 4));
  CHECK(idle.give(1, 20, 4));
  CHECK(idle.take(1, &x) && x == 20);
  CHECK(!idle.take(1, &x));
  CHECK(idle.take(0, &x) && x == 13);
  std::set<int> left;
  idle.drain([&](int& y) { left.insert(y); });
  CHECK(left == (std::set<int>{10, 11, 12}));
  CHECK(!idle.take(0, &x));
}
""")


@pytest.mark.parametrize("first, n", [(0, 1), (0, 4096), (1, 4096), (4095, 2), (17, 8192), (5000, 100_000), (4096, 0)])
def test_fetched_pages_are_there_and_hold_what_they_held(tmp_path, first, n):
    _run(tmp_path, """
#include <cstring>
#include <sys/mman.h>
int main() {
  const size_t first = %d, n = %d, page = 4096, pages = 40;
  char* p = (char*)mmap(nullptr, pages * page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  CHECK(p != (char*)MAP_FAILED);
  madvise(p, pages * page, MADV_NOHUGEPAGE);
  dn::fetch_pages(p + first, n);
  unsigned char there[pages];
  CHECK(mincore(p, pages * page, there) == 0);
  for (size_t q = 0; q < pages; q++) {
    const bool of_range = n && q >= first / page && q <= (first + n - 1) / page;
    CHECK((there[q] & 1) == of_range);
  }
  for (size_t i = 0; i < pages * page; i++) CHECK(p[i] == 0);
  for (size_t i = 0; i < pages * page; i++) p[i] = (char)(i * 31 + 7);
  dn::fetch_pages(p + first, n);
  for (size_t i = 0; i < pages * page; i++) CHECK(p[i] == (char)(i * 31 + 7));
}
""" % (first, n))
