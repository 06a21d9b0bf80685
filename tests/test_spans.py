"""Positions near 2^31 in the loops over a graph's arrays (csrc/spans.hpp), on the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu_workgroup_managment_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include "spans.hpp"
using namespace wgm;

// Every position of [first, stop) once, by `lanes` lanes that take `per` a step.
static bool walk(long long first, long long stop, int lanes, int per) {
  long long count = 0, sum = 0;
  for (int lane = 0; lane < lanes; lane++) {
    long long turns = 0;
    for (Span s{(uint32_t)first + (uint32_t)lane, (uint32_t)stop}; s.has(); s.next(lanes * per)) {
      if (++turns > (stop - first) / (lanes * per) + 1) return false;  // went on past the end
      for (int q = 0; q < per; q++) {
        if (!s.has(q * lanes)) continue;
        const long long at = (long long)s.at + q * lanes;
        if (at < first || at >= stop) return false;
        count++;
        sum += at - first;
      }
    }
  }
  const long long n = stop - first;
  return count == n && sum == n * (n - 1) / 2;
}

// The same in segments of k positions.
static bool segments(long long first, long long stop, int k) {
  long long at = first;
  for (Span s{(uint32_t)first, (uint32_t)stop}; s.has(); s.next(k)) {
    if ((long long)s.at != at || at >= stop) return false;
    at = s.until(k);
  }
  return at == stop;
}

// The first position whose cost (4 a position, a jump of `jump` at n / 3) reaches the target.
static bool split(long long n, long long jump, long long target) {
  auto cost = [&](long long p) { return 4 * p + (p > n / 3 ? jump : 0); };
  Split s{0u, (uint32_t)n};
  int rounds = 0;
  while (s.open()) {
    int k = 0;
    for (uint32_t lane = 0; lane < 64; lane++) {
      const long long p = s.probe(lane);
      k += p < (long long)s.b && cost(p) < target;
    }
    if (k == 0) break;
    s.narrow(k);
    if (++rounds > 40 || (long long)s.b > n) return false;
  }
  long long a = 0, b = n;
  while (a < b) {
    const long long mid = (a + b) / 2;
    if (cost(mid) < target) a = mid + 1;
    else b = mid;
  }
  return (long long)s.a == a;
}

int main(int argc, char** argv) {
  const long long stop = std::atoll(argv[1]);
  const int shapes[][2] = {{64, 4}, {8, 2}, {64, 1}, {16, 1}, {1024, 2}, {1024, 4}, {65536, 1}, {262144, 1}};
  for (long long len : {0ll, 1ll, 3ll, 4ll, 5ll, 63ll, 64ll, 65ll, 255ll, 256ll, 257ll, 4099ll, 600011ll}) {
    if (len > stop) continue;
    for (auto& s : shapes)
      if (!walk(stop - len, stop, s[0], s[1])) return std::printf("walk %lld %lld %d %d\n", stop, len, s[0], s[1]), 1;
    for (int k : {64, 2048, 524288})
      if (!segments(stop - len, stop, k)) return std::printf("segments %lld %lld %d\n", stop, len, k), 1;
  }
  for (long long jump : {0ll, 1000000ll})
    for (long long part = 0; part <= 64; part++)
      if (!split(stop, jump, (4 * stop + jump) / 64 * part + part % 3))
        return std::printf("split %lld %lld %lld\n", stop, jump, part), 1;
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("spans")
    (d / "spans.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fwrapv", "-I", CSRC, "-o", d / "spans", d / "spans.cpp"], check=True)
    return d / "spans"


@pytest.mark.parametrize("stop", [1, 64, 1000003, 2 ** 31 - 4097, 2 ** 31 - 64, 2 ** 31 - 2, 2 ** 31 - 1])
def test_positions_up_to_the_last(program, stop):
    """The largest arrays have 2^31 - 1 entries: loops visit every position, none beyond, and end."""
    r = subprocess.run([program, str(stop)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
