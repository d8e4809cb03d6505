"""Places in k_integrate's work list (reserve_items), compiled for the host and
asked for by several threads at once: lists that hold every request and lists
that do not.  Long items grow from the front and short ones from the back, no
place may be given out twice, and the places up to the counts that the first
refused request keeps are all given out, none beyond."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include <algorithm>
using std::max;
using std::min;
#include "rx_math.h"
int main(int argc, char **argv) {
  const int cap = atoi(argv[1]), n_req = atoi(argv[2]), most = atoi(argv[3]);
  for (unsigned seed = 1; seed <= 20; seed++) {
    std::atomic<uint64_t> ctr{0};
    std::vector<std::atomic<int>> slot(cap);
    for (auto &s : slot) s = 0;
    std::atomic<int> bad{0}, refused{0}, first{0};
    std::atomic<long> fit{0}, fit_s{0};
    std::vector<std::thread> th;
    for (int t = 0; t < 8; t++)
      th.emplace_back([&, t] {
        unsigned r = seed * 977u + t * 131u;
        for (int q = t; q < n_req; q += 8) {
          r = r * 1664525u + 1013904223u;
          const int tot = (r >> 8) % (most + 1), tots = (r >> 20) % 17;
          int base = -1, bases = -1;
          bool first_out = false;
          if (!rx::reserve_items([&](uint64_t v) { return ctr.fetch_add(v); }, tot, tots, cap, base, bases, first_out)) {
            refused++;
            if (first_out) {
              first++;
              fit = base;
              fit_s = bases;
            }
            continue;
          }
          for (int k = 0; k < tot + tots; k++) {
            const int at = k < tot ? base + k : cap - 1 - (bases + (k - tot));
            if (at < 0 || at >= cap || slot[at].fetch_add(1) != 0) bad++;
          }
        }
      });
    for (auto &x : th) x.join();
    if (first != (refused ? 1 : 0)) bad++;
    const long n_long = refused ? (long)fit : (long)(uint32_t)ctr.load();
    const long n_short = refused ? (long)fit_s : (long)(ctr.load() >> 32);
    for (long k = 0; k < cap; k++)
      if ((slot[k] == 1) != (k < n_long || k >= cap - n_short)) bad++;
    printf("%d %d\n", (int)bad, (int)refused);
  }
}
"""


@pytest.mark.parametrize("cap,n_req,most", [(1, 20, 2), (4000, 64, 40), (700, 64, 40), (100000, 4096, 40), (100000, 4096, 900)])
def test_places(tmp_path, cap, n_req, most):
    src, exe = tmp_path / "places.cpp", str(tmp_path / "places")
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-w", "-I", os.path.join(ROOT, "relxill_amd", "csrc"), str(src),
                    "-o", exe], check=True)
    out = subprocess.run([exe, str(cap), str(n_req), str(most)], check=True, capture_output=True, text=True).stdout
    rows = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(rows) == 20 and all(bad == 0 for bad, _ in rows)
    holds_all = cap >= n_req * (most + 16)
    assert all((refused == 0) == holds_all for _, refused in rows)
