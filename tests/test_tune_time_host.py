"""Which launches of a candidate the schedule tuners compare (host compiler, no GPU)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ed_lattice_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "tune_time.hpp"
int main(int, char** a) {
  const double warm = atof(a[1]), cold = atof(a[2]), best = atof(a[3]), latency = atof(a[4]);
  int launches = 0;
  auto clock = [&](int n) {
    double t = latency;
    for (int k = 0; k < n; ++k) t += warm + (launches++ ? 0.0 : cold);
    return t;
  };
  const double ms = edl::candidate_ms([&]() { clock(1); }, clock, best);
  std::printf("%.6f %d\n", ms, launches);
}
"""


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    d = tmp_path_factory.mktemp("tune")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(d / "t"), str(d / "main.cpp")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("warm,cold,best,latency,launches,kept", [
    (0.008, 0.4, 0.010, 0.0, 4, True),     # a kernel of a few us, its first launch forty times as long
    (0.006, 0.4, 0.006, 0.008, 4, True),   # ... as fast as the best, alone twice as long
    (0.100, 0.4, 0.010, 0.01, 4, False),   # small sectors are not cut short
    (0.500, 0.4, 0.520, 0.01, 5, True),    # headline sizes: a cold first launch is not held against it
    (0.510, 0.0, 0.520, 0.01, 4, True),    # ... a warm one counts as such
    (0.900, 0.1, 0.520, 0.01, 2, False),   # dropped by its second launch
    (1.300, 0.4, 0.520, 0.01, 1, False),   # dropped by its first
    (20.0, 0.4, 21.0, 0.01, 4, True),      # the largest sectors
    (24.0, 0.4, 21.0, 0.01, 1, False),
    (0.010, 0.4, 1e300, 0.01, 4, True),    # the first candidate
])
def test_candidate(tool, warm, cold, best, latency, launches, kept):
    ms, n = subprocess.run([tool, str(warm), str(cold), str(best), str(latency)], capture_output=True, text=True,
                           check=True).stdout.split()
    assert int(n) == launches
    if kept:  # a warm mean, nothing of the first launch
        assert warm <= float(ms) <= warm + latency
    else:     # no new best
        assert float(ms) > best
