"""Small host-and-device helpers of the native code, compiled on their own with
g++ and checked on the CPU."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ufemism_amd", "csrc")


@pytest.fixture(scope="module")
def run_driver(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("helpers")

    def run(name, source):
        (d / f"{name}.cpp").write_text(source)
        subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-pthread", f"-I{CSRC}", str(d / f"{name}.cpp"),
                        "-o", str(d / name)], check=True)
        r = subprocess.run([str(d / name)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_couplings_read_ahead_stay_inside_the_level(run_driver):
    """Every place of every block, blocks without couplings (the last one among
    them, whose start is the array's length) included, reads inside the array,
    and places that hold a coupling read their own."""
    run_driver("held_index", r"""
#include <cstdio>
#include <vector>
#include "amg_host.h"
int main() {
  for (std::vector<int> blocks : std::vector<std::vector<int>>{{1}, {5, 0}, {0, 7}, {0, 3, 0, 0}, {2048, 2049, 0}, {300, 0, 1}}) {
    int total = 0, k0 = 0;
    for (int nn : blocks) total += nn;
    for (int nn : blocks) {
      for (int i = 0; i < 8 * 256; i++) {
        const int k = ufe::amg_held_index(k0, nn, i);
        if (k < 0 || k >= total || (i < nn && k != k0 + i)) return std::printf("k0 %d nn %d place %d: %d of %d\n", k0, nn, i, k, total), 1;
      }
      k0 += nn;
    }
  }
  return 0;
}
""")


def test_patch_buffers_are_made_each_on_its_own(run_driver):
    """A call that fails or finds no room at any of the buffers leaves the others
    to the next call, which makes what is missing and nothing twice."""
    run_driver("spaces", r"""
#include <cstdio>
#include "patch_host.h"
int main() {
  for (int stop = 0; stop < 3; stop++)          // the buffer that is refused
    for (int code : {0, 7}) {                   // no room, or an error
      int made = 0, x[3];
      int *a = nullptr, *b = nullptr, *c = nullptr;
      auto make = [&](int *&p) {
        if (made == stop) return code;
        p = &x[made++];
        return 0;
      };
      const int r = ufe::patch_spaces(make, a, b, c);
      if (r != code || (a && b && c)) return std::printf("refused at %d: status %d\n", stop, r), 1;
      int made2 = made;
      auto make2 = [&](int *&p) {
        p = &x[made2++];
        return 0;
      };
      const int r2 = ufe::patch_spaces(make2, a, b, c);
      if (r2 || !a || !b || !c || made2 != 3 || a == b || b == c || a == c)
        return std::printf("after a refusal at %d: status %d, %d made\n", stop, r2, made2), 1;
    }
  return 0;
}
""")
