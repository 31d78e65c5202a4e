"""Limits of the patches (ufemism_amd/csrc/patch_host.h) that are found before a
walk, on the CPU."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from test_patch_host import colour_order
from ufemism_amd import geometry

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ufemism_amd", "csrc")
DRIVER = r"""
#include "patch_host.h"
using namespace ufe;
// least group by the colours, and the largest of the patches built
extern "C" void groups(int nA, const int *cs, const int *ca, const int64_t *cptr, const uint8_t *deg, const int32_t *col,
                       int n_neu, const int32_t *nr, const int32_t *np_, const int32_t *nc, int n_cor, const int32_t *kr,
                       const int32_t *kp, const int32_t *kc, const uint32_t *key, int own, int nu, int *out) {
  const PatchMesh m{nA, cs, ca, cptr, deg, col, n_neu, n_cor, nr, np_, nc, kr, kp, kc, key, nullptr};
  std::vector<PatchHost> parts;
  out[0] = patch_least_group(ca, (nA + own - 1) / own);
  out[1] = patch_build(m, patch_order(m), own, nu, false, true, false, parts) ? 0 : -1;
  for (const PatchHost &H : parts) out[1] = std::max(out[1], H.max_group);
  // allowed exactly that many, and one fewer
  out[2] = patch_build(m, patch_order(m), own, nu, false, true, false, parts, out[1]);
  out[3] = patch_build(m, patch_order(m), own, nu, false, true, false, parts, out[1] - 1);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("limits")
    (d / "limits.cpp").write_text(DRIVER)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-fPIC", "-shared", "-pthread", f"-I{CSRC}",
                    str(d / "limits.cpp"), "-o", str(d / "limits.so")], check=True)
    return ctypes.CDLL(str(d / "limits.so"))


@pytest.mark.parametrize("kind,n", [("dome", 600), ("marine", 5000)])
@pytest.mark.parametrize("own", [64, 500, 3000, 10**6])
@pytest.mark.parametrize("nu", [1, 2])
def test_least_group_never_exceeds_the_walked_one(lib, kind, n, own, nu):
    """So a mesh refused by it would have been refused after the walk, too; and a
    walk with a bound ends without patches exactly when one exceeds it."""
    m = colour_order(getattr(geometry, kind)(n, seed=3).mesh)
    ptr = lambda a: ctypes.c_void_p(np.ascontiguousarray(a).ctypes.data)  # noqa: E731
    out = (ctypes.c_int * 4)()
    lib.groups(m["n"], ptr(m["start"]), ptr(m["active"]), ptr(m["cptr"]), ptr(m["deg"]), ptr(m["col"]), len(m["neu"][0]),
               *map(ptr, m["neu"]), len(m["cor"][0]), *map(ptr, m["cor"]), ptr(m["key"]), min(own, m["n"]), nu, out)
    print(f"  {kind} {n} own {own}: colours {m['active']} of {m['n']}, least {out[0]}, walked {out[1]}", flush=True)
    assert 0 < out[0] <= out[1]
    assert (out[2], out[3]) == (1, 0)
