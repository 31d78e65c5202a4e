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


OUT_OF_MEMORY = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "patch_host.h"
static std::atomic<long> left{1L << 40};
void *operator new(size_t n) {
  void *p = left.fetch_sub(1) > 0 ? std::malloc(n ? n : 1) : nullptr;
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
using namespace ufe;
// a grid of n x n points, coloured so that the four neighbours of a point have the other colours; its rim: edge points
int main() {
  const int n = 300, nA = n * n;
  std::vector<int> id(nA), at(nA);
  int cs[6], ca[5], k = 0;
  auto rim = [&](int p) { return p % n == 0 || p / n == 0 || p % n == n - 1 || p / n == n - 1; };
  for (int c = 0; c < 5; c++) {
    cs[c] = k;
    for (int edge = 0; edge < 2; edge++) {
      for (int p = 0; p < nA; p++)
        if ((p % n + 2 * (p / n)) % 5 == c && rim(p) == (edge == 1)) id[k] = p, at[p] = k++;
      if (!edge) ca[c] = k - cs[c];
    }
  }
  cs[5] = nA;
  std::vector<int64_t> cptr((nA + 63) / 64 + 1);
  for (size_t i = 0; i < cptr.size(); i++) cptr[i] = 256 * (int64_t)i;
  std::vector<uint8_t> deg(nA);
  std::vector<int32_t> col(cptr.back()), er, ep{0}, ec;
  std::vector<uint32_t> key(nA);
  for (int q = 0; q < nA; q++) {
    const int p = id[q], x = p % n, y = p / n;
    key[q] = (uint32_t)p;
    int d = 0;
    for (int v : {x ? p - 1 : -1, x < n - 1 ? p + 1 : -1, y ? p - n : -1, y < n - 1 ? p + n : -1})
      if (v >= 0) col[cptr[q >> 6] + (q & 63) + 64 * d++] = at[v];
    deg[q] = (uint8_t)d;
    if (rim(p)) {                    // a corner of the rim averages its inner diagonal
      er.push_back(q);
      int inner[4], m = 0;
      for (int j = 0; j < d; j++)
        if (!rim(id[col[cptr[q >> 6] + (q & 63) + 64 * j]])) inner[m++] = col[cptr[q >> 6] + (q & 63) + 64 * j];
      if (!m) inner[m++] = at[(y ? n - 2 : 1) * n + (x ? n - 2 : 1)];
      ec.insert(ec.end(), inner, inner + m);
      ep.push_back((int32_t)ec.size());
    }
  }
  const PatchMesh m{nA, cs, ca, cptr.data(), deg.data(), col.data(), (int)er.size(), 0, er.data(), ep.data(), ec.data(),
                    nullptr, nullptr, nullptr, key.data(), nullptr};
  const std::vector<int32_t> order = patch_order(m);
  int whole = 0, refused = 0;
  for (long allow = 0; allow < 4000; allow = allow < 200 ? allow + 1 : allow + 97) {
    std::vector<PatchHost> parts;
    bool built = false;
    left = allow;
    try {
      built = patch_build(m, order, 200, 2, false, true, true, parts);
    } catch (const std::bad_alloc &) {   // on the calling thread: its C interface reports it
    }
    left = 1L << 40;
    size_t own = 0;
    for (const PatchHost &H : parts)
      for (const PatchDesc &d : H.d) own += d.own[0] + d.own[1] + d.own[2] + d.own[3] + d.own[4] + d.own_e + d.own_k;
    if (built && own != (size_t)nA) return std::printf("allowed %ld: %zu of %d points\n", allow, own, nA), 1;
    (built ? whole : refused)++;
  }
  std::printf("%d whole, %d refused\n", whole, refused);
  return whole && refused ? 0 : 2;
}
"""


def test_running_out_of_host_memory_ends_the_walk_and_not_the_process(tmp_path):
    """operator new fails after a number of allocations, on whichever thread asks."""
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    (tmp_path / "oom.cpp").write_text(OUT_OF_MEMORY)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-pthread", f"-I{CSRC}", str(tmp_path / "oom.cpp"), "-o",
                    str(tmp_path / "oom")], check=True)
    r = subprocess.run([str(tmp_path / "oom")], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


THREADS = r"""
#include <cstdio>
#include <cstring>
#include "patch_host.h"
using namespace ufe;
extern "C" int threads_for(int64_t n) { return patch_threads(n); }
extern "C" int same(int nA, const int *cs, const int *ca, const int64_t *cptr, const uint8_t *deg, const int32_t *col,
                    int n_neu, const int32_t *nr, const int32_t *np_, const int32_t *nc, int n_cor, const int32_t *kr,
                    const int32_t *kp, const int32_t *kc, const uint32_t *key, int own, int backward) {
  const PatchMesh m{nA, cs, ca, cptr, deg, col, n_neu, n_cor, nr, np_, nc, kr, kp, kc, key, nullptr};
  const std::vector<int32_t> order = patch_order(m);
  PatchHost J[2];
  for (int i = 0; i < 2; i++) {
    std::vector<PatchHost> parts;
    if (!patch_build(m, order, own, 2, backward != 0, true, true, parts, INT32_MAX, i ? 7 : 1)) return -1;
    if (parts.size() != (i ? 7u : 1u)) return -2;
    auto join = [](auto &a, auto &b) { a.insert(a.end(), b.begin(), b.end()); };
    for (PatchHost &q : parts) {
      join(J[i].d, q.d);
      join(J[i].rows, q.rows);
      join(J[i].nptr, q.nptr);
      join(J[i].sbase, q.sbase);
      join(J[i].lcol, q.lcol);
      join(J[i].ov_e, q.ov_e);
      join(J[i].ovf, q.ovf);
      join(J[i].ov_c, q.ov_c);
      join(J[i].ncol, q.ncol);
    }
  }
  if (J[0].d.size() != J[1].d.size()) return -3;
  for (size_t b = 0; b < J[0].d.size(); b++) {
    const PatchDesc &x = J[0].d[b], &y = J[1].d[b];
    auto lists = [](const PatchHost &H, const PatchDesc &d) {
      return std::vector<int32_t>(H.rows.begin() + d.list, H.rows.begin() + d.list + d.nlist);
    };
    if (x.nlist != y.nlist || x.ncs != y.ncs || x.nov != y.nov || x.list != y.list || lists(J[0], x) != lists(J[1], y)) return -4;
  }
  return J[0].sbase == J[1].sbase && J[0].lcol == J[1].lcol && J[0].ov_e == J[1].ov_e && J[0].ovf == J[1].ovf &&
         J[0].ov_c == J[1].ov_c;
}
"""


@pytest.mark.parametrize("own,backward", [(64, 0), (240, 1)])
def test_patches_do_not_depend_on_the_threads(tmp_path, own, backward):
    """A mesh of 16k vertices is walked by several threads (where the machine has
    them), with the patches of one."""
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    (tmp_path / "threads.cpp").write_text(THREADS)
    so = tmp_path / "threads.so"
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-fPIC", "-shared", "-pthread", f"-I{CSRC}",
                    str(tmp_path / "threads.cpp"), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.threads_for.argtypes = [ctypes.c_int64]
    assert lib.threads_for(200) == 1 and lib.threads_for(64000) <= lib.threads_for(1 << 22) <= 16
    if len(os.sched_getaffinity(0)) > 1:
        assert lib.threads_for(64000) > 1
    m = colour_order(geometry.marine(5000, seed=8).mesh)
    ptr = lambda a: ctypes.c_void_p(np.ascontiguousarray(a).ctypes.data)  # noqa: E731
    assert lib.same(m["n"], ptr(m["start"]), ptr(m["active"]), ptr(m["cptr"]), ptr(m["deg"]), ptr(m["col"]),
                    len(m["neu"][0]), *map(ptr, m["neu"]), len(m["cor"][0]), *map(ptr, m["cor"]), ptr(m["key"]), own,
                    backward) == 1
